// Paged-KV attention for decode ("flash-decoding", split over the context).
//
// KV cache layout (engine/kv_cache.py): K and V are each
//     [num_pages][n_kv_heads][PAGE=64][D=128] bf16
// so one page of one kv head is a contiguous 16 KiB tile.  Every query row r
// carries a block-table row (its sequence) and a context length; a query row
// is either one decode token or one prefill token (causal: ctx = pos + 1).
//
// Grid: (kv_head, row, chunk); a chunk = 4 pages = 256 keys (4 waves x 64 keys) or 16 pages (8 waves x 2 x 64).
// GQA packing: all G = Hq / Hkv query heads of a kv head are scored against the
// same K/V bytes in one pass (K/V read once per group, not once per q head).
// With one chunk the block writes the final bf16 output, otherwise fp32
// partials (m, l, o) for the combine kernel.
#include "common.h"

namespace {

constexpr int PAGE = 64;
constexpr int HD = 128;
constexpr int CHUNK = 4 * PAGE;

// One wave takes a page (64 keys) of a chunk at a time, all of its loads before any arithmetic, and keeps the
// running maximum, sum and output of its pages in registers; the waves of a workgroup meet once, at the end.
//   S^T[key][head] = K . Q^T  v_mfma_f32_16x16x32_bf16: A = 16 keys x 32 numbers from the page, B = the query heads,
//                             padded to 16 with zeros; lane (head, key quarter) then holds the scores of
//                             keys 16 b + 4 quarter + j
//   O[head][number] += P . V  v_mfma_f32_4x4x1f32 of 16 blocks: a lane holds 8 numbers of one V row (quarter = which
//                             of 4 keys, so a load is 4 whole rows of 256 B), and the quarter's probabilities
//                             of 4 heads are the scores' registers as they are (broadcast from the quarter's first
//                             lanes).  P stays fp32 and V is not moved: no LDS, no transposition.
// What bounds it: the K and V bytes, 32 KB in flight per wave.  The form before it (16 waves of 16 keys, products by
// the vector unit from LDS, a 16-way merge of 32 KB) was bound by its LDS traffic, and its order of the grid (chunks
// first) gave XCDs 0 and 4 the chunks that every row has and 3 and 7 those that few rows have; heads come first now.
// With the combine, per launch: 19 rows of up to 900 keys, 8 kv heads of 4 (37 MB) 27.8 -> 14.8 us; 20 rows of 200 keys
// 11.0 -> 8.1; 1 row of 1000 12.7 -> 10.3; 64 rows of 500 (131 MB) 41.0 -> 31.8.
// <4, 1>: a page per wave, 256-key chunks.  <8, 2>: 1024-key chunks, a quarter of the partial outputs and two pages in
// turn per wave: 32 rows of 8000 keys 209.6 -> 199.3 us, 2 rows of 30000 55.8 -> 52.3; but at 4 rows of 1000
// 10.9 against 17.8, so only where its workgroups are two per CU.
template <int G, int NW, int PPW>
__global__ __launch_bounds__(NW * 64) void paged_attn_kernel(
    const bf16* __restrict__ q, int ldq, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ bt, int bt_stride, const int* __restrict__ row_bt,
    const int* __restrict__ ctx_lens, int Hkv, float scale, int n_chunks, bf16* __restrict__ out,
    int ldo, float* __restrict__ part_o, float* __restrict__ part_ml) {
  constexpr int HG = (G + 3) / 4;  // groups of 4 heads
  constexpr bool ONE = G == 1;
  const int h = blockIdx.x, r = blockIdx.y, c = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, qd = lane >> 4;
  __shared__ float so[NW][G][HD];
  __shared__ float sm[NW][G], sl[NW][G];

  // independent loads together: the context length, the block-table row, q
  const int ctx = ctx_lens[r];
  const int rb = row_bt ? row_bt[r] : r;  // null: row r uses block-table row r (decode)
  bf16x8 qf[4];
  {
    const bf16x2* qp = reinterpret_cast<const bf16x2*>(q + (size_t)r * ldq + (size_t)(h * G + min(n, G - 1)) * HD + 8 * qd);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16x2 x = qp[16 * s + i];
        qf[s][2 * i] = ONE || n < G ? x[0] : (bf16)0.f;
        qf[s][2 * i + 1] = ONE || n < G ? x[1] : (bf16)0.f;
      }
  }
  const int p0 = c * NW * PPW + w;  // this wave's pages: p0, p0 + NW, ...
  int page[PPW];
#pragma unroll
  for (int t = 0; t < PPW; ++t) page[t] = bt[(size_t)rb * bt_stride + min(p0 + t * NW, bt_stride - 1)];
  if (c * NW * PPW * PAGE >= ctx) return;  // block-uniform: the whole chunk is past the context

  f32x4 acc[HG][8];
#pragma unroll
  for (int g = 0; g < HG; ++g)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[g][e] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int t = 0; t < PPW; ++t) {
    const int nv = min(ctx - (p0 + t * NW) * PAGE, PAGE);  // keys of the page inside the context
    if (nv <= 0) break;                                    // wave-uniform
    // rows past the context are not read (what they hold may be anything): they are beyond the buffers' end, zero for both
    // products (the last valid row in their place would make 0 * inf of its infinite values)
    const size_t base = ((size_t)__builtin_amdgcn_readfirstlane(page[t]) * Hkv + h) * PAGE * HD;
    const int bytes = nv * HD * (int)sizeof(bf16);
    const __amdgpu_buffer_rsrc_t keys = __builtin_amdgcn_make_buffer_rsrc((void*)(kc + base), 0, bytes, 0x00027000);
    const __amdgpu_buffer_rsrc_t values = __builtin_amdgcn_make_buffer_rsrc((void*)(vc + base), 0, bytes, 0x00027000);
    auto load = [](const __amdgpu_buffer_rsrc_t& rows, int at) {
      return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rows, at * (int)sizeof(bf16), 0, 0));
    };
    bf16x8 kr[4][4], vr[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int s = 0; s < 4; ++s) kr[b][s] = load(keys, (16 * b + n) * HD + 32 * s + 8 * qd);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) vr[b][j] = load(values, (16 * b + 4 * qd + j) * HD + 8 * n);
    __builtin_amdgcn_sched_barrier(0);  // all 32 loads are on their way before the first product waits
    f32x4 st[4];
    float mx = -INFINITY;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      st[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) st[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[b][s], qf[s], st[b], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        st[b][j] = 16 * b + 4 * qd + j < nv ? st[b][j] * scale : -INFINITY;
        mx = fmaxf(mx, st[b][j]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m1 = fmaxf(m, mx), alpha = __expf(m - m1);
    m = m1;
    float ls = 0.f;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        st[b][j] = __expf(st[b][j] - m);  // -inf -> 0
        ls += st[b][j];
      }
    l = fmaf(l, alpha, ls);
    if (t > 0) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha), g));
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g >> 2][e][g & 3] *= a;
      }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float v = (float)vr[b][j][e];
          if constexpr (ONE) {
            acc[0][e][0] = fmaf(st[b][j], v, acc[0][e][0]);
            continue;
          }
          acc[0][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(st[b][j], v, acc[0][e], 2, 0, 0);
          if constexpr (HG > 1) acc[1][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(st[b][j], v, acc[1][e], 2, 1, 0);
        }
  }
  // The four quarters hold four keys' parts of the same 8 numbers: each keeps two of them, summed.
  const auto add32 = [](float a, float b) {  // lanes below 32: a's sum, the others b's
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(x[0]) + __uint_as_float(x[1]);
  };
  const auto add16 = [](float a, float b) {  // even rows of 16 lanes: a's sum, odd ones b's
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(x[0]) + __uint_as_float(x[1]);
  };
  const int d0 = 8 * n + 4 * (qd >> 1) + 2 * (qd & 1);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = add32(acc[g >> 2][e][g & 3], acc[g >> 2][e + 4][g & 3]);
    so[w][g][d0] = add16(y[0], y[2]);
    so[w][g][d0 + 1] = add16(y[1], y[3]);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lane < G) {
    sm[w][lane] = m;
    sl[w][lane] = l;
  }
  __syncthreads();
  const int Hq = Hkv * G;
  for (int i = tid; i < G * HD; i += NW * 64) {
    const int g = i / HD, d = i % HD;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, sm[ww][g]);
    float num = 0.f, den = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const float e = __expf(sm[ww][g] - M);
        num = fmaf(e, so[ww][g][d], num);
        den = fmaf(e, sl[ww][g], den);
      }
    }
    const int hq = h * G + g;
    if (n_chunks == 1) {
      out[(size_t)r * ldo + (size_t)hq * HD + d] = f2bf(num / den);
    } else {
      const size_t pidx = ((size_t)r * Hq + hq) * n_chunks + c;
      part_o[pidx * HD + d] = num;
      if (d == 0) {
        part_ml[pidx * 2] = M;
        part_ml[pidx * 2 + 1] = den;
      }
    }
  }
}

// Split-K combine: one block per (row, q head).  The chunk statistics go to LDS first
// (one load per chunk, all in flight together), then CG groups of HD threads each sum
// the partial outputs of every CG-th chunk with 8 loads in flight per thread, and the
// groups meet in LDS.  (A serial per-dimension loop over the chunks leaves one load
// in flight per thread: ~85 us per layer at a 32K context.)
constexpr int CG = 8;                  // chunk groups per block
constexpr int MAX_CHUNKS = 131072 / CHUNK;  // 128K-token contexts
__global__ __launch_bounds__(HD * CG) void attn_combine_kernel(const float* __restrict__ part_o,
                                                               const float* __restrict__ part_ml,
                                                               const int* __restrict__ ctx_lens,
                                                               int Hq, int n_chunks, int chunk,
                                                               bf16* __restrict__ out, int ldo) {
  __shared__ float s_e[MAX_CHUNKS];  // exp(m_c - M)
  __shared__ float s_l[MAX_CHUNKS];
  __shared__ float s_red[CG][HD];
  __shared__ float s_wmax[HD * CG / 64];
  const int r = blockIdx.x, hq = blockIdx.y, tid = threadIdx.x;
  const int d = tid % HD, grp = tid / HD;
  const int nc = min(min((ctx_lens[r] + chunk - 1) / chunk, n_chunks), MAX_CHUNKS);
  const size_t base = ((size_t)r * Hq + hq) * n_chunks;
  float mloc = -INFINITY;
  for (int c = tid; c < nc; c += HD * CG) {
    const float m = part_ml[(base + c) * 2];
    s_e[c] = m;
    s_l[c] = part_ml[(base + c) * 2 + 1];
    mloc = fmaxf(mloc, m);
  }
  mloc = wave_max(mloc);
  if ((tid & 63) == 0) s_wmax[tid >> 6] = mloc;
  __syncthreads();
  float M = -INFINITY;
#pragma unroll
  for (int i = 0; i < HD * CG / 64; ++i) M = fmaxf(M, s_wmax[i]);
  __syncthreads();
  for (int c = tid; c < nc; c += HD * CG) s_e[c] = s_e[c] == -INFINITY ? 0.f : __expf(s_e[c] - M);
  __syncthreads();
  float num = 0.f;
  const float* po = part_o + base * HD + d;
  int c = grp;
  for (; c + 7 * CG < nc; c += 8 * CG) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = po[(size_t)(c + u * CG) * HD];
#pragma unroll
    for (int u = 0; u < 8; ++u) num = fmaf(s_e[c + u * CG], v[u], num);
  }
  for (; c < nc; c += CG) num = fmaf(s_e[c], po[(size_t)c * HD], num);
  s_red[grp][d] = num;
  __syncthreads();
  if (grp == 0) {
    float tot = 0.f, den = 0.f;
#pragma unroll
    for (int g = 0; g < CG; ++g) tot += s_red[g][d];
    for (int i = 0; i < nc; ++i) den = fmaf(s_e[i], s_l[i], den);
    out[(size_t)r * ldo + (size_t)hq * HD + d] = f2bf(den > 0.f ? tot / den : 0.f);
  }
}

// The same for at most FEW chunks: a thread per output number, every load of it in flight at once.
constexpr int FEW = 8;
__global__ __launch_bounds__(4 * HD) void attn_combine_few_kernel(const float* __restrict__ part_o,
                                                                  const float* __restrict__ part_ml,
                                                                  const int* __restrict__ ctx_lens,
                                                                  int Hq, int n_chunks, int chunk,
                                                                  bf16* __restrict__ out, int ldo) {
  const int r = blockIdx.x, hq = blockIdx.y * 4 + threadIdx.x / HD, d = threadIdx.x % HD;
  if (hq >= Hq) return;
  const int ctx = ctx_lens[r];
  const size_t base = ((size_t)r * Hq + hq) * n_chunks;
  float o[FEW], m[FEW], l[FEW];
#pragma unroll
  for (int c = 0; c < FEW; ++c) {
    const size_t i = base + min(c, n_chunks - 1);
    o[c] = part_o[i * HD + d];
    m[c] = part_ml[2 * i];
    l[c] = part_ml[2 * i + 1];
  }
  const int nc = min((ctx + chunk - 1) / chunk, n_chunks);
  float M = -INFINITY, num = 0.f, den = 0.f;
#pragma unroll
  for (int c = 0; c < FEW; ++c) M = c < nc ? fmaxf(M, m[c]) : M;
#pragma unroll
  for (int c = 0; c < FEW; ++c) {
    // chunks past the context were not written: not read into the sums either
    const float e = c < nc && m[c] != -INFINITY ? __expf(m[c] - M) : 0.f;
    num = fmaf(e, c < nc ? o[c] : 0.f, num);
    den = fmaf(e, c < nc ? l[c] : 0.f, den);
  }
  out[(size_t)r * ldo + (size_t)hq * HD + d] = f2bf(den > 0.f ? num / den : 0.f);
}

// ---- single-chunk decode attention on MFMA (contexts <= 256 keys: chat decode) ----
// Opt-in, P in bf16 and V through LDS: 4 waves x 64 keys (= one KV page per wave, so one
// block-table load per wave) run both products on v_mfma_f32_16x16x32_bf16 with the
// query heads on the MFMA's N axis (G <= 16, padded with zero rows):
//   S^T[key][head] = K . Q^T   (A = 16 keys x 32 dims straight from the page, 16 B per
//                               lane; B = q fragments, loaded once)
//   O[head][dim]  += P . V     (A = P: the S^T accumulator registers after the softmax ARE
//                               the A fragment -- lane (head, key group) -- with the 32
//                               keys of a k-step taken as two 16-key blocks; B = V^T
//                               fragments read from the wave's V rows in LDS with the
//                               same key permutation)
// and the 4 wave partials merge once through LDS.
constexpr int MW = 4;            // waves
constexpr int MKPW = 64;         // keys per wave = one page
constexpr int MVS = HD + 8;      // V row stride (bf16) in LDS: conflict-free 16-B writes

template <int G>
__global__ __launch_bounds__(MW * 64) void paged_attn_mfma_kernel(
    const bf16* __restrict__ q, int ldq, const bf16* __restrict__ kc, const bf16* __restrict__ vc,
    const int* __restrict__ bt, int bt_stride, const int* __restrict__ row_bt,
    const int* __restrict__ ctx_lens, int Hkv, float scale, bf16* __restrict__ out, int ldo) {
  static_assert(G >= 1 && G <= 16, "query heads on the MFMA N axis");
  __shared__ __attribute__((aligned(16))) bf16 vs[MW][MKPW][MVS];
  __shared__ float so[MW][G][HD];
  __shared__ float sm[MW][G], sl[MW][G];
  const int h = blockIdx.x, r = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int kk = lane & 15, qd = lane >> 4;
  const int ctx = ctx_lens[r];
  const int rb = row_bt ? row_bt[r] : r;
  const int page = bt[(size_t)rb * bt_stride + min(w, bt_stride - 1)];  // wave-uniform
  const size_t pbase = ((size_t)page * Hkv + h) * PAGE * HD;

  // loads: K and V rows of this wave's 64 keys (block b = keys 16b.., lane row kk, dims
  // 32s + 8qd..), q fragments of the G heads (rows kk >= G are zero)
  bf16x8 kr[4][4], vr[4][4], qf[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const bf16x8* kp = reinterpret_cast<const bf16x8*>(kc + pbase + (size_t)(16 * b + kk) * HD + 8 * qd);
    const bf16x8* vp = reinterpret_cast<const bf16x8*>(vc + pbase + (size_t)(16 * b + kk) * HD + 8 * qd);
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) kr[b][s2] = kp[4 * s2];
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) vr[b][s2] = vp[4 * s2];
  }
  {
    const bf16x8* qp = reinterpret_cast<const bf16x8*>(q + (size_t)r * ldq +
                                                       (size_t)(h * G + min(kk, G - 1)) * HD + 8 * qd);
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2) qf[s2] = kk < G ? qp[4 * s2] : zero_bf16x8();
  }
  const int n_valid = min(max(ctx - w * MKPW, 0), MKPW);  // wave-uniform

  // V rows -> LDS (this wave's region only: a wave barrier orders them for its reads)
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int s2 = 0; s2 < 4; ++s2)
      *reinterpret_cast<bf16x8*>(&vs[w][16 * b + kk][32 * s2 + 8 * qd]) = vr[b][s2];

  float mg = -INFINITY, lg = 0.f;  // per head kk (every lane of column kk agrees)
  f32x4 o[HD / 16];
#pragma unroll
  for (int c = 0; c < HD / 16; ++c) o[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (n_valid > 0) {
    // S^T blocks: lane holds keys 16b + 4qd + j (j < 4) of head kk
    f32x4 st[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      st[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s2 = 0; s2 < 4; ++s2)
        st[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kr[b][s2], qf[s2], st[b], 0, 0, 0);
    }
    float m = -INFINITY;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool ok = 16 * b + 4 * qd + j < n_valid;
        st[b][j] = ok ? st[b][j] * scale : -INFINITY;
        m = fmaxf(m, st[b][j]);
      }
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    float l = 0.f;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p = __expf(st[b][j] - m);  // -inf -> 0
        st[b][j] = p;
        l += p;
      }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    mg = m;
    lg = l;
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's V rows are in LDS
    __builtin_amdgcn_wave_barrier();
    // P.V: k-step t covers key blocks 2t (A slots 0-3) and 2t+1 (slots 4-7)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      bf16x8 pa;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        pa[j] = f2bf(st[2 * t][j]);
        pa[4 + j] = f2bf(st[2 * t + 1][j]);
      }
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) {
        bf16x8 vb;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          vb[j] = vs[w][32 * t + 4 * qd + j][16 * c + kk];
          vb[4 + j] = vs[w][32 * t + 16 + 4 * qd + j][16 * c + kk];
        }
        o[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa, vb, o[c], 0, 0, 0);
      }
    }
  }
  // O accumulators: lane holds O[head 4qd + j][dim 16c + kk]
#pragma unroll
  for (int c = 0; c < HD / 16; ++c)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int hd = 4 * qd + j;
      if (hd < G) so[w][hd][16 * c + kk] = o[c][j];
    }
  if (qd == 0 && kk < G) {
    sm[w][kk] = mg;
    sl[w][kk] = lg;
  }
  __syncthreads();
  for (int i = tid; i < G * HD; i += MW * 64) {
    const int hd = i / HD, d = i % HD;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < MW; ++ww) M = fmaxf(M, sm[ww][hd]);
    float num = 0.f, den = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < MW; ++ww) {
        const float e = __expf(sm[ww][hd] - M);
        num = fmaf(e, so[ww][hd][d], num);
        den = fmaf(e, sl[ww][hd], den);
      }
    }
    out[(size_t)r * ldo + (size_t)(h * G + hd) * HD + d] = f2bf(den > 0.f ? num / den : 0.f);
  }
}

// Opt-in (p2p_paged_attention_mfma(1)): 7.7-7.9 us per launch at 44-256 keys, no faster than fp32 probabilities
// (profiles/r2_decode_attn_mfma.jsonl): bound by the block-table -> K/V load chain, not by the arithmetic.
static int g_attn_mfma = 0;

template <int G, int NW, int PPW>
int launch_pages(const void* q, int ldq, const void* kc, const void* vc, const int* bt, int bt_stride,
                 const int* row_bt, const int* ctx, int R, int Hkv, float scale, int max_ctx, void* out,
                 int ldo, float* part_o, float* part_ml, hipStream_t st) {
  constexpr int chunk = NW * PPW * PAGE;
  const int n_chunks = (max_ctx + chunk - 1) / chunk;
  hipLaunchKernelGGL((paged_attn_kernel<G, NW, PPW>), dim3(Hkv, R, n_chunks), dim3(NW * 64), 0, st,
                     (const bf16*)q, ldq, (const bf16*)kc, (const bf16*)vc, bt, bt_stride, row_bt,
                     ctx, Hkv, scale, n_chunks, (bf16*)out, ldo, part_o, part_ml);
  int e = (int)hipGetLastError();
  if (e || n_chunks == 1) return e;
  if (n_chunks <= FEW)
    hipLaunchKernelGGL(attn_combine_few_kernel, dim3(R, (Hkv * G + 3) / 4), dim3(4 * HD), 0, st, part_o, part_ml,
                       ctx, Hkv * G, n_chunks, chunk, (bf16*)out, ldo);
  else
    hipLaunchKernelGGL(attn_combine_kernel, dim3(R, Hkv * G), dim3(HD * CG), 0, st, part_o, part_ml, ctx,
                     Hkv * G, n_chunks, chunk, (bf16*)out, ldo);
  return (int)hipGetLastError();
}

template <int G>
int launch_attn(const void* q, int ldq, const void* kc, const void* vc, const int* bt,
                int bt_stride, const int* row_bt, const int* ctx, int R, int Hkv, float scale,
                int max_ctx, void* out, int ldo, float* part_o, float* part_ml, hipStream_t st) {
  if (max_ctx <= CHUNK && g_attn_mfma) {
    hipLaunchKernelGGL((paged_attn_mfma_kernel<G>), dim3(Hkv, R), dim3(MW * 64), 0, st,
                       (const bf16*)q, ldq, (const bf16*)kc, (const bf16*)vc, bt, bt_stride, row_bt,
                       ctx, Hkv, scale, (bf16*)out, ldo);
    return (int)hipGetLastError();
  }
  // 1024-key chunks where they give 512 workgroups and more (measured at the kernel); 640 where up to 4 heads to a kv head
  // and several chunks meet: 512 end as one round of which contexts below their bucket leave CUs idle (8 kv heads of 4, 8
  // rows of 5120 keys in a bucket of 8192: 31.3 us with 256-key chunks, 39.5 with these; one head, 8 rows 30.0 / 35.5)
  const long long groups = max_ctx < 1024 ? 0 : (long long)R * Hkv * ((max_ctx + 1023) / 1024);
  if (groups >= (G == 8 || max_ctx == 1024 ? 512 : 640))
    return launch_pages<G, 8, 2>(q, ldq, kc, vc, bt, bt_stride, row_bt, ctx, R, Hkv, scale, max_ctx, out, ldo, part_o, part_ml, st);
  return launch_pages<G, 4, 1>(q, ldq, kc, vc, bt, bt_stride, row_bt, ctx, R, Hkv, scale, max_ctx, out, ldo, part_o, part_ml, st);
}

}  // namespace

// 1: contexts <= 256 keys run the kernel with bf16 probabilities; 0 (default): paged_attn_kernel.
P2P_API void p2p_paged_attention_mfma(int on) { g_attn_mfma = on; }

// row_bt null = identity (decode batches: row r is sequence r), one dependent load less
// on the kernel's critical path (row_bt -> page -> K/V becomes page -> K/V).
// max_ctx bounds the number of chunks (grid.z); workgroups past a row's context
// exit early.  part_o / part_ml: workspace of R*Hq*n_chunks*(128 | 2) floats,
// unused when max_ctx <= 256.
P2P_API int p2p_paged_attention(const void* q, int ldq, const void* k_cache, const void* v_cache,
                                const int* block_tables, int bt_stride, const int* row_bt,
                                const int* ctx_lens, int R, int Hq, int Hkv, int head_dim,
                                float scale, int max_ctx, void* out, int ldo, float* part_o,
                                float* part_ml, hipStream_t stream) {
  if (head_dim != HD || Hkv <= 0 || Hq % Hkv != 0 || R <= 0) return (int)hipErrorInvalidValue;
  const int n_chunks = (max_ctx + CHUNK - 1) / CHUNK;
  if (n_chunks > 1 && (!part_o || !part_ml)) return (int)hipErrorInvalidValue;
  if (n_chunks > MAX_CHUNKS) return (int)hipErrorInvalidValue;
  switch (Hq / Hkv) {
    case 1: return launch_attn<1>(q, ldq, k_cache, v_cache, block_tables, bt_stride, row_bt, ctx_lens, R, Hkv, scale, max_ctx, out, ldo, part_o, part_ml, stream);
    case 2: return launch_attn<2>(q, ldq, k_cache, v_cache, block_tables, bt_stride, row_bt, ctx_lens, R, Hkv, scale, max_ctx, out, ldo, part_o, part_ml, stream);
    case 4: return launch_attn<4>(q, ldq, k_cache, v_cache, block_tables, bt_stride, row_bt, ctx_lens, R, Hkv, scale, max_ctx, out, ldo, part_o, part_ml, stream);
    case 8: return launch_attn<8>(q, ldq, k_cache, v_cache, block_tables, bt_stride, row_bt, ctx_lens, R, Hkv, scale, max_ctx, out, ldo, part_o, part_ml, stream);
  }
  return (int)hipErrorInvalidValue;
}
