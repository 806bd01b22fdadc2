// Causal prefill attention on MFMA (flash-attention style) over the paged KV
// cache, GQA-packed: one workgroup = one KV head x one tile of <= 16
// consecutive query tokens of one sequence; wave w of the G = Hq/Hkv waves
// owns q-head kvh*G + w, so every K/V tile staged in LDS feeds G heads.
//
// Per 32-key tile and wave (everything transposed so no register shuffles are
// needed between the two GEMMs):
//   S^T[32 keys x 16 tok] = K[keys x 128] . Q^T          8 x mfma_16x16x32_bf16
//   (online softmax per token column; lane owns one token and 8 keys)
//   O^T[128 x 16 tok]   += V^T[128 x 32 keys] . P^T      8 x mfma_16x16x32_bf16
// The MFMA reduction index k is a permutation of the 32 keys chosen so that
// the S^T accumulator registers of a lane ARE its P^T B-operand (slot (g, j)
// <-> key 4g+j for j<4, 16+4g+j-4 otherwise); V^T uses the same permutation.
//
// Tiles come by LDS DMA three stages deep, one barrier each, and V^T is read transposed from V's rows.  What bounds it: a
// wave's chain per tile (scores, maximum, exponentials, second product).  One prompt, 32 heads on 8, per layer: 64 rows
// 6.2 -> 6.0 us, 256 14.1 -> 11.7, 700 34.1 -> 29.0, 100 rows at 4000 167 -> 115 against K and V through registers, V
// transposed by 2-byte stores and two barriers a tile; the same results to the bit.
//
// Replaces the per-row decode kernel for long prompts, whose K/V traffic is
// O(T^2): here each K/V tile is read once per 16 query tokens x G heads.
// Behavioural parity: the reference delegates prompt processing to an external
// Ollama server (`web/streamlit_app.py:89-101`), see SURVEY.md §2B.2 B2.3.
#include <type_traits>

#include "common.h"
#include "lds_pipe.h"

namespace {

constexpr int PAGE = 64, HD = 128, KT = 32, QT = 16;

struct Tile {
  int row0, n, seq, pos0;
};

template <int G, int NST>   // stages
__global__ __launch_bounds__(64 * G) void flash_prefill_kernel(
    const bf16* __restrict__ q, int ldq, const bf16* __restrict__ kc,
    const bf16* __restrict__ vc, const int* __restrict__ bt, int bt_stride,
    const Tile* __restrict__ tiles, int n_tiles, int Hkv, float scale_log2,
    bf16* __restrict__ out, int ldo) {
  constexpr int TE = KT * HD, AHEAD = NST - 1;              // numbers of a tile's K (V); tiles copied ahead
  __shared__ __attribute__((aligned(16))) bf16 lds[NST * 2 * TE];   // K, V of every stage

  const int nb = n_tiles * Hkv;
  const int b = xcd_remap(blockIdx.x, nb);
  const int ti = b / Hkv, kvh = b % Hkv;  // consecutive ids: same tile, all heads
  const Tile T = tiles[ti];
  if (T.n <= 0) return;  // padding tile of a graph-captured prefill (fixed grid)
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, col = lane & 15;
  const int h = kvh * G + w;

  const int last = T.pos0 + T.n - 1;
  const int n_kt = last / KT + 1;
  const int* btr = bt + (size_t)T.seq * bt_stride;
  const size_t head_off = (size_t)kvh * PAGE * HD;
  const size_t page_sz = (size_t)Hkv * PAGE * HD;

  // copies: an instruction takes four rows of 256 bytes, piece p of row r to p ^ (r & 15) (K) or p ^ 2 (r & 7) (V); rows
  // past the last key (whatever they hold) are that key's again
  constexpr int CP = 8 / G;
  const unsigned l0 = __builtin_amdgcn_readfirstlane(ldsp::lds_off(lds)) + w * 1024;
  const int cr = 4 * w + (lane >> 4), cp = lane & 15;
  auto copy = [&](int kt, int page, int st) {
    const int k0 = kt * KT, lim = last - k0;
    const size_t base = (size_t)page * page_sz + head_off + (size_t)(k0 % PAGE) * HD;
    const unsigned dst = l0 + st * (2 * TE * 2);
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      const int r = cr + 4 * G * i, at = min(r, lim) * (HD * 2);
      ldsp::dma_lds16(kc + base, at + ((cp ^ (r & 15)) << 4), dst + i * G * 1024);
      ldsp::dma_lds16(vc + base, at + ((cp ^ (2 * (r & 7))) << 4), dst + TE * 2 + i * G * 1024);
    }
  };
  auto page_of = [&](int kt) { return btr[min(kt, n_kt - 1) * KT / PAGE]; };
  copy(0, page_of(0), 0);
  if (AHEAD > 1 && n_kt > 1) copy(1, page_of(1), 1);
  int pa = page_of(AHEAD);

  // Q^T B-operand fragments: token col, d = 32s + 8g + j
  const int tok = col < T.n ? col : T.n - 1;
  const int my_pos = T.pos0 + tok;
  bf16x8 qf[4];
  {
    const bf16* qp = q + (size_t)(T.row0 + tok) * ldq + h * HD + 8 * g;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 32 * s);
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) asm volatile("" : "+v"(qf[s]));   // loaded before the loop counts its copies

  f32x4 acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;

  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* lds4_t;
  const int vrow = 4 * g + (col >> 2), vx = 2 * (vrow & 7);       // (16 rows further: the same permutation)
  int st = 0, sa = AHEAD;                                    // stages of tile kt and kt + AHEAD
  for (int kt = 0; kt < n_kt; ++kt) {
    // this wave's copies of the tile have landed, then every wave's; the stage of the tile before is used up
    // (its own reads of it are done, too)
    if (AHEAD > 1 && kt + 1 < n_kt) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * CP) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + AHEAD < n_kt) copy(kt + AHEAD, pa, sa);
    pa = page_of(kt + AHEAD + 1);
    const bf16* Ks = lds + st * 2 * TE;
    const bf16* Vs = Ks + TE;
    sa = st;
    st = st == NST - 1 ? 0 : st + 1;

    // S^T = K Q^T : two 16-key row tiles
    bf16x8 kf[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        kf[mt][ks] = *reinterpret_cast<const bf16x8*>(&Ks[(16 * mt + col) * HD + (((4 * ks + g) ^ col) << 3)]);
    f32x4 s[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      s[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) s[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[mt][ks], qf[ks], s[mt], 0, 0, 0);
    }
    // V^T fragments on their way while the weights are formed: A row = d (16dt + col), k-slot (g, j) -> key
    // 16(j>>2) + 4g + (j&3)
    bf16x8 vf[8];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const bf16* p = Vs + vrow * HD + (((2 * dt + ((col >> 1) & 1)) ^ vx) << 3) + 4 * (col & 1);
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t)p);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t)(p + 16 * HD));
      vf[dt] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    __builtin_amdgcn_sched_barrier(0);
    // online softmax for token `col`; this lane holds keys 16mt + 4g + j
    const int k0 = kt * KT;
    float mx = -INFINITY;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int key = k0 + 16 * mt + 4 * g + j;
        const float v = key <= my_pos ? s[mt][j] * scale_log2 : -INFINITY;
        s[mt][j] = v;
        mx = fmaxf(mx, v);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    const float alpha = __builtin_amdgcn_exp2f(m - mn);  // m - mn <= 0; -inf -> 0
    m = mn;
    bf16x8 pf;
    float ps = 0.f;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p = __builtin_amdgcn_exp2f(s[mt][j] - mn);
        ps += p;
        pf[4 * mt + j] = f2bf(p);
      }
    l = l * alpha + ps;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) acc[dt] *= alpha;

    // O^T += V^T P^T
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[dt], pf, acc[dt], 0, 0, 0);
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (col < T.n) {
    const float inv = 1.f / l;
    bf16* op = out + (size_t)(T.row0 + col) * ldo + h * HD + 4 * g;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      bf16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = f2bf(acc[dt][j] * inv);
      *reinterpret_cast<bf16x4*>(op + 16 * dt) = o;
    }
  }
}

template <int G>
int launch(const bf16* q, int ldq, const bf16* kc, const bf16* vc, const int* bt, int bt_stride,
           const Tile* tiles, int n_tiles, int Hkv, float scale, bf16* out, int ldo,
           hipStream_t st) {
  const float sl2 = scale * 1.4426950408889634f;
  // Three stages are 48 KB: three workgroups to a CU.  Where those are one or two waves each and there are more of them, two
  // stages hide as much by the other two workgroups that then fit: 32 heads on 32, 32 prompts of 8 on 900 earlier tokens,
  // 1024 workgroups, 99 us with three, 82 with two; 32 on 16, 20 prompts of 44, 960 workgroups, 9.0 and 6.6.
  if constexpr (G <= 2) {
    if ((long)n_tiles * Hkv > 768) {
      hipLaunchKernelGGL((flash_prefill_kernel<G, 2>), dim3(n_tiles * Hkv), dim3(64 * G), 0, st, q, ldq,
                         kc, vc, bt, bt_stride, tiles, n_tiles, Hkv, sl2, out, ldo);
      P2P_CHECK_LAUNCH();
    }
  }
  hipLaunchKernelGGL((flash_prefill_kernel<G, 3>), dim3(n_tiles * Hkv), dim3(64 * G), 0, st, q, ldq,
                     kc, vc, bt, bt_stride, tiles, n_tiles, Hkv, sl2, out, ldo);
  P2P_CHECK_LAUNCH();
}

// ---------------------------------------------------------------------------------
// v2: 128 or 256 query rows per workgroup (NW = 4 or 8 waves x 32 rows), one 64-key page per K/V tile,
// v_mfma_f32_32x32x16_bf16 throughout.
//
// A workgroup = one KV head x QT = 32 NW / G consecutive tokens of one sequence; wave w
// owns q head kvh*G + w/(NW/G) and 32 of the tokens, so every K/V page staged in LDS
// feeds 128 or 256 (token, head) rows -- 8x or 16x the reuse of v1 (16 tokens x G heads).
// Per 64-key tile and wave, both products keep the query row on the lane:
//   S^T[32 keys x 32 rows] = K . Q^T   (per 32-key half: 8 MFMAs over d = 128)
//   O^T[128 d  x 32 rows] += V^T . P^T (4 d-blocks x 2 halves x 2 k-steps = 16 MFMAs)
// so the online-softmax statistics and the O rescale are per lane (no cross-lane
// moves but one xor-32 for the row max / sum).  The S^T accumulator registers are
// directly the P^T B operand: register 8s+j of lane half h holds S^T row
// 16s + 8(j>>2) + 4h + (j&3); the K rows are loaded permuted (row rho <- key
// kappa(rho)) so that this row is key 16s + 8h + j, i.e. the eight keys a lane
// contributes to one k-step are CONSECUTIVE.  Rows of 256 bytes in LDS, 16-byte piece p of row r at
// p ^ (r & 15) (K: 16 rows x a piece per read) and p ^ 4 (r & 3) (V: 4 rows x 64 bytes): no bank conflicts.
// What bounds it: a wavefront's chain per page (scores, maximum, exponentials, second product), with one or two
// wavefronts per SIMD to fill it.  So the page's K and V come by LDS DMA (no registers, no stores), V is read
// transposed (ds_read_b64_tr_b16) from the rows as they are, and a page's exponentials run between the products of the
// page before with V (K is a page ahead of V for that; two stages of each).
// One prompt, 32 heads on 8, per layer: 128 rows (16-token tiles) 9.1 -> 8.2 us with 4 waves, 256 14.5 -> 10.7, 512 25.5 ->
// 16.0, 700 34.6 -> 20.9; 1024 (8 waves, K and V through registers, V transposed by 2-byte stores) 39 -> 28.5, 2048
// 69 -> 55.  With 8 waves 1024 39 -> 38, 4096 149 -> 148, 8192 554 -> 557 (4 waves 156 and 564).  Same results to the bit.
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ int kperm(int rho) {  // S^T row rho -> key within the 32-key half
  const int s = rho >> 4, r = rho & 15;
  return 16 * s + 8 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
}

template <int G, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2, 2))) void flash_prefill2_kernel(
    const bf16* __restrict__ q, int ldq, const bf16* __restrict__ kc,
    const bf16* __restrict__ vc, const int* __restrict__ bt, int bt_stride,
    const Tile* __restrict__ tiles, int n_tiles, int Hkv, float scale_log2,
    bf16* __restrict__ out, int ldo) {
  constexpr int WPH = NW / G;  // waves per q head
  constexpr int PG = PAGE * HD;                                  // numbers of a page's K (V)
  __shared__ __attribute__((aligned(16))) bf16 lds[4 * PG];      // K, K, V, V

  // heads outermost, heaviest (latest) tiles first; one head's tiles share an XCD's L2
  const int nb = n_tiles * Hkv;
  const int b = xcd_remap(blockIdx.x, nb);
  const int kvh = b / n_tiles, ti = n_tiles - 1 - b % n_tiles;
  const Tile T = tiles[ti];
  if (T.n <= 0) return;  // padding tile of a graph-captured prefill (fixed grid)
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r32 = lane & 31, hh = lane >> 5;
  const int h = kvh * G + w / WPH;
  const int t = (w % WPH) * 32 + r32;      // token of this lane's query row
  const int tok = t < T.n ? t : T.n - 1;
  const int my_pos = T.pos0 + tok;
  const int row = T.row0 + tok;

  const int last = T.pos0 + T.n - 1;
  const int n_kt = last / PAGE + 1;
  const int* btr = bt + (size_t)T.seq * bt_stride;
  const size_t head_off = (size_t)kvh * PG;
  const size_t page_sz = (size_t)Hkv * PG;

  // copies: an instruction takes four rows; this wave's are rows 4 (w + NW i) + lane / 16.  Rows past the last key
  // (whatever they hold) are that key's again
  constexpr int CP = 16 / NW;
  const unsigned l0 = __builtin_amdgcn_readfirstlane(ldsp::lds_off(lds)) + w * 1024;
  const int cr = 4 * w + (lane >> 4), cp = lane & 15;
  auto copy = [&](const bf16* pool, int kt, int page, unsigned dst, bool is_v) {
    const void* base = pool + (size_t)page * page_sz + head_off;
    const int lim = last - kt * PAGE;
#pragma unroll
    for (int i = 0; i < CP; ++i) {
      const int r = cr + 4 * NW * i;
      ldsp::dma_lds16(base, min(r, lim) * (HD * 2) + ((cp ^ (is_v ? 4 * (r & 3) : r & 15)) << 4), dst + i * NW * 1024);
    }
  };
  auto copy_k = [&](int kt, int page) { copy(kc, kt, page, l0 + (kt & 1) * (PG * 2), false); };
  auto copy_v = [&](int kt, int page) { copy(vc, kt, page, l0 + (2 + (kt & 1)) * (PG * 2), true); };
  auto page_of = [&](int kt) { return btr[min(kt, n_kt - 1)]; };
  int p0 = page_of(0), p1 = page_of(1);    // pages kt and kt + 1
  copy_k(0, p0);

  // Q^T B fragments: k-step s covers d = 16s .. 16s+15, lane half hh holds 8hh .. 8hh+7
  bf16x8 qf[8];
  {
    const bf16* qp = q + (size_t)row * ldq + h * HD + 8 * hh;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = *reinterpret_cast<const bf16x8*>(qp + 16 * s);
  }
  f32x16_t o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
  float m = -INFINITY, l = 0.f;

  // K rows kperm(r32) and 32 further; V: lane L of 16 names row L / 4 of four and 4 of 16 numbers, see read_v
  const int krow = kperm(r32), L = lane & 15;
  const bf16* kl = lds + krow * HD;
  const bf16* vl = lds + 2 * PG + (8 * hh + (L >> 2)) * HD + 4 * (L & 1);
  const int vp = 2 * ((lane >> 4) & 1) + ((L >> 1) & 1);
  auto read_k = [&](int st, int kh, int s) {
    return *reinterpret_cast<const bf16x8*>(kl + st * PG + 32 * kh * HD + (((2 * s + hh) ^ (krow & 15)) << 3));
  };
  // V^T of numbers 32 db + r32, keys 32 kh + 16 s2 + 8 hh + 0 .. 7
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s16x4* lds4_t;
  auto read_v = [&](int st, int db, int kh, int s2) {
    const bf16* p = vl + st * PG + (32 * kh + 16 * s2) * HD + ((((db ^ (L >> 2)) << 2) | vp) << 3);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t)p);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t)(p + 4 * HD));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  f32x16_t sc[2];
  bf16x8 pf[2][2];   // P^T of the page before
  // O^T += V^T . P^T of page `of`, in eight pairs of products; LDS reads go out a pair ahead of the products that take
  // them, and between the pairs runs `work`
  auto second_product = [&](int of, auto&& work) {
    const int st = of & 1;
    bf16x8 vf[2][2];
    auto read_v2 = [&](int j) {   // half j & 1 of the keys, numbers 32 (j / 2) ..
#pragma unroll
      for (int i = 0; i < 2; ++i) vf[j & 1][i] = read_v(st, j >> 1, j & 1, i);
    };
    read_v2(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < 7) read_v2(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        o[j >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[j & 1][i], pf[j & 1][i], o[j >> 1], 0, 0, 0);
      work(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  for (int kt = 0; kt < n_kt; ++kt) {
    // K of this page and V of the one before have landed; every wave is past the last page's K and the V before it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    copy_v(kt, p0);
    if (kt + 1 < n_kt) copy_k(kt + 1, p1);
    p0 = p1;
    p1 = page_of(kt + 2);
    // ---- S^T = K . Q^T, two 32-key halves ----
    {
      bf16x8 kf[2][2];
      auto read_k2 = [&](int s) {
#pragma unroll
        for (int kh = 0; kh < 2; ++kh) kf[s & 1][kh] = read_k(kt & 1, kh, s);
      };
      read_k2(0);
#pragma unroll
      for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kh][i] = 0.f;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        if (s < 7) read_k2(s + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kh = 0; kh < 2; ++kh)
          sc[kh] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s & 1][kh], qf[s], sc[kh], 0, 0, 0);
      }
    }
    // ---- online softmax for this lane's query row (keys of reg rr: 16(rr>>3)+8hh+(rr&7)) ----
    // m is the running max of the RAW scores; p = exp2(s * c - m * c) is one FMA + exp.
    // Deferred rescale: O and l are rescaled only when some
    // row's max grew by more than RESCALE_THR (log2 units) -- wave-uniform decision, each
    // lane with its own factor -- so most tiles skip the 64-register multiply; the
    // unrescaled p stay <= 2^RESCALE_THR, exact in fp32 and safe in bf16.
    constexpr float RESCALE_THR = 8.f;
    const int k0 = kt * PAGE;
    // some key of the tile may be in the future (workgroup-uniform: a real branch, so the
    // mask's compares and selects run on diagonal tiles only)
    if (__builtin_amdgcn_readfirstlane(k0 + PAGE - 1 > T.pos0)) {
#pragma unroll
      for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          const int key = k0 + 32 * kh + 16 * (rr >> 3) + 8 * hh + (rr & 7);
          if (key > my_pos) sc[kh][rr] = -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) mx = fmaxf(mx, sc[kh][rr]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const bool rescale = __any((mx - m) * scale_log2 > RESCALE_THR);
    float alpha = 1.f;
    if (rescale) {
      const float mn = fmaxf(m, mx);
      alpha = exp2f((m - mn) * scale_log2);
      m = mn;
      l *= alpha;
    }
    const float mc = m * scale_log2;
    float ps = 0.f;
    bf16x8 pn[2][2];
    auto exps = [&](int j) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int kh = j >> 2, rr = (j & 3) * 4 + e;
        // raw v_exp_f32 (arguments <= RESCALE_THR; underflow to 0 is what we want)
        const float p = __builtin_amdgcn_exp2f(fmaf(sc[kh][rr], scale_log2, -mc));
        ps += p;
        pn[kh][rr >> 3][rr & 7] = f2bf(p);
      }
    };
    if (kt > 0) {
      second_product(kt - 1, exps);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) exps(j);
    }
    l += ps;
    if (rescale) {   // (O has the page before by now, which the old maximum scaled)
#pragma unroll
      for (int db = 0; db < 4; ++db) o[db] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) pf[i >> 1][i & 1] = pn[i >> 1][i & 1];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  second_product(n_kt - 1, [](int) {});

  l += __shfl_xor(l, 32, 64);
  if (t < T.n) {
    const float inv = 1.f / l;
    bf16* op = out + (size_t)row * ldo + h * HD + 4 * hh;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {  // regs 4g4..4g4+3 = d 32db + 8g4 + 4hh + 0..3
        bf16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = f2bf(o[db][4 * g4 + j] * inv);
        *reinterpret_cast<bf16x4*>(op + 32 * db + 8 * g4) = v;
      }
  }
}

template <int G, int NW>
int launch2(const bf16* q, int ldq, const bf16* kc, const bf16* vc, const int* bt, int bt_stride,
            const Tile* tiles, int n_tiles, int Hkv, float scale, bf16* out, int ldo,
            hipStream_t st) {
  const float sl2 = scale * 1.4426950408889634f;
  hipLaunchKernelGGL((flash_prefill2_kernel<G, NW>), dim3(n_tiles * Hkv), dim3(64 * NW), 0, st, q, ldq, kc,
                     vc, bt, bt_stride, tiles, n_tiles, Hkv, sl2, out, ldo);
  P2P_CHECK_LAUNCH();
}

}  // namespace

// v2 entry: tiles of at most `tile` tokens, 256 / (Hq/Hkv) (p2p_flash_prefill_tile) or fewer, otherwise as
// p2p_flash_prefill.  K/V pages must be whole 64-key pages of the block table.
P2P_API int p2p_flash_prefill_tile(int Hq, int Hkv) {
  if (Hkv <= 0 || Hq % Hkv) return 0;
  const int G = Hq / Hkv;
  return (G == 1 || G == 2 || G == 4 || G == 8) ? 256 / G : 0;
}

P2P_API int p2p_flash_prefill2(const void* q, int ldq, const void* kc, const void* vc,
                               const int* bt, int bt_stride, const int* tiles, int n_tiles,
                               int Hq, int Hkv, int head_dim, float scale, void* out, int ldo,
                               int tile, void* stream) {
  if (head_dim != HD || Hkv <= 0 || Hq % Hkv || tile < 1 || tile > p2p_flash_prefill_tile(Hq, Hkv)) return 1;
  if (n_tiles <= 0) return 0;
  auto Q = (const bf16*)q;
  auto K = (const bf16*)kc;
  auto V = (const bf16*)vc;
  auto T = (const Tile*)tiles;
  auto O = (bf16*)out;
  auto st = (hipStream_t)stream;
  const bool narrow = tile * (Hq / Hkv) <= 128;   // four waves hold the tile
#define FLASH2(G, NW) launch2<G, NW>(Q, ldq, K, V, bt, bt_stride, T, n_tiles, Hkv, scale, O, ldo, st)
  switch (Hq / Hkv) {
    case 1: return narrow ? FLASH2(1, 4) : FLASH2(1, 8);
    case 2: return narrow ? FLASH2(2, 4) : FLASH2(2, 8);
    case 4: return narrow ? FLASH2(4, 4) : FLASH2(4, 8);
    case 8: return FLASH2(8, 8);
    default: return 2;
  }
#undef FLASH2
}

// tiles: int32 [n_tiles, 4] = (first row, n tokens <= 16, sequence, first position);
// n = 0 marks a padding tile (a captured prefill graph launches a fixed tile count);
// a tile's rows are consecutive positions of one sequence whose K/V (positions
// 0 .. pos0+n-1) are already in the paged cache.  head_dim must be 128.
P2P_API int p2p_flash_prefill(const void* q, int ldq, const void* kc, const void* vc,
                              const int* bt, int bt_stride, const int* tiles, int n_tiles,
                              int Hq, int Hkv, int head_dim, float scale, void* out, int ldo,
                              void* stream) {
  if (head_dim != HD || Hkv <= 0 || Hq % Hkv) return 1;
  if (n_tiles <= 0) return 0;
  auto Q = (const bf16*)q;
  auto K = (const bf16*)kc;
  auto V = (const bf16*)vc;
  auto T = (const Tile*)tiles;
  auto O = (bf16*)out;
  auto st = (hipStream_t)stream;
  switch (Hq / Hkv) {
    case 1: return launch<1>(Q, ldq, K, V, bt, bt_stride, T, n_tiles, Hkv, scale, O, ldo, st);
    case 2: return launch<2>(Q, ldq, K, V, bt, bt_stride, T, n_tiles, Hkv, scale, O, ldo, st);
    case 4: return launch<4>(Q, ldq, K, V, bt, bt_stride, T, n_tiles, Hkv, scale, O, ldo, st);
    case 8: return launch<8>(Q, ldq, K, V, bt, bt_stride, T, n_tiles, Hkv, scale, O, ldo, st);
    default: return 2;
  }
}
