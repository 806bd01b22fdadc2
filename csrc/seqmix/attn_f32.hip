// Attention in fp32 on the fp32 matrix instruction: float32 models' grouped-query window attention
// (window_attn_k has the options and how blocks and kept tokens join the keys) and latent attention
// (one key/value head whose keys and values are the same cached row).
//
// A workgroup owns 16 (row, head) pairs of one key/value head -- 16 / HS consecutive rows x HS heads -- and
// its four wavefronts take every fourth tile of 16 keys, each with a softmax of its own; they are merged
// in LDS at the end.  Per tile, with v_mfma_f32_16x16x4_f32:
//   S^T[16 keys x 16 pairs] = K . Q^T     keys from the cache as 16-byte pieces: a lane's four numbers
//                                         are one k index of four products
//   O[16 pairs x V]        += P . V       a lane's four weights are the k indices of four products, its
//                                         16 bytes of a value row the column of four output tiles
// so neither operand goes through LDS (only the queries do), and no wavefront waits for another.
// The instruction takes 32 cycles for 4 keys or channels, four times what reading its operands takes: at
// rank 512 a tile is 8192 cycles of products.
//
// Bound by the products where there are enough pairs, by the wait for a tile's operands where a SIMD has one
// wavefront.  Two prompts of 389 and 117 rows, 8 heads: latents of 512 numbers 114 us against 4330 us for
// latent_attn_k (one workgroup per row, scalar products); 8 heads of 128 on 2, capped and penalised, 47
// against 300 for window_attn_k.
#include "attn_tile.h"
using namespace sm;

struct AttnF32Args {
  const float* q;
  long sqh, sqr, sqm;      // strides of heads, rows and maps
  const float* pool;
  int ldpool, vbase;       // a pool row: keys of G * maps heads from 0, values of G heads from vbase
  const int* bt;
  int max_pages;
  const int *row_ent, *pos, *units;
  const float* sink;
  float scale;
  int win;
  float* out;
  long soh, sor, som;
  int U, H, G, D, V, page, HS, splits;
  float* part;
  float out_scale, cap;
  const float *r1, *r2;
  const float* gate;
  int ldg, gate_pc;
  const float* blk;
  int P, keep, maps;
};

__device__ __forceinline__ float out_factor(const AttnF32Args& a, int row, int h, int c) {
  if (!a.gate) return a.out_scale;
  return a.out_scale * sigmoidf_(a.gate[(size_t)row * a.ldg + (a.gate_pc ? (size_t)h * a.V + c : h)]);
}

template <int NB>  // value channels in blocks of 64
__global__ void __launch_bounds__(256)
attn_f32_k(AttnF32Args a) {
  constexpr int VP = NB * 64;
  extern __shared__ __align__(16) float smem[];   // queries [16][LDQ], at the end sums [16][VP]
  __shared__ float sM[5][16], sL[5][16];          // per wavefront, then all together
  __shared__ int sBad[4];                         // a wavefront's sums are not finite
  const int tid = threadIdx.x, lane = tid & 63, n16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int HG = a.H / a.G, hblocks = (HG + a.HS - 1) / a.HS;
  const int unit = a.U - 1 - blockIdx.x;   // the last rows see the most keys
  const int gk = blockIdx.y / hblocks, hb0 = (blockIdx.y % hblocks) * a.HS, g = gk / a.maps, map = gk % a.maps;
  const int r0 = a.units[2 * unit], nr = a.units[2 * unit + 1];
  const int D = a.D, V = a.V, page = a.page, win = a.win, DP = (D + 15) & ~15, LDQ = DP + 4;
  const int koff = gk * D, voff = a.vbase + g * V;
  const int prow = n16 / a.HS, phs = hb0 + n16 % a.HS;
  const bool pvalid = prow < nr && phs < HG;
  const int ph = g * HG + min(phs, HG - 1), ppos = pvalid ? a.pos[r0 + prow] : -1;
  const int* pages = a.bt + (size_t)a.row_ent[r0] * a.max_pages;
  const int p_hi = a.pos[r0 + nr - 1], w_lo = max(0, a.pos[r0] - win + 1);
  // places 0 .. nb-1 are blocks (all that the group's last row sees) or the kept tokens before the
  // group's first window, place u >= nb is token u + shift
  int nb = 0, pnb = 0, SB = 1;
  if (a.blk) {
    nb = max(0, p_hi - win + 1) / a.P;
    pnb = pvalid ? max(0, ppos - win + 1) / a.P : 0;   // blocks this lane's row sees
    SB = (page + a.P - 1) / a.P;
  } else {
    nb = min(a.keep, w_lo);
  }
  const int shift = w_lo - nb, last = p_hi - shift;
  int t_lo = 0, t_hi = last / 16 + 1;   // tiles
  if (a.splits > 1) {
    const int per = (t_hi + a.splits - 1) / a.splits;
    t_lo = blockIdx.z * per;
    t_hi = min(t_hi, t_lo + per);
  }
  auto key_row = [&](int u) -> const float* {   // places past the last one: its row (their weights are zero)
    u = min(u, last);
    if (a.blk && u < nb) {
      const int t = u * a.P + a.P - 1;
      return a.blk + ((size_t)pages[t / page] * SB + (t % page) / a.P) * a.ldpool;
    }
    const int j = u < nb ? u : u + shift;
    return a.pool + ((size_t)pages[j / page] * page + j % page) * a.ldpool;
  };
  for (int i = tid; i < 16 * (DP / 4); i += 256) {
    const int m = i / (DP / 4), c = i % (DP / 4) * 4, mr = m / a.HS, ms = hb0 + m % a.HS;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (mr < nr && ms < HG && c < D)
      v = *(const f32x4*)(a.q + (g * HG + ms) * a.sqh + (r0 + mr) * a.sqr + map * a.sqm + c);
    *(f32x4*)(smem + m * LDQ + c) = v;
  }
  float m_run = pvalid ? -1e30f : 0.0f, l_part = 0.0f;
  const float pr1 = (pvalid && a.r1) ? a.r1[ph] : 0.0f, pr2 = (pvalid && a.r1) ? a.r2[ph] : 0.0f;
  f32x4 acc[NB * 4];   // pairs quad * 4 + e, column (t / 4) * 64 + n16 * 4 + t % 4
#pragma unroll
  for (int t = 0; t < NB * 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();

  const float* krow = t_lo + wave < t_hi ? key_row((t_lo + wave) * 16 + n16) : nullptr;
  for (int ti = t_lo + wave; ti < t_hi; ti += 4) {
    const int u0 = ti * 16;
    const float* nxt = ti + 4 < t_hi ? key_row(u0 + 64 + n16) : nullptr;
    // the values of keys quad * 4 + e
    const float* vrow[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
      vrow[e] = (const float*)__shfl((unsigned long long)krow, quad * 4 + e, 64) + voff;
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
    const float* kp = krow + koff;
    const float* qp = smem + n16 * LDQ + quad * 4;
#pragma unroll 8
    for (int c = 0; c < DP; c += 16) {
      // beyond D: the key's start (D may be less than the 16 numbers of a step), which meets zeros
      const f32x4 kv = *(const f32x4*)(kp + (c + quad * 4 < D ? c + quad * 4 : 0));
      const f32x4 qv = *(const f32x4*)(qp + c);   // zero beyond D
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[0], qv[0], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[1], qv[1], s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[2], qv[2], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[3], qv[3], s1, 0, 0, 0);
    }
    // scores of pair n16 at places u0 + quad * 4 + e
    float sv[4], tmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int u = u0 + quad * 4 + e, jt = u < nb ? u : u + shift;
      bool ok = pvalid && u <= last;
      if (a.blk) ok = ok && (u < nb ? u < pnb : jt <= ppos && jt > ppos - win);
      else ok = ok && jt <= ppos && (jt > ppos - win || jt < a.keep);
      float v = -INFINITY;
      if (ok) {
        v = (s0[e] + s1[e]) * a.scale;
        if (a.cap > 0.0f) v = a.cap * tanhf(v / a.cap);
        if (a.r1) v -= pr1 * log1pf(pr2 * (float)(ppos - jt));
      }
      sv[e] = v;
      tmax = fmaxf(tmax, v);
    }
    if (__any(tmax > m_run + 8.0f)) {   // the running maximum follows in strides of e^8
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m_run, tmax), alpha = expf(m_run - m_new);
      m_run = m_new;
      l_part *= alpha;
      float al[4];
#pragma unroll
      for (int e = 0; e < 4; e++) al[e] = __shfl(alpha, quad * 4 + e, 64);
#pragma unroll
      for (int t = 0; t < NB * 4; t++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[t][e] *= al[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      sv[e] = expf(sv[e] - m_run);   // exp(-inf) = 0 for places out of sight
      l_part += sv[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int b = 0; b < NB; b++) {   // columns beyond V are not written
        const int c = b * 64 + n16 * 4;
        const f32x4 vv = *(const f32x4*)(vrow[e] + (c < V ? c : 0));
#pragma unroll
        for (int t = 0; t < 4; t++)
          acc[b * 4 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[e], vv[t], acc[b * 4 + t], 0, 0, 0);
      }
    krow = nxt;
  }
  // the wavefronts' sums under their common maximum, one after the other; the sink (of the first run) is a fifth
  float l = l_part + __shfl_xor(l_part, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (quad == 0) {
    sM[wave][n16] = m_run;
    sL[wave][n16] = l;
  }
  float z = 0.0f;
#pragma unroll
  for (int t = 0; t < NB * 4; t++) not_finite(acc[t], z);
  const bool bad = __any(z != z);
  if (lane == 0) sBad[wave] = bad;
  __syncthreads();   // (and every wavefront is past its queries)
  if (__builtin_expect(uniform(sBad[0] | sBad[1] | sBad[2] | sBad[3]), 0)) {   // see not_finite()
#pragma unroll 1
    for (int m = wave * 4; m < wave * 4 + 4; m++) {
      const int row = r0 + m / a.HS, hs = hb0 + m % a.HS, h = g * HG + hs;
      if (m / a.HS >= nr || hs >= HG) continue;
      const int p = a.pos[row], blocks = a.blk ? max(0, p - win + 1) / a.P : 0;
      PairSums<NB> sums;
      sums.begin(a.sink ? a.sink[h] : 0.0f, a.sink && blockIdx.z == 0);
#pragma unroll 1
      for (int u = t_lo * 16; u < min(t_hi * 16, last + 1); u++) {
        const int j = u < nb ? u : u + shift;
        if (!(a.blk && u < nb ? u < blocks : j <= p && (j > p - win || (!a.blk && j < a.keep)))) continue;
        const float* kr = key_row(u);
        float s = wave_dot(a.q + h * a.sqh + row * a.sqr + map * a.sqm, kr + koff, D) * a.scale;
        if (a.cap > 0.0f) s = a.cap * tanhf(s / a.cap);
        if (a.r1) s -= a.r1[h] * log1pf(a.r2[h] * (float)(p - j));
        sums.add(s, kr + voff, V);
      }
      float* rec = a.part + (((size_t)unit * gridDim.y + blockIdx.y) * a.splits + blockIdx.z) * 16 * (VP + 2) + m * (VP + 2);
#pragma unroll
      for (int t = 0; t < NB; t++) {
        const int c = t * 64 + lane;
        if (c >= V) continue;
        if (a.splits > 1) rec[c] = sums.o[t];
        else a.out[h * a.soh + row * a.sor + map * a.som + c] =
            sums.l != 0.0f ? sums.o[t] / sums.l * out_factor(a, row, h, c) : 0.0f;
      }
      if (a.splits > 1 && lane == 0) rec[VP] = sums.m, rec[VP + 1] = sums.l;
    }
    return;
  }
  if (tid < 16) {
    const bool sunk = a.sink && blockIdx.z == 0 && tid / a.HS < nr && hb0 + tid % a.HS < HG;
    const float sink = sunk ? a.sink[g * HG + hb0 + tid % a.HS] : -INFINITY;
    const float m = fmaxf(fmaxf(fmaxf(sM[0][tid], sM[1][tid]), fmaxf(sM[2][tid], sM[3][tid])), sink);
    float sum = expf(sink - m);
    for (int w = 0; w < 4; w++) sum += sL[w][tid] * expf(sM[w][tid] - m);
    sM[4][tid] = m;
    sL[4][tid] = sum;
  }
  __syncthreads();
  float f[4];
#pragma unroll
  for (int e = 0; e < 4; e++) f[e] = expf(sM[wave][quad * 4 + e] - sM[4][quad * 4 + e]);
  for (int w = 0; w < 4; w++) {
    if (wave == w) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          f32x4* o = (f32x4*)(smem + (quad * 4 + e) * VP + b * 64 + n16 * 4);
          f32x4 v = {acc[b * 4][e] * f[e], acc[b * 4 + 1][e] * f[e], acc[b * 4 + 2][e] * f[e], acc[b * 4 + 3][e] * f[e]};
          if (w > 0) v += *o;
          *o = v;
        }
    }
    __syncthreads();
  }
  float* rec = a.splits > 1 ? a.part + (((size_t)unit * gridDim.y + blockIdx.y) * a.splits + blockIdx.z) * 16 * (VP + 2)
                            : nullptr;
  for (int i = tid; i < 16 * VP; i += 256) {
    const int m = i / VP, c = i % VP, mr = m / a.HS, ms = hb0 + m % a.HS;
    if (mr >= nr || ms >= HG || c >= V) continue;
    if (rec) {
      rec[m * (VP + 2) + c] = smem[i];
      if (c == 0) {
        rec[m * (VP + 2) + VP] = sM[4][m];
        rec[m * (VP + 2) + VP + 1] = sL[4][m];
      }
      continue;
    }
    const float L = sL[4][m];
    const int h = g * HG + ms;
    a.out[h * a.soh + (r0 + mr) * a.sor + map * a.som + c] =
        L != 0.0f ? smem[i] / L * out_factor(a, r0 + mr, h, c) : 0.0f;
  }
}

// merges the runs of a window that is cut (see window_attn_merge_k); one block per (unit, head block, pair)
__global__ void __launch_bounds__(128) attn_f32_merge_k(AttnF32Args a, int VP) {
  __shared__ float sw[65];
  const int HG = a.H / a.G, hblocks = (HG + a.HS - 1) / a.HS;
  const int gk = blockIdx.y / hblocks, hb0 = (blockIdx.y % hblocks) * a.HS, g = gk / a.maps, map = gk % a.maps;
  const int r0 = a.units[2 * blockIdx.x], nr = a.units[2 * blockIdx.x + 1];
  const int m = blockIdx.z, mr = m / a.HS, ms = hb0 + m % a.HS;
  if (mr >= nr || ms >= HG) return;
  const size_t zs = (size_t)16 * (VP + 2);   // stride between runs
  const float* rec = a.part + ((size_t)blockIdx.x * gridDim.y + blockIdx.y) * a.splits * zs + (size_t)m * (VP + 2);
  if (threadIdx.x < 64) {
    const int z = threadIdx.x;
    const float mz = z < a.splits ? rec[z * zs + VP] : -INFINITY;
    float M = mz;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
    const float w = z < a.splits ? expf(mz - M) : 0.0f;
    const float d = wave_sum(z < a.splits ? w * rec[z * zs + VP + 1] : 0.0f);
    sw[z] = w;
    if (z == 0) sw[64] = d;
  }
  __syncthreads();
  const float d = sw[64];
  const int h = g * HG + ms;
  for (int c = threadIdx.x; c < a.V; c += blockDim.x) {
    float num = 0.0f;
    for (int z = 0; z < a.splits; z++) num += sw[z] * rec[z * zs + c];
    a.out[h * a.soh + (r0 + mr) * a.sor + map * a.som + c] = d != 0.0f ? num / d * out_factor(a, r0 + mr, h, c) : 0.0f;
  }
}

static int value_blocks(int V) {
  const int n = (V + 63) / 64;
  return n <= 1 ? 1 : n <= 2 ? 2 : n <= 4 ? 4 : 8;
}
static int head_slots(int HG) {
  int hs = 1;
  while (hs < HG && hs < 16) hs *= 2;
  return hs;
}

template <int NB>
static int launch_f32(const AttnF32Args& a, dim3 grid, hipStream_t st) {
  const size_t queries = (size_t)16 * (((a.D + 15) & ~15) + 4) * 4, sums = (size_t)16 * NB * 64 * 4;
  hipLaunchKernelGGL((attn_f32_k<NB>), grid, dim3(256), queries > sums ? queries : sums, st, a);
  return (int)hipGetLastError();
}

extern "C" {

// 1 when the kernel serves these key and value sizes (and 16-byte aligned rows)
int p2p_sm_attn_f32_ok(int D, int V) { return D >= 4 && V >= 4 && D % 4 == 0 && V % 4 == 0 && D <= 512 && V <= 512; }

// floats of workspace for `splits` runs per window (0 when splits <= 1)
long p2p_sm_attn_f32_ws(int U, int H, int G, int V, int splits, int maps) {
  if (splits <= 1 || G < 1 || H % G) return 0;
  const int HG = H / G, HS = head_slots(HG);
  return (long)U * G * maps * ((HG + HS - 1) / HS) * splits * 16 * (value_blocks(V) * 64 + 2);
}

// units: row groups of at most 16 / HS rows, HS the power of two >= min(H / G, 16)
int p2p_sm_attn_f32(const float* q, long sqh, long sqr, long sqm, const float* pool, int ldpool, int vbase,
                    const int* bt, int max_pages, const int* row_ent, const int* pos, const int* units, int U,
                    const float* sink, float scale, int win, float* out, long soh, long sor, long som, int H, int G,
                    int D, int V, int page, int splits, float* part, float out_scale, float cap, const float* r1,
                    const float* r2, const float* gate, int ldg, int gate_pc, const float* blk, int P, int keep,
                    int maps, hipStream_t st) {
  if (U <= 0) return 0;
  if (H < 1 || G < 1 || H % G || !p2p_sm_attn_f32_ok(D, V) || win < 1 || (r1 && !r2) || cap < 0.0f || keep < 0 ||
      (keep && blk) || maps < 1 || maps > 2 || (maps == 2 && (sink || gate || blk)) || (blk && (P < 1 || r1)) ||
      splits < 1 || splits > 64 || (splits > 1 && !part) || ldpool % 4 || sqh % 4 || sqr % 4 || sqm % 4 || vbase % 4)
    return (int)hipErrorInvalidValue;
  const int HG = H / G, HS = head_slots(HG);
  const AttnF32Args a = {q, sqh, sqr, sqm, pool, ldpool, vbase, bt, max_pages, row_ent, pos, units, sink, scale, win,
                         out, soh, sor, som, U, H, G, D, V, page, HS, splits, part, out_scale, cap, r1, r2, gate, ldg,
                         gate_pc, blk, P, keep, maps};
  const dim3 grid(U, G * maps * ((HG + HS - 1) / HS), splits);
  const int nb = value_blocks(V);
  const int err = nb == 1 ? launch_f32<1>(a, grid, st) : nb == 2 ? launch_f32<2>(a, grid, st)
                : nb == 4 ? launch_f32<4>(a, grid, st) : launch_f32<8>(a, grid, st);
  if (err || splits == 1) return err;
  hipLaunchKernelGGL(attn_f32_merge_k, dim3(grid.x, grid.y, 16), dim3(128), 0, st, a, nb * 64);
  return (int)hipGetLastError();
}

}  // extern "C"
