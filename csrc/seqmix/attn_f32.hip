// Attention in fp32 on the fp32 matrix instruction: float32 models' grouped-query window attention
// (window_attn_k has the options and how blocks and kept tokens join the keys) and latent attention
// (one key/value head whose keys and values are the same cached row).
//
// A workgroup owns 16 (row, head) pairs of one key/value head -- 16 / HS consecutive rows x HS heads.  Per tile of 16
// keys, with v_mfma_f32_16x16x4_f32:
//   S^T[16 keys x 16 pairs] = K . Q^T     keys from the cache as 16-byte pieces: a lane's four numbers
//                                         are one k index of four products
//   O[16 pairs x V]        += P . V       a lane's four weights are the k indices of four products, its
//                                         16 bytes of a value row the column of four output tiles
// so neither operand goes through LDS.  The four wavefronts take every fourth tile each, with a softmax of its own, and are
// merged in LDS at the end (attn_f32_k), or take longer keys and values together, a quarter of the channels each
// (attn_f32_wide_k): a tile of 512 numbers is 8192 cycles of products, which one wavefront would walk through alone
// behind its tile's loads.  Where registers hold them, the next tile's keys and this one's values are asked for ahead of the
// products.  form_of() has the choice.
//
// Bound by a tile's loads (a key load touches 16 half lines) and its products, which overlap only across the two workgroups
// of a CU.  8 heads, us, a wavefront per tile without loads ahead / now: latents of 512, prompts of 389 and 117 rows 101 / 64
// (4330 with latent_attn_k, one workgroup per row, scalar products), one of 2000 rows 953 / 437, single tokens at 300 and
// 90 43 / 22, 16 at 500 42 / 24; 8 heads of 128 on 2, capped, 389 and 117 rows 30 / 30 (300 with window_attn_k), two tokens
// 17 / 15.
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

// What a workgroup has to do: 16 (row, head) pairs of one key/value head, places t_lo * 16 .. t_hi * 16 - 1 of their keys
struct Work {
  int unit, gk, g, map, hb0, HG, r0, nr, nb, shift, last, t_lo, t_hi, SB;
  const int* pages;
};
__device__ __forceinline__ Work find_work(const AttnF32Args& a) {
  Work w;
  w.HG = a.H / a.G;
  const int hblocks = (w.HG + a.HS - 1) / a.HS;
  w.unit = a.U - 1 - blockIdx.x;   // the last rows see the most keys
  w.gk = blockIdx.y / hblocks;
  w.hb0 = (blockIdx.y % hblocks) * a.HS;
  w.g = w.gk / a.maps;
  w.map = w.gk % a.maps;
  w.r0 = a.units[2 * w.unit];
  w.nr = a.units[2 * w.unit + 1];
  w.pages = a.bt + (size_t)a.row_ent[w.r0] * a.max_pages;
  const int p_hi = a.pos[w.r0 + w.nr - 1], w_lo = max(0, a.pos[w.r0] - a.win + 1);
  // places 0 .. nb-1 are blocks (all that the group's last row sees) or the kept tokens before the
  // group's first window, place u >= nb is token u + shift
  w.nb = a.blk ? max(0, p_hi - a.win + 1) / a.P : min(a.keep, w_lo);
  w.SB = a.blk ? (a.page + a.P - 1) / a.P : 1;
  w.shift = w_lo - w.nb;
  w.last = p_hi - w.shift;
  w.t_lo = 0;
  w.t_hi = w.last / 16 + 1;   // tiles
  if (a.splits > 1) {
    const int per = (w.t_hi + a.splits - 1) / a.splits;
    w.t_lo = blockIdx.z * per;
    w.t_hi = min(w.t_hi, w.t_lo + per);
  }
  return w;
}
__device__ __forceinline__ const float* key_row(const AttnF32Args& a, const Work& w, int u) {   // past the last: its row
  u = min(u, w.last);                                                                           // (their weights are zero)
  if (a.blk && u < w.nb) {
    const int t = u * a.P + a.P - 1;
    return a.blk + ((size_t)w.pages[t / a.page] * w.SB + (t % a.page) / a.P) * a.ldpool;
  }
  const int j = u < w.nb ? u : u + w.shift;
  return a.pool + ((size_t)w.pages[j / a.page] * a.page + j % a.page) * a.ldpool;
}

// the pair of a lane: pair n16 of the group
struct Pair {
  bool valid;
  int head, pos, blocks;   // blocks: how many of them the row sees
  float r1, r2;
};
__device__ __forceinline__ Pair find_pair(const AttnF32Args& a, const Work& w, int n16) {
  Pair p;
  const int row = n16 / a.HS, hs = w.hb0 + n16 % a.HS;
  p.valid = row < w.nr && hs < w.HG;
  p.head = w.g * w.HG + min(hs, w.HG - 1);
  p.pos = p.valid ? a.pos[w.r0 + row] : -1;
  p.blocks = p.valid && a.blk ? max(0, p.pos - a.win + 1) / a.P : 0;
  p.r1 = p.valid && a.r1 ? a.r1[p.head] : 0.0f;
  p.r2 = p.valid && a.r1 ? a.r2[p.head] : 0.0f;
  return p;
}
// scores of the pair at places u0 .. u0 + 3 from its products
__device__ __forceinline__ float scores_of(const AttnF32Args& a, const Work& w, const Pair& p, int u0, const f32x4& dot,
                                           float (&sv)[4]) {
  float tmax = -INFINITY;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int u = u0 + e, jt = u < w.nb ? u : u + w.shift;
    bool ok = p.valid && u <= w.last;
    if (a.blk) ok = ok && (u < w.nb ? u < p.blocks : jt <= p.pos && jt > p.pos - a.win);
    else ok = ok && jt <= p.pos && (jt > p.pos - a.win || jt < a.keep);
    float v = -INFINITY;
    if (ok) {
      v = dot[e] * a.scale;
      if (a.cap > 0.0f) v = a.cap * tanhf(v / a.cap);
      if (a.r1) v -= p.r1 * log1pf(p.r2 * (float)(p.pos - jt));
    }
    sv[e] = v;
    tmax = fmaxf(tmax, v);
  }
  return tmax;
}
// The running maximum follows in strides of e^8; sums are rescaled with it and scores become weights
template <int N>
__device__ __forceinline__ void weights_of(float (&sv)[4], float tmax, float& m_run, float& l_part, f32x4 (&acc)[N], int quad) {
  if (__any(tmax > m_run + 8.0f)) {
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax), alpha = expf(m_run - m_new);
    m_run = m_new;
    l_part *= alpha;
    float al[4];
#pragma unroll
    for (int e = 0; e < 4; e++) al[e] = __shfl(alpha, quad * 4 + e, 64);
#pragma unroll
    for (int t = 0; t < N; t++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[t][e] *= al[e];
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    sv[e] = expf(sv[e] - m_run);   // exp(-inf) = 0 for places out of sight
    l_part += sv[e];
  }
}

// the group pair by pair, see not_finite()
template <int NB>
__device__ __forceinline__ void pairs_alone(const AttnF32Args& a, const Work& w, int wave, int lane) {
  constexpr int VP = NB * 64;
  const int koff = w.gk * a.D, voff = a.vbase + w.g * a.V;
#pragma unroll 1
  for (int m = wave * 4; m < wave * 4 + 4; m++) {
    const int row = w.r0 + m / a.HS, hs = w.hb0 + m % a.HS, h = w.g * w.HG + hs;
    if (m / a.HS >= w.nr || hs >= w.HG) continue;
    const int p = a.pos[row], blocks = a.blk ? max(0, p - a.win + 1) / a.P : 0;
    PairSums<NB> sums;
    sums.begin(a.sink ? a.sink[h] : 0.0f, a.sink && blockIdx.z == 0);
#pragma unroll 1
    for (int u = w.t_lo * 16; u < min(w.t_hi * 16, w.last + 1); u++) {
      const int j = u < w.nb ? u : u + w.shift;
      if (!(a.blk && u < w.nb ? u < blocks : j <= p && (j > p - a.win || (!a.blk && j < a.keep)))) continue;
      const float* kr = key_row(a, w, u);
      float s = wave_dot(a.q + h * a.sqh + row * a.sqr + w.map * a.sqm, kr + koff, a.D) * a.scale;
      if (a.cap > 0.0f) s = a.cap * tanhf(s / a.cap);
      if (a.r1) s -= a.r1[h] * log1pf(a.r2[h] * (float)(p - j));
      sums.add(s, kr + voff, a.V);
    }
    float* rec = a.part + (((size_t)w.unit * gridDim.y + blockIdx.y) * a.splits + blockIdx.z) * 16 * (VP + 2) + m * (VP + 2);
#pragma unroll
    for (int t = 0; t < NB; t++) {
      const int c = t * 64 + lane;
      if (c >= a.V) continue;
      if (a.splits > 1) rec[c] = sums.o[t];
      else a.out[h * a.soh + row * a.sor + w.map * a.som + c] =
          sums.l != 0.0f ? sums.o[t] / sums.l * out_factor(a, row, h, c) : 0.0f;
    }
    if (a.splits > 1 && lane == 0) rec[VP] = sums.m, rec[VP + 1] = sums.l;
  }
}

// A wavefront takes every fourth tile of 16 keys on its own.  NK > 0, keys and values of up to 128 numbers: the next tile's
// keys and this one's values are asked for ahead (loads that the compiler can count: no branch around one, or it waits for
// younger ones too); 0: as they are used, with registers for more wavefronts or longer rows
template <int NB, int NK>  // value channels in blocks of 64, key channels in steps of 16
__global__ void __launch_bounds__(256, NK ? 2 : 1)
attn_f32_k(AttnF32Args a) {
  constexpr int VP = NB * 64;
  extern __shared__ __align__(16) float smem[];   // queries [16][LDQ], at the end sums [16][VP]
  __shared__ float sM[5][16], sL[5][16];          // per wavefront, then all together
  __shared__ int sBad[4];                         // a wavefront's sums are not finite
  const int tid = threadIdx.x, lane = tid & 63, n16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Work w = find_work(a);
  const int D = a.D, V = a.V, DP = NK ? NK * 16 : (D + 15) & ~15, LDQ = DP + 4;
  const int koff = w.gk * D, voff = a.vbase + w.g * V;
  const Pair pr = find_pair(a, w, n16);
  for (int i = tid; i < 16 * (DP / 4); i += 256) {
    const int m = i / (DP / 4), c = i % (DP / 4) * 4, mr = m / a.HS, ms = w.hb0 + m % a.HS;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (mr < w.nr && ms < w.HG && c < D)
      v = *(const f32x4*)(a.q + (w.g * w.HG + ms) * a.sqh + (w.r0 + mr) * a.sqr + w.map * a.sqm + c);
    *(f32x4*)(smem + m * LDQ + c) = v;
  }
  float m_run = pr.valid ? -1e30f : 0.0f, l_part = 0.0f;
  f32x4 acc[NB * 4];   // pairs quad * 4 + e, column (t / 4) * 64 + n16 * 4 + t % 4
#pragma unroll
  for (int t = 0; t < NB * 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();

  // The next tile's keys are asked for when this one's are used up, a tile's values before its scores: what a wavefront
  // waits for came out behind the products of the one or the other
  f32x4 kv[NK ? NK : 1];
  auto ask = [&](const float* row) {   // beyond D: the key's start, which meets zeros
#pragma unroll
    for (int i = 0; i < NK; i++) kv[i] = *(const f32x4*)(row + koff + (i * 16 + quad * 4 < D ? i * 16 + quad * 4 : 0));
  };
  const float* krow = NK || w.t_lo + wave < w.t_hi ? key_row(a, w, (w.t_lo + wave) * 16 + n16) : nullptr;
  if (NK) ask(krow);
  for (int ti = w.t_lo + wave; ti < w.t_hi; ti += 4) {
    const int u0 = ti * 16;
    const float* nxt = NK || ti + 4 < w.t_hi ? key_row(a, w, u0 + 64 + n16) : nullptr;
    // the values of keys quad * 4 + e
    const float* vrow[4];
#pragma unroll
    for (int e = 0; e < 4; e++) vrow[e] = (const float*)__shfl((unsigned long long)krow, quad * 4 + e, 64) + voff;
    auto value = [&](int e, int b) {   // columns beyond V are not written
      const int c = b * 64 + n16 * 4;
      return *(const f32x4*)(vrow[e] + (c < V ? c : 0));
    };
    f32x4 vv[4][NB];
    if constexpr (NK > 0) {
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int b = 0; b < NB; b++) vv[e][b] = value(e, b);
    }
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
    const float* qp = smem + n16 * LDQ + quad * 4;
    auto product = [&](const f32x4& k, const f32x4& q) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[0], q[0], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[1], q[1], s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[2], q[2], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[3], q[3], s1, 0, 0, 0);
    };
    if constexpr (NK > 0) {
#pragma unroll
      for (int i = 0; i < NK; i++) product(kv[i], *(const f32x4*)(qp + i * 16));   // (queries: zero beyond D)
      ask(nxt);
    } else {
#pragma unroll 8
      for (int c = 0; c < DP; c += 16)
        product(*(const f32x4*)(krow + koff + (c + quad * 4 < D ? c + quad * 4 : 0)), *(const f32x4*)(qp + c));
    }
    float sv[4];
    const float tmax = scores_of(a, w, pr, u0 + quad * 4, s0 + s1, sv);
    weights_of(sv, tmax, m_run, l_part, acc, quad);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
          if constexpr (NK == 0)
            if (t == 0) vv[e][b] = value(e, b);
          acc[b * 4 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[e], vv[e][b][t], acc[b * 4 + t], 0, 0, 0);
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
  if (__builtin_expect(uniform(sBad[0] | sBad[1] | sBad[2] | sBad[3]), 0)) return pairs_alone<NB>(a, w, wave, lane);
  if (tid < 16) {
    const bool sunk = a.sink && blockIdx.z == 0 && tid / a.HS < w.nr && w.hb0 + tid % a.HS < w.HG;
    const float sink = sunk ? a.sink[w.g * w.HG + w.hb0 + tid % a.HS] : -INFINITY;
    const float m = fmaxf(fmaxf(fmaxf(sM[0][tid], sM[1][tid]), fmaxf(sM[2][tid], sM[3][tid])), sink);
    float sum = expf(sink - m);
    for (int u = 0; u < 4; u++) sum += sL[u][tid] * expf(sM[u][tid] - m);
    sM[4][tid] = m;
    sL[4][tid] = sum;
  }
  __syncthreads();
  float f[4];
#pragma unroll
  for (int e = 0; e < 4; e++) f[e] = expf(sM[wave][quad * 4 + e] - sM[4][quad * 4 + e]);
  for (int u = 0; u < 4; u++) {
    if (wave == u) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          f32x4* o = (f32x4*)(smem + (quad * 4 + e) * VP + b * 64 + n16 * 4);
          f32x4 v = {acc[b * 4][e] * f[e], acc[b * 4 + 1][e] * f[e], acc[b * 4 + 2][e] * f[e], acc[b * 4 + 3][e] * f[e]};
          if (u > 0) v += *o;
          *o = v;
        }
    }
    __syncthreads();
  }
  float* rec = a.splits > 1 ? a.part + (((size_t)w.unit * gridDim.y + blockIdx.y) * a.splits + blockIdx.z) * 16 * (VP + 2)
                            : nullptr;
  for (int i = tid; i < 16 * VP; i += 256) {
    const int m = i / VP, c = i % VP, mr = m / a.HS, ms = w.hb0 + m % a.HS;
    if (mr >= w.nr || ms >= w.HG || c >= V) continue;
    if (rec) {
      rec[m * (VP + 2) + c] = smem[i];
      if (c == 0) {
        rec[m * (VP + 2) + VP] = sM[4][m];
        rec[m * (VP + 2) + VP + 1] = sL[4][m];
      }
      continue;
    }
    const float L = sL[4][m];
    const int h = w.g * w.HG + ms;
    a.out[h * a.soh + (w.r0 + mr) * a.sor + w.map * a.som + c] =
        L != 0.0f ? smem[i] / L * out_factor(a, w.r0 + mr, h, c) : 0.0f;
  }
}

// Longer keys or values (latents): the four wavefronts take all tiles together.  Each has a quarter of the channels for
// the scores, whose partial sums meet in LDS, and every fourth 64 value columns; the weights are the same in all of them,
// so nothing is merged at the end.  Queries, two tiles' quarter of the keys and one of the values are in registers.
template <int NB, int NK>  // value channels in blocks of 64, four or eight; key channels in steps of 64
__global__ void __launch_bounds__(256, 2)
attn_f32_wide_k(AttnF32Args a) {
  constexpr int VP = NB * 64, NV = NB / 4;
  __shared__ f32x4 part[2][4][64];
  __shared__ int sBad[4];
  const int tid = threadIdx.x, lane = tid & 63, n16 = lane & 15, quad = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Work w = find_work(a);
  const int D = a.D, V = a.V, koff = w.gk * D, voff = a.vbase + w.g * V;
  const Pair pr = find_pair(a, w, n16);
  // this lane's channels: 16-number steps 2 wave and the next of every eight
  auto channel = [&](int i) { return ((i >> 1) * 8 + wave * 2 + (i & 1)) * 16 + quad * 4; };
  f32x4 q[NK];
  {
    const int row = min(n16 / a.HS, w.nr - 1);
    const float* qr = a.q + pr.head * a.sqh + (w.r0 + row) * a.sqr + w.map * a.sqm;
#pragma unroll
    for (int i = 0; i < NK; i++) {
      q[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (pr.valid && channel(i) < D) q[i] = *(const f32x4*)(qr + channel(i));
    }
  }
  float m_run = pr.valid ? -1e30f : 0.0f, l_part = 0.0f;
  f32x4 acc[NV * 4];   // pairs quad * 4 + e, column (wave + 4 (t / 4)) * 64 + n16 * 4 + t % 4
#pragma unroll
  for (int t = 0; t < NV * 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 kv[2][NK], vv[4][NV];
  auto ask = [&](const float* row, f32x4 (&k)[NK]) {   // beyond D: the key's start, which meets zeros
#pragma unroll
    for (int i = 0; i < NK; i++) k[i] = *(const f32x4*)(row + koff + (channel(i) < D ? channel(i) : 0));
  };
  auto tile = [&](int ti, const float* krow, const float* nxt, f32x4 (&k)[NK], f32x4 (&kn)[NK], f32x4 (&meet)[4][64]) {
#pragma unroll
    for (int e = 0; e < 4; e++) {   // the values of keys quad * 4 + e
      const float* vrow = (const float*)__shfl((unsigned long long)krow, quad * 4 + e, 64) + voff;
#pragma unroll
      for (int b = 0; b < NV; b++) {   // columns beyond V are not written
        const int c = (wave + 4 * b) * 64 + n16 * 4;
        vv[e][b] = *(const f32x4*)(vrow + (c < V ? c : 0));
      }
    }
    ask(nxt, kn);
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int i = 0; i < NK; i++) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][0], q[i][0], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][1], q[i][1], s1, 0, 0, 0);
      s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][2], q[i][2], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i][3], q[i][3], s1, 0, 0, 0);
    }
    meet[wave][lane] = s0 + s1;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (leaves the loads in flight)
    const f32x4 dot = (meet[0][lane] + meet[1][lane]) + (meet[2][lane] + meet[3][lane]);
    float sv[4];
    const float tmax = scores_of(a, w, pr, ti * 16 + quad * 4, dot, sv);
    weights_of(sv, tmax, m_run, l_part, acc, quad);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int b = 0; b < NV; b++)
#pragma unroll
        for (int t = 0; t < 4; t++)
          acc[b * 4 + t] = __builtin_amdgcn_mfma_f32_16x16x4f32(sv[e], vv[e][b][t], acc[b * 4 + t], 0, 0, 0);
  };
  const float* krow = key_row(a, w, w.t_lo * 16 + n16);
  ask(krow, kv[0]);
  for (int ti = w.t_lo; ti < w.t_hi; ti += 2) {   // (the sums' two places by turns: a barrier lies between a tile's reads
    const float* second = key_row(a, w, ti * 16 + 16 + n16);   // and the next writes there)
    tile(ti, krow, second, kv[0], kv[1], part[0]);
    if (ti + 1 >= w.t_hi) break;
    krow = key_row(a, w, ti * 16 + 32 + n16);
    tile(ti + 1, second, krow, kv[1], kv[0], part[1]);
  }
  float l = l_part + __shfl_xor(l_part, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float z = 0.0f;
#pragma unroll
  for (int t = 0; t < NV * 4; t++) not_finite(acc[t], z);
  const bool bad = __any(z != z);
  if (lane == 0) sBad[wave] = bad;
  __syncthreads();
  if (__builtin_expect(uniform(sBad[0] | sBad[1] | sBad[2] | sBad[3]), 0)) return pairs_alone<NB>(a, w, wave, lane);
  const float sink = a.sink && blockIdx.z == 0 && pr.valid ? a.sink[pr.head] : -INFINITY;
  const float m = fmaxf(m_run, sink), f = expf(m_run - m);
  l = expf(sink - m) + l * f;
  float* rec = a.splits > 1 ? a.part + (((size_t)w.unit * gridDim.y + blockIdx.y) * a.splits + blockIdx.z) * 16 * (VP + 2)
                            : nullptr;
  if (rec && wave == 0 && quad == 0 && pr.valid) {
    rec[n16 * (VP + 2) + VP] = m;
    rec[n16 * (VP + 2) + VP + 1] = l;
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int pair = quad * 4 + e, mr = pair / a.HS, ms = w.hb0 + pair % a.HS;
    const float fe = __shfl(f, pair, 64), le = __shfl(l, pair, 64);
    if (mr >= w.nr || ms >= w.HG) continue;
    const int h = w.g * w.HG + ms, row = w.r0 + mr;
#pragma unroll
    for (int b = 0; b < NV; b++)
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int c = (wave + 4 * b) * 64 + n16 * 4 + t;
        if (c >= V) continue;
        const float v = acc[b * 4 + t][e] * fe;
        if (rec) rec[pair * (VP + 2) + c] = v;
        else a.out[h * a.soh + row * a.sor + w.map * a.som + c] = le != 0.0f ? v / le * out_factor(a, row, h, c) : 0.0f;
      }
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

// The kernel of a shape: attn_f32_k without loads ahead, with them, or attn_f32_wide_k.  us, waves / ahead / wide:
// * up to 128 numbers: ahead.  8 heads of 128 on 2, 400 and 400 rows 29 / 22 / 49, one token at 500 15.3 / 13.3 / 15.6;
// * longer values: wide while there are few groups of rows, whose workgroups share a tile's loads and products; with many
//   they hide each other's waits, and waves that meet at no barrier are ahead.  Groups (before windows are cut into runs),
//   wide / waves: 16 heads, latents of 256, 210 (160 keys) 30 / 36, 320 31 / 35 (564 keys: 92 / 82), 333 (423) 59 / 56, 512 (600) 85 / 78;
//   4 heads of 136 and 200 on 2, 54 (160) 18.6 / 20.4, 84 27 / 29, 200 level, 250 (1500) 122 / 114; 16 on one with keys of 64
//   and values of 256, 40 (130) 16.8 / 18.7, 100 (190) 22.7 / 23.6, (600) 14 % less, 333 (333) 46 / 34;
// * keys above 128 alone: waves.  8 heads of 192 and 128 on 2, 1000 rows 151 / 98, 32 tokens at 500 22.0 / 19.7, at 90 17.2 /
//   14.1, with one key each 7.8 / 9.6;
// * more than 256: wide (what waves would hold does not fit their registers), but for keys alone with many workgroups: 8 heads
//   of 384 and 128 on 2, one token 8.1 / 12.2, 1000 rows 203 / 178.
enum Form { WAVES, AHEAD, WIDE };
static Form form_of(int D, int V, long groups, int splits) {
  if (D > 256 || V > 256) return V <= 256 && groups * splits >= 128 ? WAVES : WIDE;
  if (V > 128) return groups <= (D > 192 ? 256 : D > 128 ? 127 : 95) ? WIDE : WAVES;
  return D > 128 ? WAVES : AHEAD;
}
// value channels of that kernel in blocks of 64
static int value_blocks(int V, Form form) {
  const int n = (V + 63) / 64;
  return form == WIDE ? n <= 4 ? 4 : 8 : n <= 2 ? n : 4;
}
static int head_slots(int HG) {
  int hs = 1;
  while (hs < HG && hs < 16) hs *= 2;
  return hs;
}

template <int NB>
static void launch_waves(const AttnF32Args& a, bool ahead, dim3 grid, hipStream_t st) {
  const int steps = !ahead ? (a.D + 15) / 16 : a.D <= 16 ? 1 : a.D <= 32 ? 2 : a.D <= 64 ? 4 : 8;
  const size_t queries = (size_t)16 * (steps * 16 + 4) * 4, sums = (size_t)16 * NB * 64 * 4;
  const size_t shm = queries > sums ? queries : sums;
  if constexpr (NB <= 2) {
    if (ahead) {
      if (steps == 1) hipLaunchKernelGGL((attn_f32_k<NB, 1>), grid, dim3(256), shm, st, a);
      else if (steps == 2) hipLaunchKernelGGL((attn_f32_k<NB, 2>), grid, dim3(256), shm, st, a);
      else if (steps == 4) hipLaunchKernelGGL((attn_f32_k<NB, 4>), grid, dim3(256), shm, st, a);
      else hipLaunchKernelGGL((attn_f32_k<NB, 8>), grid, dim3(256), shm, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((attn_f32_k<NB, 0>), grid, dim3(256), shm, st, a);
}
template <int NB>
static void launch_wide(const AttnF32Args& a, dim3 grid, hipStream_t st) {
  if (a.D <= 256) hipLaunchKernelGGL((attn_f32_wide_k<NB, 4>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((attn_f32_wide_k<NB, 8>), grid, dim3(256), 0, st, a);
}

extern "C" {

// 1 when the kernel serves these key and value sizes (and 16-byte aligned rows)
int p2p_sm_attn_f32_ok(int D, int V) { return D >= 4 && V >= 4 && D % 4 == 0 && V % 4 == 0 && D <= 512 && V <= 512; }

// floats of workspace for `splits` runs per window (0 when splits <= 1)
long p2p_sm_attn_f32_ws(int U, int H, int G, int D, int V, int splits, int maps) {
  if (splits <= 1 || G < 1 || H % G) return 0;
  const int HG = H / G, HS = head_slots(HG);
  const long groups = (long)U * G * maps * ((HG + HS - 1) / HS);
  return groups * splits * 16 * (value_blocks(V, form_of(D, V, groups, splits)) * 64 + 2);
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
  const Form form = form_of(D, V, (long)grid.x * grid.y, splits);
  const int nb = value_blocks(V, form);
  if (form == WIDE) nb == 4 ? launch_wide<4>(a, grid, st) : launch_wide<8>(a, grid, st);
  else if (nb == 4) launch_waves<4>(a, false, grid, st);
  else if (nb == 2) launch_waves<2>(a, form == AHEAD, grid, st);
  else launch_waves<1>(a, form == AHEAD, grid, st);
  if (const int err = (int)hipGetLastError()) return err;
  if (splits == 1) return 0;
  hipLaunchKernelGGL(attn_f32_merge_k, dim3(grid.x, grid.y, 16), dim3(128), 0, st, a, nb * 64);
  return (int)hipGetLastError();
}

}  // extern "C"
