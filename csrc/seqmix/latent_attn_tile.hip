// Latent attention for prompts: the same inputs and outputs as latent_attn_mfma_k (bf16 activations,
// fp32 scores / softmax / sums), with key tiles that four wavefronts share.
//
// All heads attend to the same latents, which are keys and values at once.  A workgroup owns 64 (row,
// head) pairs -- 64 / HS consecutive rows x HS heads -- and walks the union of their windows 32 latents at
// a time; a tile is copied straight from the cache into LDS (attn_tile.h) while the one before is used, and
// stays there row by row for both products:
//   S^T[32 keys x 16 pairs] = C . Q^T      a wavefront for its own 16 pairs, Q in registers
//   online softmax in the accumulator layout (see window_attn_tile.hip), weights to LDS
//   O[64 pairs x rank / 4] += P . C         a wavefront for its quarter of the columns, C read transposed
// The second product is cut by columns and not by pairs: a wavefront then reads a quarter of the tile
// and 4 KB of weights instead of the whole tile, and one barrier per tile pays for it.
//
// What bounds it: LDS reads, 32 KB for the first product and 12 KB for the second per wavefront and tile
// at rank 512, and the copies; two workgroups fit a CU as long as a wavefront keeps to 256 registers (a
// spill's reload would wait for the copies: 292 us instead of 128).  16 heads, rank 512, 2048 rows: 152 us
// (450 TFLOP/s; 133 with a maximum that lagged, see window_attn_tile.hip) against 706 us for latent_attn_mfma_k; a window
// of 256: 45 against 184; 32 heads of rank 256 143 against 456.
#include "attn_tile.h"
#include "latent_attn.h"
using namespace sm;

#define LOG2E_ 1.4426950408889634f
#define NO_KEY_YET -1e30f   // running maximum of a pair that has seen no key

template <int NT2>  // rank padded to NT2 * 32
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
latent_attn_tile_k(LatentArgs a) {
  constexpr int RP = NT2 * 32, KT = 32, PC = RP / 8, MC = PC < 16 ? PC - 1 : 15;
  constexpr int CT = NT2 / 2;                 // 16-wide column tiles of a wavefront
  constexpr int STAGE = KT * RP;              // bf16 per stage
  extern __shared__ __align__(16) unsigned short lds[];   // [2][KT latents]
  __shared__ __align__(16) unsigned short sP[64 * KT];    // weights [pair][slot], see read_keys_by_channel
  __shared__ __align__(16) float sAl[64];                 // rescale factors of this tile, then the sums
  __shared__ int sUp[4], sBad[4];                         // wavefront w's pairs are rescaled; its sums are not finite
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), n16 = lane & 15, quad = lane >> 4;
  const int hg = (a.H + a.HS - 1) / a.HS, at = folded_block(), unit = a.U - 1 - at / hg, h0 = (at % hg) * a.HS;
  const int r0 = a.units[2 * unit], nr = a.units[2 * unit + 1];
  const int rank = a.rank, page = a.page, win = a.win;
  // this lane's pair (as a column of S^T)
  const int prow = (wave * 16 + n16) / a.HS, ph = h0 + n16 % a.HS;
  const bool pvalid = prow < nr && ph < a.H;
  const int ppos = pvalid ? a.pos[r0 + prow] : -1;
  const int* pages = a.bt + (size_t)a.row_ent[r0] * a.max_pages;
  const int p_lo = a.pos[r0], p_hi = a.pos[r0 + nr - 1], w_lo = max(0, p_lo - win + 1);
  // tiles start at multiples of KT, so that each lies in one page
  int i_lo = w_lo / KT, i_hi = p_hi / KT;
  if (a.splits > 1) {   // this workgroup's run of them
    const int per = (i_hi - i_lo + a.splits) / a.splits;
    i_lo += blockIdx.y * per;
    i_hi = min(i_hi, i_lo + per - 1);
  }

  // Copies of a tile: thread t takes 16-byte pieces t, t + 256, ..  Numbers beyond the rank (which meet zero
  // queries, or columns that are not written) are some numbers of the same row; a tile that reaches over
  // the windows' ends takes their first (last) row again there.
  constexpr int CC = KT * PC / 256;
  const unsigned lds0 = lds_address(lds) + wave * 1024;
  auto copy_tile = [&](int i, int st, int pg) {
    const int j0 = i * KT, lo = max(w_lo - j0, 0), hi = min(p_hi - j0, KT - 1);
    const char* src = (const char*)a.cache + ((size_t)uniform(pg) * page + j0 % page) * rank * 2;
    const unsigned dst = lds0 + st * STAGE * 2;
    int tid = threadIdx.x;
    if (NT2 == 16) again(tid);
#pragma unroll
    for (int c = 0; c < CC; c++) {
      // (at 64 pieces a row is one wavefront's and its number uniform)
      const int r = c * (256 / PC) + (PC >= 64 ? wave * 64 / PC : tid / PC);
      const int c8 = ((tid % PC) ^ swz(r, MC)) * 8;
      copy_lds16_at(src, (min(max(r, lo), hi) * rank + (c8 < rank ? c8 : 0)) * 2, dst + c * 4096);
    }
  };

  // queries in registers (zero rows for unused pairs, zero columns beyond the rank)
  bf16x8 qf[NT2];
#pragma unroll
  for (int kk = 0; kk < NT2; kk++) {
    const int c8 = kk * 32 + quad * 8;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (pvalid && c8 < rank) v = *(const uint4*)(a.qa + (size_t)ph * a.sqh + (size_t)(r0 + prow) * a.sqr + c8);
    qf[kk] = __builtin_bit_cast(bf16x8, v);
  }
  const float sl2 = a.scale * LOG2E_;
  float m_run = pvalid ? NO_KEY_YET : 0.0f;   // in powers of two
  float l_part = 0.0f;
  f32x4 acc[4][CT];   // pairs 16 m + quad * 4 + e, columns (wave * CT + t) * 16 + n16
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int t = 0; t < CT; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  int next_page = 0;
  if (i_lo <= i_hi) {
    copy_tile(i_lo, 0, pages[i_lo * KT / page]);
    if (i_lo < i_hi) next_page = pages[(i_lo + 1) * KT / page];
  }
  int st = 0;
  for (int i = i_lo; i <= i_hi; i++, st ^= 1) {
    tile_wait();
    __syncthreads();   // the tile has landed; the other stage and the weights are free
    // (the page after next is looked up now and not touched before the next wait: its use would wait
    // for the copies too)
    if (i < i_hi) copy_tile(i + 1, st ^ 1, next_page);
    if (i + 2 <= i_hi) next_page = pages[(i + 2) * KT / page];
    const unsigned short* sC = lds + st * STAGE;
    int ln = lane;
    if (NT2 == 16) again(ln);
    const int n16 = ln & 15, quad = ln >> 4;
    const int jl = i * KT + quad * 4;   // this lane's keys: jl + sub * 16 + e
    f32x4 s[2];
    s[0] = s[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int KB = NT2 < 8 ? NT2 : NT2 == 8 ? 8 : 4;   // reads in flight together (what the registers hold)
#pragma unroll
    for (int k0 = 0; k0 < NT2; k0 += KB) {
      bf16x8 kf[2][KB];
#pragma unroll
      for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int sub = 0; sub < 2; sub++) {
          const int r = sub * 16 + n16, piece = ((k0 + kk) * 4 + quad) ^ swz(r, MC);
          kf[sub][kk] = __builtin_bit_cast(bf16x8, *(const uint4*)(sC + (r * PC + piece) * 8));
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < KB; kk++)
#pragma unroll
        for (int sub = 0; sub < 2; sub++)
          s[sub] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[sub][kk], qf[k0 + kk], s[sub], 0, 0, 0);
      if (NT2 == 16) __builtin_amdgcn_sched_barrier(0);
    }
    const bool fresh = m_run == NO_KEY_YET;
    const float base = fresh ? 0.0f : m_run;
#pragma unroll
    for (int sub = 0; sub < 2; sub++)
#pragma unroll
      for (int e = 0; e < 4; e++) s[sub][e] = fmaf(s[sub][e], sl2, -base);
    if (i * KT + KT - 1 > p_lo || i * KT <= p_hi - win) {   // some key is out of some row's sight
      const int from = ppos - win + 1 - jl, to = ppos + 1 - jl;
#pragma unroll
      for (int sub = 0; sub < 2; sub++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int k = sub * 16 + e;
          if (k < from || k >= to) s[sub][e] = -INFINITY;
        }
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int sub = 0; sub < 2; sub++)
#pragma unroll
      for (int e = 0; e < 4; e++) tmax = fmaxf(tmax, s[sub][e]);
    const bool rescale = __any(tmax > (fresh ? -INFINITY : 0.0f));
    if (rescale) {
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const bool none = fresh && tmax == -INFINITY;
      const float up = none ? 0.0f : fresh ? tmax : fmaxf(tmax, 0.0f);
      const float alpha = fresh ? 1.0f : exp2_(-up);   // a fresh pair's sums are zero
      m_run = none ? NO_KEY_YET : base + up;
      l_part *= alpha;
#pragma unroll
      for (int sub = 0; sub < 2; sub++) s[sub] -= up;
      if (quad == 0) sAl[wave * 16 + n16] = alpha;
    }
    if (lane == 0) sUp[wave] = rescale;
    f32x8 pw;
    float psum = 0.0f;   // of the weights as the product has them
#pragma unroll
    for (int sub = 0; sub < 2; sub++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        pw[sub * 4 + e] = exp2_(s[sub][e]);   // 0 for keys out of sight
      }
    const bf16x8 pb = to_bf16(pw);
#pragma unroll
    for (int e = 0; e < 8; e++) psum += (float)pb[e];
    l_part += psum;
    *(bf16x8*)(sP + (wave * 16 + n16) * KT + quad * 8) = pb;
    __syncthreads();   // the weights are in LDS
    const int4 up4 = *(const int4*)sUp;
    const int ups[4] = {up4.x, up4.y, up4.z, up4.w};
    bf16x8 pf[4];
#pragma unroll
    for (int m = 0; m < 4; m++) pf[m] = *(const bf16x8*)(sP + (m * 16 + n16) * KT + quad * 8);
#pragma unroll
    for (int m = 0; m < 4; m++)
      if (uniform(ups[m])) {
        const f32x4 al = *(const f32x4*)(sAl + m * 16 + quad * 4);
#pragma unroll
        for (int t = 0; t < CT; t++) acc[m][t] *= al;
      }
    constexpr int VB = CT < 4 ? CT : 4;
#pragma unroll
    for (int t0 = 0; t0 < CT; t0 += VB) {
      bf16x8 vf[VB];
#pragma unroll
      for (int t = 0; t < VB; t++) vf[t] = read_keys_by_channel<PC>(sC, 0, (wave * CT + t0 + t) * 16, ln);
#pragma unroll
      for (int t = 0; t < VB; t++)
#pragma unroll
        for (int m = 0; m < 4; m++)
          acc[m][t0 + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[m], vf[t], acc[m][t0 + t], 0, 0, 0);
      if (NT2 == 16) __builtin_amdgcn_sched_barrier(0);
    }
  }
  float z = 0.0f;
#pragma unroll
  for (int m = 0; m < 4; m++)
#pragma unroll
    for (int t = 0; t < CT; t++) not_finite(acc[m][t], z);
  const bool bad = __any(z != z);
  if (lane == 0) sBad[wave] = bad;
  __syncthreads();   // (and the last tile's factors have been read)
  if (__builtin_expect(uniform(sBad[0] | sBad[1] | sBad[2] | sBad[3]), 0)) {   // see not_finite()
#pragma unroll 1
    for (int m = wave * 16; m < wave * 16 + 16; m++) {
      const int row = r0 + m / a.HS, h = h0 + m % a.HS;
      if (m / a.HS >= nr || h >= a.H) continue;
      const int p = a.pos[row];
      PairSums<RP / 64> sums;
      sums.begin(a.sink ? a.sink[h] : 0.0f, a.sink && blockIdx.y == 0);
#pragma unroll 1
      for (int j = max(i_lo * KT, max(0, p - win + 1)); j <= min(p, i_hi * KT + KT - 1); j++) {
        const bf16* c = a.cache + ((size_t)pages[j / page] * page + j % page) * rank;
        sums.add(wave_dot(a.qa + (size_t)h * a.sqh + (size_t)row * a.sqr, c, rank) * a.scale, c, rank);
      }
      float* rec = a.part + (((size_t)unit * hg + at % hg) * a.splits + blockIdx.y) * 64 * (RP + 2) + m * (RP + 2);
      const float f = a.splits > 1 ? 1.0f : sums.l != 0.0f ? 1.0f / sums.l : 0.0f;
#pragma unroll
      for (int t = 0; t < RP / 64; t++) {
        const int c = t * 64 + lane;
        if (c >= rank) continue;
        if (a.splits > 1) rec[c] = sums.o[t];
        else a.out[(size_t)h * a.soh + (size_t)row * a.sor + c] = __float2bfloat16(sums.o[t] * f);
      }
      if (a.splits > 1 && lane == 0) rec[RP] = sums.m, rec[RP + 1] = sums.l;
    }
    return;
  }
  float l = l_part + __shfl_xor(l_part, 16, 64);
  l += __shfl_xor(l, 32, 64);
  m_run *= 1.0f / LOG2E_;   // natural from here on
  // the sink joins the finished sums (see window_attn_tile.hip)
  float sf = 1.0f;          // rescales the sums of this lane's pair
  int pair = threadIdx.x & 15;
  again(pair);              // (its row and head are not kept in registers until here)
  if (a.sink && blockIdx.y == 0 && (wave * 16 + pair) / a.HS < nr && h0 + pair % a.HS < a.H) {
    const float sink = a.sink[h0 + pair % a.HS], m = fmaxf(m_run, sink);
    sf = expf(m_run - m);
    l = l * sf + expf(sink - m);
    m_run = m;
  }
  if (quad == 0) sAl[wave * 16 + n16] = a.splits > 1 ? sf : l != 0.0f ? sf / l : 0.0f;
  __syncthreads();
  if (a.splits > 1) {
    // partial record of this run: [64 pairs][RP + 2] = unnormalised sums, running max (natural), sum
    float* rec = a.part + (((size_t)unit * hg + at % hg) * a.splits + blockIdx.y) * 64 * (RP + 2);
    if (quad == 0) {
      rec[(wave * 16 + n16) * (RP + 2) + RP] = m_run;
      rec[(wave * 16 + n16) * (RP + 2) + RP + 1] = l;
    }
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const f32x4 f = *(const f32x4*)(sAl + m * 16 + quad * 4);
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int t = 0; t < CT; t++)
          rec[(m * 16 + quad * 4 + e) * (RP + 2) + (wave * CT + t) * 16 + n16] = acc[m][t][e] * f[e];
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const f32x4 inv = *(const f32x4*)(sAl + m * 16 + quad * 4);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int pr = m * 16 + quad * 4 + e, mr = pr / a.HS, mh = h0 + pr % a.HS;
      if (mr < nr && mh < a.H) {
        bf16* o = a.out + (size_t)mh * a.soh + (size_t)(r0 + mr) * a.sor;
#pragma unroll
        for (int t = 0; t < CT; t++) {
          const int c = (wave * CT + t) * 16 + n16;
          if (c < rank) o[c] = __float2bfloat16(acc[m][t][e] * inv[e]);
        }
      }
    }
  }
}

template <int NT2>
static int launch_tile(const LatentArgs& a, hipStream_t st) {
  const size_t shm = (size_t)2 * 32 * NT2 * 32 * 2;
  if (shm > 32 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)latent_attn_tile_k<NT2>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL((latent_attn_tile_k<NT2>), dim3(a.U * ((a.H + a.HS - 1) / a.HS), a.splits), dim3(256), shm,
                     st, a);
  return (int)hipGetLastError();
}

int latent_attn_tile(const LatentArgs& a, hipStream_t st) {
  if (a.page < 32 || a.page % 32) return (int)hipErrorInvalidValue;
  const int n = (a.rank + 31) / 32;
  return n <= 2 ? launch_tile<2>(a, st) : n <= 4 ? launch_tile<4>(a, st) : n <= 8 ? launch_tile<8>(a, st)
                                                                                  : launch_tile<16>(a, st);
}
