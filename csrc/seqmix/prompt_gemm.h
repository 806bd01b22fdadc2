// Products of prompts: out[M, N] = x[M, K] . w[N, K]^T (+ bias), bf16 or fp32 with fp32 sums, both operands row-major as the models hold
// them, and what follows the product in its epilogue: a tanh of the columns from tanh_from on (of the rounded result), or the
// gated unit of a feed-forward, whose gate rows and up rows of w a tile takes together (the result is rounded once, after it).
//
// A workgroup owns BM rows x BN columns; WM x WN wavefronts of 16 FM x 16 FN each, WK groups of them that take every WK-th 64
// numbers of K and meet in LDS at the end.  Both operands go to LDS by copies of 8 rows x 128 bytes (whole lines: a CU takes those
// in at 95 KB/us, 16 rows x 64 bytes at 58), 16-byte piece p of a row at p ^ its key, ST stages deep; the next half stage is read
// under the products of the present one, and the copies are issued between products, into the slot that every wavefront has in
// registers.  W is the product's left operand, its rows dealt so that a lane ends with neighbouring columns of one row of out.
//
// What bounds it: below some 1000 rows the copies into LDS (64 x 64: 16 KB for 128 cycles of the matrix cores) and the few
// workgroups, which is why K is cut inside a workgroup (2048 x 8192, 20 rows: 128 workgroups of 32 x 16 with four groups 11.7 us,
// 32 x 32 16.7) and eight wavefronts pay where four leave each SIMD one (128 x 128, 2048 x 8192, 2048 rows: 92 us, eight 79);
// above, LDS: 256 x 256 reads and writes it for as many cycles as the matrix cores take (16384 x 2048, 2048 rows 111 us, 1240
// TFLOP/s; on four wavefronts of 128 x 128, which read a third less, a stage takes 1.42 us for 1.61, but start and end of a tile
// 20 us more).  The code behind the products is run once per tile and comes from memory, so it is kept short: with tanhf() and
// the stores of single numbers unrolled in it, 128 x 128 took 79 us where it takes 67, 256 x 256 60 us where 56.
// us, the library's -> this: 10304 x 2048, 48, 300, 1024, 2048 rows 15.0 -> 12.6, 25.5 -> 20.2, 51 -> 48, 100 -> 84; 2048 x 8192,
// 300 and 2048 rows 32 -> 32, 82 -> 65; 2048 x 2048, 48 and 2048 rows 8.6 -> 5.0, 21.5 -> 18.9.
#pragma once
#include <algorithm>
#include <type_traits>

#include "attn_tile.h"
#include "unit_act.h"
using namespace sm;

struct GemmArgs {
  const void* x;
  const int* rows;      // which rows of x (null: 0 .. M - 1)
  int ldx;
  const void *w, *bias;
  void* out;
  int ldo, M, N, K;     // N: columns of out (a gated unit's w has 2 N rows)
  int tanh_from;
  int act;              // gated units: see unit_act
  float limit, alpha;
  int m_tiles, n_tiles, wide;
};

// at most `pending` stages of L copies each under way
template <int L>
__device__ __forceinline__ void wait_stages(int pending) {
  switch (pending) {
    case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * L) : "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * L) : "memory"); break;
  }
}

template <typename T, int BM, int BN, int WM, int WN, int WK, int ST, bool ACT>
__global__ void __launch_bounds__(64 * WM * WN * WK) prompt_gemm_k(GemmArgs a) {
  typedef std::conditional_t<sizeof(T) == 2, bf16x8, f32x4> Frag;      // 16 bytes of a row
  constexpr int KS = 128 / sizeof(T);                                  // numbers of K per stage
  constexpr int FM = BM / (16 * WM), FN = BN / (16 * WN), WPK = WM * WN;
  constexpr int AI = BM / 8 / WPK, BI = BN / 8 / WPK, L = AI + BI;   // copies of a wavefront per stage
  constexpr int KG = (BM + BN) * 128, STAGE = WK * KG;               // bytes
  constexpr int RUN = (ACT ? 2 : 4) * FN;                            // neighbouring columns of a lane
  static_assert(AI * 8 * WPK == BM && BI * 8 * WPK == BN && FM * 16 * WM == BM && FN * 16 * WN == BN, "tile");
  static_assert(!ACT || FN % 2 == 0, "gate and up");
  static_assert(3 * L < 64 && ST >= 2 && ST <= 5, "counted copies");
  extern __shared__ __align__(16) char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), i16 = lane & 15, k4 = lane >> 4;
  const int kg = wave / WPK, wk = wave % WPK, wm = wk / WN, wn = wk % WN;
  // an XCD's workgroups are neighbours in a list that walks bands of rows, columns outside
  constexpr int GM = 1024 / BM;
  const int nb = a.m_tiles * a.n_tiles, per = nb / 8, over = nb % 8, xcd = blockIdx.x % 8;
  const int tile = (xcd < over ? xcd * (per + 1) : over * (per + 1) + (xcd - over) * per) + blockIdx.x / 8;
  const int band = tile / (GM * a.n_tiles), first = band * GM, gm = min(a.m_tiles - first, GM), in = tile - band * GM * a.n_tiles;
  const int m0 = (first + in % gm) * BM, n0 = in / gm * (ACT ? BN / 2 : BN);
  const int nk = (a.K + KS - 1) / KS, n = (nk + WK - 1) / WK;

  // copies: an address of the wavefront's per stage, a lane's offset that stays
  const char* xs = (const char*)((const T*)a.x + (a.rows ? 0 : (size_t)m0 * a.ldx));
  const char* ws = (const char*)((const T*)a.w + (size_t)n0 * a.K);
  const int p8 = lane & 7, r8 = lane >> 3;
  const bool half = a.K < KS;                  // rows of 64 bytes: their pieces twice, the second half stage is not multiplied
  const int pieces = half ? 3 : 7;
  int at[L];
#pragma unroll
  for (int i = 0; i < AI; i++) {
    const int r = 8 * (wk + WPK * i) + r8;
    const int m = min(m0 + r, a.M - 1);
    at[i] = (a.rows ? a.rows[m] : m - m0) * a.ldx * (int)sizeof(T) + (((p8 ^ (r & 7)) & pieces) << 4);
  }
  auto w_key = [](int r) { return (r & 3) | ((r / RUN) & 1) << 2; };   // r: row among those of a wavefront
#pragma unroll
  for (int i = 0; i < BI; i++) {
    const int r = 8 * (wk + WPK * i) + r8, rw = r % (16 * FN);
    int row = ACT ? r / (16 * FN) * (8 * FN) + rw % (8 * FN) : r;
    row = min(n0 + row, a.N - 1) - n0 + (ACT && rw >= 8 * FN ? a.N : 0);
    at[AI + i] = row * a.K * (int)sizeof(T) + (((p8 ^ w_key(rw)) & pieces) << 4);
  }
  const unsigned lds0 = lds_address(lds) + kg * KG + wk * 1024;
  auto copy = [&](int i, int t) {   // the i-th of this wavefront's copies of stage t
    const unsigned to = lds0 + (t % ST) * STAGE + (i < AI ? i * (WPK * 1024) : BM * 128 + (i - AI) * (WPK * 1024));
    const int kt = WK == 1 ? t : min(t * WK + kg, nk - 1);
    copy_lds16_at((i < AI ? xs : ws) + (size_t)kt * 128, at[i], to);
  };
#pragma unroll
  for (int t = 0; t < ST; t++)
    if (t < n)
#pragma unroll
      for (int i = 0; i < L; i++) copy(i, t);

  // this lane's rows in a stage
  const char* base = lds + kg * KG;
  const int xr = wm * FM * 16 + i16, xk = i16 & 7;
  const int wr = (i16 >> 2) * RUN + (i16 & 3), wkey = (i16 & 3) | ((i16 >> 2) & 1) << 2;
  // Tiles of more products read them one fragment row at a time under the products of the one before (256 x 256, 10304 x 2048,
  // 1500 rows: all at once 60 us, a row at a time 55; 64 x 64, 2048 x 8192, 20 rows 31.6 and 34)
  constexpr bool SPREAD = FM * FN >= 8;
  auto read1 = [&](int t, int ks, int i, Frag(&xf)[FM], Frag(&wf)[FN]) {   // the i-th of FM parts
    const char* s = base + (t % ST) * STAGE;
#pragma unroll
    for (int j = i * FN / FM; j < (i + 1) * FN / FM; j++) {
      const int r = wn * 16 * FN + (ACT && j >= FN / 2 ? 8 * FN + (j - FN / 2) * 4 : j * 4) + wr;
      wf[j] = *(const Frag*)(s + BM * 128 + r * 128 + (((4 * ks + k4) ^ wkey) << 4));
    }
    xf[i] = *(const Frag*)(s + (xr + i * 16) * 128 + (((4 * ks + k4) ^ xk) << 4));
  };
  auto read = [&](int t, int ks, Frag(&xf)[FM], Frag(&wf)[FN]) {
#pragma unroll
    for (int i = 0; i < FM; i++) read1(t, ks, i, xf, wf);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto products = [&](const Frag(&xf)[FM], const Frag(&wf)[FN], auto&& between) {
#pragma unroll
    for (int i = 0; i < FM; i++) {
      if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], xf[i], acc[i][j], 0, 0, 0);
      } else {   // (which four of 16 numbers of K a product takes is free, as long as both operands hold the same)
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[j][e], xf[i][e], acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      between(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto nothing = [](int) {};
  auto meet = [] {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto used_up = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  Frag x0[FM], w0[FN], x1[FM], w1[FN];
  wait_stages<L>(min(ST - 1, n - 1));
  meet();
  __builtin_amdgcn_s_waitcnt(0xc07f);   // (seen by the compiler: no scalar load is under way where the loop begins)
  read(0, 0, x0, w0);
  int t = 0;
  auto half0 = [&](int t) {
    if constexpr (!SPREAD) read(t, 1, x1, w1);
    products(x0, w0, [&](int i) {
      if constexpr (SPREAD) read1(t, 1, i, x1, w1);
    });
    used_up();
  };
  auto half1 = [&](int t, bool more) {
    if constexpr (!SPREAD) read(t + 1, 0, x0, w0);
    products(x1, w1, [&](int i) {
      if constexpr (SPREAD) read1(t + 1, 0, i, x0, w0);
      if (more) {
#pragma unroll
        for (int c = i * L / FM; c < (i + 1) * L / FM; c++) copy(c, t + ST);
      }
    });
  };
  // (stage t + 1 is there, for every wavefront once they met.  One loop for all stages takes 24 registers fewer, which 256
  // columns do not have; 128 x 64, 4096 x 2048, 398 rows are 12.8 us with a loop for the last stages, 15.5 without)
  if constexpr (BM * BN >= 192 * 256) {
    for (; t + 1 < n; t++) {
      const bool more = t + ST < n;
      half0(t);
      wait_stages<L>(more ? ST - 2 : min(ST - 2, n - 2 - t));
      meet();
      half1(t, more);
    }
  } else {
    for (; t + ST < n; t++) {
      half0(t);
      wait_stages<L>(ST - 2);
      meet();
      half1(t, true);
    }
    for (; t + 1 < n; t++) {
      half0(t);
      wait_stages<L>(min(ST - 2, n - 2 - t));
      meet();
      half1(t, false);
    }
  }
  if (WK == 1 || t * WK + kg < nk) {
    read(t, 1, x1, w1);
    products(x0, w0, nothing);
    if (!half) products(x1, w1, nothing);
  }
  if constexpr (WK > 1) {   // the groups' sums, in their order
    used_up();
    __syncthreads();
    f32x4* sx = (f32x4*)lds;
    if (kg > 0)
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) sx[(((kg - 1) * WPK + wk) * FM * FN + i * FN + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 0; g < WK - 1; g++)
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] += sx[((g * WPK + wk) * FM * FN + i * FN + j) * 64 + lane];
  }
  // this lane's columns c0 .. c0 + RUN - 1 of FM rows.  (Little code: a tile runs through it once, from memory)
  const int cw = n0 + wn * 4 * RUN, c0 = cw + k4 * RUN;
  float bias[RUN];
  if (!ACT && a.bias) {
#pragma unroll
    for (int e = 0; e < RUN; e++) bias[e] = ldf((const T*)a.bias, min(c0 + e, a.N - 1));
  }
  const bool tanhs = !ACT && sizeof(T) == 2 && cw + 4 * RUN > a.tanh_from;   // (tanh_ is as exact as bf16 needs)
  if (!a.wide) __syncthreads();   // (LDS is used again)
#pragma unroll
  for (int i = 0; i < FM; i++) {
    alignas(16) T o[RUN];
#pragma unroll
    for (int e = 0; e < RUN; e++) {
      float v = acc[i][e / 4][e % 4];
      if constexpr (ACT) v = unit_act<sizeof(T) == 4>(a.act, v, acc[i][FN / 2 + e / 4][e % 4], a.limit, a.alpha);
      else if (a.bias) v += bias[e];
      stf(o, e, v);
    }
    if constexpr (!ACT && sizeof(T) == 2) if (tanhs) {
#pragma unroll
      for (int e = 0; e < RUN; e++)
        if (c0 + e >= a.tanh_from) stf(o, e, tanh_(ldf(o, e)));
    }
    const int m1 = m0 + wm * FM * 16 + i * 16, m = m1 + i16;
    if (a.wide) {
      T* to = (T*)a.out + (size_t)m * a.ldo + c0;
      constexpr int V = sizeof(T) == 2 && RUN % 8 == 0 ? 8 : 4;   // numbers per store
      if (a.wide >= V) {
#pragma unroll
        for (int e = 0; e < RUN; e += V)
          if (m < a.M && c0 + e < a.N) {
            if constexpr (V * sizeof(T) == 16) *(uint4*)(to + e) = *(const uint4*)(o + e);
            else *(uint2*)(to + e) = *(const uint2*)(o + e);
          }
      } else {
#pragma unroll
        for (int e = 0; e < RUN; e += 4)
          if (m < a.M && c0 + e < a.N) *(uint2*)(to + e) = *(const uint2*)(o + e);
      }
      continue;
    }
    // rows or columns that wide stores do not fit: one number at a time, from the wavefront's own place in LDS
    T* const so = (T*)lds + wk * (64 * RUN);
#pragma unroll
    for (int e = 0; e < RUN; e++) so[(k4 * RUN + e) * 16 + i16] = o[e];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 1
    for (int q = lane; q < 64 * RUN; q += 64) {
      const int r = m1 + q / (4 * RUN), c = cw + q % (4 * RUN);
      if (r < a.M && c < a.N) ((T*)a.out)[(size_t)r * a.ldo + c] = so[q % (4 * RUN) * 16 + q / (4 * RUN)];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

template <typename T, int BM, int BN, int WM, int WN, int WK, int ST>
static int launch_gemm(GemmArgs a, hipStream_t st) {
  a.m_tiles = (a.M + BM - 1) / BM;
  const int cols = a.act >= 0 ? BN / 2 : BN;
  a.n_tiles = (a.N + cols - 1) / cols;
  constexpr size_t stages = (size_t)ST * WK * (BM + BN) * 128, sums = (size_t)(WK - 1) * BM * BN * 4, shm = stages > sums ? stages : sums;
  constexpr bool UNITS = BN / (16 * WN) % 2 == 0;   // takes gate and up
  if (a.act >= 0 && !UNITS) return (int)hipErrorInvalidValue;
  const void* const f[] = {(const void*)prompt_gemm_k<T, BM, BN, WM, WN, WK, ST, false>,
                           (const void*)prompt_gemm_k<T, BM, BN, WM, WN, WK, ST, UNITS>};
  static const hipError_t attr = [&] {
    for (const void* k : f)
      if (const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm)) return e;
    return hipSuccess;
  }();
  if (attr != hipSuccess) return (int)attr;
  void* args[] = {&a};
  return (int)hipLaunchKernel(f[a.act >= 0], dim3(a.m_tiles * a.n_tiles), dim3(64 * WM * WN * WK), args, shm, st);
}

// The tiles, and what a product takes on them: us(q) = start + (q - 1) round + S (q == 1 ? alone : max(alone, each q)) for
// q workgroups per CU and S stages of K.
struct Tile {
  int bm, bn;
  bool units;   // a wavefront's columns are an even number of 16
  float start, round, alone, each;
};
template <int COUNT>
static int pick_tile(const Tile (&tiles)[COUNT], int M, int N, int stages, bool units) {   // N: rows of w
  int best = 0;
  float least = 0.0f;
  for (int i = 0; i < COUNT; i++) {
    const Tile& t = tiles[i];
    if (units && !t.units) continue;
    const long q = ((long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) + 255) / 256;
    const float us = t.start + (q - 1) * t.round + stages * (q == 1 ? t.alone : std::max(t.alone, t.each * q));
    if (!best || us < least) best = i + 1, least = us;
  }
  return best;
}

int prompt_gemm_f32(const GemmArgs& a, int tile, hipStream_t st);
