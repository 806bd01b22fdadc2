// Matrix products of few rows: y[m, n] = sum_k x[m, k] W[n, k] (+ bias[n]), m < M <= 16, weights as a checkpoint has
// them (row-major [N, K]), bf16 or fp32 with fp32 sums, one rounding at the end.
//
// A step of few rows reads every weight once and does little else, so the kernel is built around the loads: a
// workgroup takes 16 rows of W, its eight wavefronts take the K index 128 bytes at a time in turn (together they
// read 1 KB of each row), and each keeps two such pieces of all 16 rows in flight while it multiplies
// (v_mfma_f32_16x16x32_bf16; fp32: four v_mfma_f32_16x16x4_f32 per 16-byte fragment).  The eight partial sums meet
// in LDS.
//
// Bound by the weight stream at large N * K and by the chain of one launch otherwise (about 2.3 us at K = 32; the
// activations are read by every workgroup, which is what 16 rows cost over one).  8 rows in bf16, in a captured
// graph, microseconds, vendor product -> this: 1024 x 1024 5.8 -> 3.8, 4096 x 1024 6.1 -> 4.3, 2048 x 2048
// 8.3 -> 5.4, 2048 x 4096 12.5 -> 8.3, 10304 x 2048 15.9 -> 13.2 (3.2 TB/s), one row 16.0 -> 11.6; fp32 1024 x 1024
// 8.2 -> 5.4, 2048 x 2048 10.5 -> 8.5.  32 columns per workgroup leave half as many workgroups (2048 x 2048: 7.4),
// 16 wavefronts or four pieces in flight measured the same within 0.2.
#include "attn_tile.h"
using namespace sm;

struct SkinnyArgs {
  const void *x, *w, *bias;
  void* y;
  int ldx, M, N, K;
};

template <typename T>
__device__ __forceinline__ f32x4 mfma_frag(uint4 a, uint4 b, f32x4 c) {
  if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int i = 0; i < 4; i++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], c, 0, 0, 0);
    return c;
  }
}

template <typename T>
__global__ void __launch_bounds__(512) skinny_k(SkinnyArgs a) {
  constexpr int WAVES = 8, DEPTH = 2;
  constexpr int EP = 16 / sizeof(T), KB = 8 * EP;   // numbers per fragment, per 128 bytes
  __shared__ f32x4 red[WAVES - 1][64];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), n16 = lane & 15, quad = lane >> 4;
  const int n0 = blockIdx.x * 16, n = n0 + n16, K = a.K;
  // rows that do not exist are the last ones, their results are dropped
  const T* xp = (const T*)a.x + (size_t)min(n16, a.M - 1) * a.ldx + quad * EP;
  const T* wp = (const T*)a.w + (size_t)min(n, a.N - 1) * K + quad * EP;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  uint4 av[DEPTH][2], bv[DEPTH][2];
  auto load = [&](int k, uint4 (&A)[2], uint4 (&B)[2]) {   // a piece past K is zero
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int at = k + s * 4 * EP;
      const bool in = at + quad * EP < K;
      const int o = in ? at : -quad * EP;
      B[s] = *(const uint4*)(wp + o);
      A[s] = *(const uint4*)(xp + o);
      if (!in) {
        B[s] = make_uint4(0, 0, 0, 0);
        A[s] = make_uint4(0, 0, 0, 0);
      }
    }
  };
  const int kb = wave * KB, step = WAVES * KB;
#pragma unroll
  for (int d = 0; d < DEPTH; d++)
    if (kb + d * step < K) load(kb + d * step, av[d], bv[d]);
  for (int k0 = kb; k0 < K; k0 += DEPTH * step) {
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
      const int k = k0 + d * step;
      if (k < K) {
#pragma unroll
        for (int s = 0; s < 2; s++) acc = mfma_frag<T>(av[d][s], bv[d][s], acc);
        if (k + DEPTH * step < K) load(k + DEPTH * step, av[d], bv[d]);
      }
    }
  }
  if (wave > 0) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave > 0 || n >= a.N) return;
#pragma unroll
  for (int w = 0; w < WAVES - 1; w++) acc += red[w][lane];
  const float b = a.bias ? ldf((const T*)a.bias, n) : 0.0f;
#pragma unroll
  for (int e = 0; e < 4; e++)
    if (quad * 4 + e < a.M) stf((T*)a.y, (size_t)(quad * 4 + e) * a.N + n, acc[e] + b);
}

// The same for the rows of a short prompt, bf16: a workgroup takes 32 rows x 64 columns, its eight wavefronts the K index
// 128 bytes at a time in turn, straight from memory into fragments, two such pieces in flight; each finishes one of the
// eight 16 x 16 parts.
//
// A short prompt is bound by the host: a vendor product costs it 22 us (the library looks its kernel up at each call), this
// one 5, and a pass has 22 to 25 of them.  The kernel itself is bound by what a CU can take in (some 40 KB/us): 64 rows,
// 1024 x 1024 7.8 us (library 6.6), 8192 x 1024 8.5 (9.0), 2048 x 2048 13.3 (8.9), 10272 x 2048 28.7 (14.3).
// `_rows` in ops/seqmix.py draws the line.
__global__ void __launch_bounds__(512) rows_k(SkinnyArgs a) {
  typedef bf16 T;
  constexpr int WAVES = 8, MT = 2, NT = 4;
  constexpr int EP = 16 / sizeof(T), KB = 8 * EP;   // numbers per fragment, per 128 bytes
  __shared__ f32x4 red[WAVES][MT * NT][64];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), n16 = lane & 15, quad = lane >> 4;
  const int n0 = blockIdx.x * 64, m0 = blockIdx.y * 32, K = a.K;
  // rows that do not exist are the last ones, their results are dropped
  const T *xp[MT], *wp[NT];
#pragma unroll
  for (int t = 0; t < MT; t++) xp[t] = (const T*)a.x + (size_t)min(m0 + t * 16 + n16, a.M - 1) * a.ldx + quad * EP;
#pragma unroll
  for (int t = 0; t < NT; t++) wp[t] = (const T*)a.w + (size_t)min(n0 + t * 16 + n16, a.N - 1) * K + quad * EP;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint4 av[2][2][MT], bv[2][2][NT];
  auto load = [&](int k, uint4 (&A)[2][MT], uint4 (&B)[2][NT]) {   // a piece past K is zero
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int at = k + s * 4 * EP;
      const bool in = at + quad * EP < K;
      const int o = in ? at : -quad * EP;
#pragma unroll
      for (int t = 0; t < NT; t++) B[s][t] = *(const uint4*)(wp[t] + o);
#pragma unroll
      for (int t = 0; t < MT; t++) A[s][t] = *(const uint4*)(xp[t] + o);
      if (!in) {
#pragma unroll
        for (int t = 0; t < NT; t++) B[s][t] = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int t = 0; t < MT; t++) A[s][t] = make_uint4(0, 0, 0, 0);
      }
    }
  };
  const int kb = wave * KB, step = WAVES * KB;
#pragma unroll
  for (int d = 0; d < 2; d++)
    if (kb + d * step < K) load(kb + d * step, av[d], bv[d]);
  for (int k0 = kb; k0 < K; k0 += 2 * step) {
#pragma unroll
    for (int d = 0; d < 2; d++) {
      const int k = k0 + d * step;
      if (k < K) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = mfma_frag<T>(av[d][s][i], bv[d][s][j], acc[i][j]);
        if (k + 2 * step < K) load(k + 2 * step, av[d], bv[d]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) red[wave][i * NT + j][lane] = acc[i][j];
  __syncthreads();
  // eight 16 x 16 parts, one per wavefront
  const int i = wave / NT, n = n0 + (wave % NT) * 16 + n16;
  f32x4 s = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < WAVES; w++) s += red[w][wave][lane];
  if (n >= a.N) return;
  const float b = a.bias ? ldf((const T*)a.bias, n) : 0.0f;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int m = m0 + i * 16 + quad * 4 + e;
    if (m < a.M) stf((T*)a.y, (size_t)m * a.N + n, s[e] + b);
  }
}

extern "C" {

// x rows are ldx numbers apart and, like w, aligned to 16 bytes; y [M, N] is packed
int p2p_sm_skinny(const void* x, int ldx, const void* w, const void* bias, void* y, int M, int N, int K, int f32,
                  hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int ep = f32 ? 4 : 8;
  if (M > 16 || K < ep || K % ep || ldx % ep || (size_t)x % 16 || (size_t)w % 16) return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, bias, y, ldx, M, N, K};
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((skinny_k<T>), dim3((N + 15) / 16), dim3(512), 0, st, a));
  return (int)hipGetLastError();
}

// the same arguments, any number of rows, bf16
int p2p_sm_rows(const void* x, int ldx, const void* w, const void* bias, void* y, int M, int N, int K, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 65535 * 32 || K < 8 || K % 8 || ldx % 8 || (size_t)x % 16 || (size_t)w % 16) return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, bias, y, ldx, M, N, K};
  hipLaunchKernelGGL(rows_k, dim3((N + 63) / 64, (M + 31) / 32), dim3(512), 0, st, a);
  return (int)hipGetLastError();
}

}  // extern "C"
