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
  int ldx, M, N, K, ldy;
  // products side by side (blockIdx.y): numbers from one's x, w and y to the next one's
  long xb, wb, yb;
  // what happens to a result, rounded to its type, on its way out: columns from tanh_from on pass a tanh; g: times the
  // sigmoid of a gate per column (row ldg apart, columns of all products in a row), per_head: of one per product
  int tanh_from;
  const void* g;
  int ldg, per_head;
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
  const int p = blockIdx.y;
  const T* xp = (const T*)a.x + p * a.xb + (size_t)min(n16, a.M - 1) * a.ldx + quad * EP;
  const T* wp = (const T*)a.w + p * a.wb + (size_t)min(n, a.N - 1) * K + quad * EP;
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
  for (int e = 0; e < 4; e++) {
    const int m = quad * 4 + e;
    if (m >= a.M) break;
    T o[1];
    stf(o, 0, acc[e] + b);
    if (n >= a.tanh_from) stf(o, 0, tanhf(ldf(o, 0)));
    if (a.g) stf(o, 0, ldf(o, 0) * sigmoidf_(ldf((const T*)a.g, (size_t)m * a.ldg + (a.per_head ? p : p * a.N + n))));
    ((T*)a.y)[p * a.yb + (size_t)m * a.ldy + n] = o[0];
  }
}

extern "C" {

// x rows are ldx numbers apart and, like w, aligned to 16 bytes; y [M, N] is packed; columns from tanh_from on (N: none)
// pass a tanh
int p2p_sm_skinny(const void* x, int ldx, const void* w, const void* bias, void* y, int M, int N, int K, int tanh_from,
                  int f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int ep = f32 ? 4 : 8;
  if (M > 16 || K < ep || K % ep || ldx % ep || (size_t)x % 16 || (size_t)w % 16) return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, bias, y, ldx, M, N, K, N, 0, 0, 0, tanh_from, nullptr, 0, 0};
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((skinny_k<T>), dim3((N + 15) / 16), dim3(512), 0, st, a));
  return (int)hipGetLastError();
}

// H products of M <= 16 rows, bf16: y[m, h * N + n] = (x[h, m] . w[h, n]) * sigmoid(g[m, h * N + n]), per_head: of g[m, h].
// x rows are ldx numbers apart, heads xb; w [H, N, K] is packed.  A head of 512 numbers and 128 columns took the library
// 16 workgroups and 14 us for 8 rows and 16 heads, and the gates a launch of 4.6; 5.4 here.
int p2p_sm_skinny_heads(const void* x, long xb, int ldx, const void* w, const void* g, int ldg, int per_head, void* y,
                        int ldy, int M, int H, int N, int K, hipStream_t st) {
  if (M <= 0 || N <= 0 || H <= 0) return 0;
  if (M > 16 || H > 65535 || K < 8 || K % 8 || ldx % 8 || xb % 8 || (size_t)x % 16 || (size_t)w % 16 || !g)
    return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, nullptr, y, ldx, M, N, K, ldy, xb, (long)N * K, N, N, g, ldg, per_head};
  hipLaunchKernelGGL((skinny_k<bf16>), dim3((N + 15) / 16, H), dim3(512), 0, st, a);
  return (int)hipGetLastError();
}

}  // extern "C"
