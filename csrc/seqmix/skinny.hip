// Matrix products of few rows: y[m, n] = sum_k x[m, k] W[n, k] (+ bias[n]), m < M <= 16, weights as a checkpoint has
// them (row-major [N, K]), bf16 or fp32 with fp32 sums, one rounding at the end.
//
// A step of few rows reads every weight once and does little else, so the kernels are built around the loads: a
// workgroup takes 16 rows of W at a time, its eight wavefronts take the K index 128 bytes at a time in turn (together
// they read 1 KB of each row) and multiply (v_mfma_f32_16x16x32_bf16; fp32: four v_mfma_f32_16x16x4_f32 per 16-byte
// fragment).  The eight partial sums meet in LDS.  Bound by the weight stream at large N * K and by the chain of one
// launch otherwise (about 2.3 us at K = 32).  Two kernels with the same sums in the same order:
//  * walk_k, where four such pieces hold K (2048 numbers of bf16, 1024 of fp32): a workgroup reads the activations
//    once, keeps them in registers and walks over tiles of 16 columns; the next tile's weights (up to 64 KB) are
//    asked for in one burst while this one is multiplied and summed.
//  * skinny_k, above, for few columns and for K that fills its pieces badly: one tile per workgroup, two pieces of weights
//    and activations in flight.
// In a captured graph with cold weights, us, vendor product / skinny_k / walk_k.  bf16, 8 rows: 2048 x 2048 11.2 / 6.0 /
// 5.8, 4096 x 2048 11.7 / 6.7 / 6.2, 10304 x 2048 14.5 / 13.6 / 11.0, 18432 x 2048 58.7 / 21.3 / 17.0 (4.4 TB/s),
// 32000 x 2048 34.5 / 32.5 / 26.5 (4.9), 16384 x 512 11.7 / 6.5 / 5.4; 16 rows 10304 x 2048 14.5 / 16.1 / 11.4, one
// row 14.5 / 11.9 / 10.4.  fp32, 8 rows: 4096 x 1024 11.5 / 6.9 / 6.5, 16384 x 1024 18.2 / 19.5 / 15.5.  Eight pieces in
// registers are no better: fp32 4096 x 2048 13.0 / 10.2 / 11.1, bf16 2048 x 4096 14.9 / 8.8 / 8.6.
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

// rows quad * 4 .. + 3 of column n of product p.  ACT: with the tanh and the gate, whose code a plain product need not fetch
template <typename T, bool ACT>
__device__ __forceinline__ void store_tile(const SkinnyArgs& a, int p, int n, int quad, f32x4 acc) {
  const float b = a.bias ? ldf((const T*)a.bias, n) : 0.0f;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int m = quad * 4 + e;
    if (m >= a.M) break;
    T o[1];
    stf(o, 0, acc[e] + b);
    if constexpr (ACT) {
      if (n >= a.tanh_from) stf(o, 0, tanhf(ldf(o, 0)));
      if (a.g) stf(o, 0, ldf(o, 0) * sigmoidf_(ldf((const T*)a.g, (size_t)m * a.ldg + (a.per_head ? p : p * a.N + n))));
    }
    ((T*)a.y)[p * a.yb + (size_t)m * a.ldy + n] = o[0];
  }
}

template <typename T, bool ACT>
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
  store_tile<T, ACT>(a, p, n, quad, acc);
}

// NP: pieces of 128 bytes per wavefront that hold a row of K numbers
template <typename T, int NP, bool ACT>
__global__ void __launch_bounds__(512) walk_k(SkinnyArgs a) {
  constexpr int WAVES = 8;
  constexpr int EP = 16 / sizeof(T), KB = 8 * EP;   // numbers per fragment, per 128 bytes
  // by turns: the next tile's sums go to the other half, and the one after that starts behind the next barrier
  __shared__ f32x4 red[2][WAVES][64];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), n16 = lane & 15, quad = lane >> 4;
  const int p = blockIdx.y, tiles = (a.N + 15) / 16, stride = gridDim.x;
  // rows that do not exist are the last ones, their results are dropped
  const T* xp = (const T*)a.x + p * a.xb + (size_t)min(n16, a.M - 1) * a.ldx;
  auto row = [&](int t) { return (const T*)a.w + p * a.wb + (size_t)min(t * 16 + n16, a.N - 1) * a.K; };
  uint4 av[NP][2], bv[NP][2];
  int at[NP][2];   // a fragment past K reads the row's first numbers and counts as zero on both sides
  bool in[NP][2];
  int t = blockIdx.x;
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++) {
      const int k = (i * WAVES + wave) * KB + (s * 4 + quad) * EP;
      in[i][s] = k < a.K;
      at[i][s] = in[i][s] ? k : 0;
    }
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++) av[i][s] = *(const uint4*)(xp + at[i][s]);
  const T* first = row(t);
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++) bv[i][s] = *(const uint4*)(first + at[i][s]);
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++)
      if (!in[i][s]) av[i][s] = make_uint4(0, 0, 0, 0);
  for (int turn = 0; t < tiles; t += stride, turn++) {
    const bool more = t + stride < tiles;
    const T* next = row(t + stride);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    // the whole tile is there before the first of the next one is asked for: asked for one by one, as each is used, the
    // halves of a line come apart (32000 x 2048 31 us, this 26.5)
    __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll
    for (int i = 0; i < NP; i++)
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const uint4 w = in[i][s] ? bv[i][s] : make_uint4(0, 0, 0, 0);
        acc = mfma_frag<T>(av[i][s], w, acc);
        if (more) bv[i][s] = *(const uint4*)(next + at[i][s]);
      }
    f32x4 (&sums)[WAVES][64] = red[turn & 1];
    sums[wave][lane] = acc;
    // a barrier that leaves the loads in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (wave == (turn & (WAVES - 1))) {
      acc = sums[0][lane];
#pragma unroll
      for (int w = 1; w < WAVES; w++) acc += sums[w][lane];
      const int n = t * 16 + n16;
      if (n < a.N) store_tile<T, ACT>(a, p, n, quad, acc);
    }
  }
}

// One workgroup per CU, all products together, each with the same number of tiles but for the last ones (8 rows in bf16,
// 10304 x 2048: 215 workgroups 11.1 us, 256 11.3, 322 14.0, 512 11.8); two where a tile is only 16 KB (16384 x 512: 5.5
// beside 6.4, while 16384 x 1024 has 8.5 beside 8.2).
static int walkers(int tiles, int products, int pieces) {
  const int most = max(1, 256 * (pieces > 1 ? 1 : 2) / products), each = (tiles + most - 1) / most;
  return (tiles + each - 1) / each;
}

// Whether to walk; both kernels give the same sums.  A wavefront of walk_k loads whole pieces, also past K, and holds them
// all before it multiplies, where skinny_k leaves out what is past K and multiplies what comes first.  us, bf16, skinny_k /
// walk_k (fp32 at half the K the same within 5 %):
//  * a tile per workgroup: 8 rows, 1024 columns, K = 64 2.3 / 2.8, 256 2.5 / 2.8, 512 2.9 / 2.8, 640 3.3 / 3.7, 1024 3.9 /
//    3.9; three and four pieces: 2048 x 2048 5.4 / 5.5, 4096 x 2048 7.1 / 6.5, 4096 x 1792 6.5 / 6.3;
//  * several: 8192 columns, K = 512, one row 3.8 / 3.7, 16 rows 4.5 / 4.2; K = 768, one row 4.9 / 5.2, 8 rows 5.6 / 5.5, 16
//    rows 6.4 / 5.6; K = 896, one row 5.4 / 5.4, 8 rows 6.5 / 5.7; 16384 columns, K = 64, 8 rows 3.0 / 4.7, K = 384 5.7 /
//    5.2, K = 640, 8 rows 8.0 / 8.0, 16 rows 9.3 / 8.3, K = 1024, 8 rows 11.2 / 8.3.
static bool walks(int tiles, int pieces, int eighths, int M) {
  if (pieces > 4) return false;
  if (tiles <= 256) return eighths == 8 && (pieces <= 2 || tiles >= 192);
  if (eighths >= 7) return true;
  return M > 4 && eighths == 6 ? tiles >= (pieces > 1 ? 512 : 768) : M > 8 && eighths == 5 && tiles >= 768;
}

template <typename T, bool ACT>
static void launch_tiles(const SkinnyArgs& a, int products, hipStream_t st) {
  constexpr int PIECE = 64 * 16 / (int)sizeof(T);   // numbers of K that the eight wavefronts' pieces hold
  const int tiles = (a.N + 15) / 16, pieces = (a.K + PIECE - 1) / PIECE;
  const dim3 g(walkers(tiles, products, pieces), products), b(512);
  if (!walks(tiles * products, pieces, a.K * 8 / (pieces * PIECE), a.M))
    hipLaunchKernelGGL((skinny_k<T, ACT>), dim3(tiles, products), b, 0, st, a);
  else if (pieces == 4) hipLaunchKernelGGL((walk_k<T, 4, ACT>), g, b, 0, st, a);
  else if (pieces == 3) hipLaunchKernelGGL((walk_k<T, 3, ACT>), g, b, 0, st, a);
  else if (pieces == 2) hipLaunchKernelGGL((walk_k<T, 2, ACT>), g, b, 0, st, a);
  else hipLaunchKernelGGL((walk_k<T, 1, ACT>), g, b, 0, st, a);
}

template <typename T>
static void launch_skinny(const SkinnyArgs& a, int products, hipStream_t st) {
  if (a.g || a.tanh_from < a.N) launch_tiles<T, true>(a, products, st);
  else launch_tiles<T, false>(a, products, st);
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
  SM_DISPATCH_T(f32, launch_skinny<T>(a, 1, st));
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
  launch_skinny<bf16>(a, H, st);
  return (int)hipGetLastError();
}

}  // extern "C"
