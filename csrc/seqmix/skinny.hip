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
  // logits: y is fp32 and holds cap * tanh(scale * result / cap), cap 0: scale * result
  int logits;
  float cap, scale;
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
      if (a.logits) {
        const float z = ldf(o, 0) * a.scale;
        ((float*)a.y)[(size_t)m * a.ldy + n] = a.cap > 0.0f ? a.cap * tanhf(z / a.cap) : z;
        continue;
      }
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

// A row pass as the way into a product (norm_scale_add_k in norms.hip has the sums, in the same order):
//   xo = x + y / sqrt(mean(y^2) + eps) * w * ls,   h = xo, or with w2 xo / sqrt(mean(xo^2) + eps) * w2
// Every workgroup forms all rows of h for itself; one writes xo (not over x, which others may still read).
struct PreArgs {
  const float* x;
  const void* y;
  int ldy;
  const float *w, *ls, *w2;
  float eps;
  float* xo;
};

// A short causal convolution + bias + silu behind a product whose rows are one token each (mamba_conv_k in mamba.hip):
// columns c0 .. c0 + C - 1 of a row, rounded to their type, with the K - 1 raw inputs before them from the slot's tail,
// which moves on.  Row r is entry r.
struct ConvArgs {
  int c0, C, K;
  const float *cw, *cb;
  float* tail;
  const int* ent;
  void* out;
  int ldo, out_f32;
};

// what a lane's four (row, column) places of one tile need for their convolution
struct ConvIn {
  float tl[4][4], w[4], b;   // (the raw input itself comes after the K - 1 before it)
};
// loads at addresses that are there whatever K and the positions are, chosen from afterwards: they go out as one batch
__device__ __forceinline__ void conv_load(const ConvArgs& c, const int2 (&start_slot)[4], int n, ConvIn& v) {
  const int ch = min(max(n - c.c0, 0), c.C - 1);
  v.b = c.cb[ch];
#pragma unroll
  for (int k = 0; k < 4; k++) v.w[k] = c.cw[(size_t)ch * c.K + min(k, c.K - 1)];
  if (c.K > 1) {
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int k = 0; k < 3; k++)
        v.tl[e][k] = c.tail[((size_t)start_slot[e].y * (c.K - 1) + min(k, c.K - 2)) * c.C + ch];
  }
}
template <typename T>
__device__ __forceinline__ void conv_store(const ConvArgs& c, const int2 (&start_slot)[4], int M, int n, int quad,
                                           const ConvIn& v, const f32x4& raw) {
  const int ch = n - c.c0;
  if (ch < 0 || ch >= c.C) return;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int m = quad * 4 + e;
    if (m >= M) break;
    T o[1];
    stf(o, 0, raw[e]);
    const float last = ldf(o, 0);
    const bool from = start_slot[e].x > 0;
    float tl[3], acc = v.b;
#pragma unroll
    for (int k = 0; k < 3; k++) tl[k] = from && k < c.K - 1 ? v.tl[e][k] : 0.0f;
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (k < c.K) acc += v.w[k] * (k < c.K - 1 ? tl[min(k, 2)] : last);
    acc = acc * sigmoidf_(acc);
    if (c.out_f32) ((float*)c.out)[(size_t)m * c.ldo + ch] = acc;
    else stf((T*)c.out, (size_t)m * c.ldo + ch, acc);
    float* to = c.tail + (size_t)start_slot[e].y * (c.K - 1) * c.C + ch;
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (k < c.K - 1) to[(size_t)k * c.C] = k + 1 < c.K - 1 ? tl[min(k + 1, 2)] : last;
  }
}

// A barrier that leaves loads in flight
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// walk_k behind a row pass, and with a convolution behind it (CONV).  Four wavefronts take a row, as the pass's workgroup
// does, and RB of their rows at once (0: the rows are there, a.x); h lies in LDS as the product reads it.  The first
// tile's weights are on their way meanwhile.  Bound by the chain of a launch: for one row of 1024 the pass (3.0 us), the
// product of 4096 columns (4.6) and the convolution (4.0) are 6.8 us, the product behind the pass alone 4.4, and the gaps
// between the launches are gone; 8 rows of 2048 in front of 10304 columns take 18.6 beside 4.7 + 12.8 (every workgroup
// reads all rows), which is why only few rows come this way.
template <typename T, int NP, bool ACT, bool CONV, int RB>
__global__ void __launch_bounds__(512) norm_walk_k(SkinnyArgs a, PreArgs pre, ConvArgs cv) {
  constexpr int WAVES = 8;
  constexpr bool PRE = RB > 0;
  constexpr int EP = 16 / sizeof(T), KB = 8 * EP;
  constexpr int NC = (NP * WAVES * KB + 1023) / 1024;   // numbers per thread of the pass / 4
  constexpr int LD = NP * WAVES * KB + EP;              // (+ 16 bytes: 16 rows' pieces spread over the banks)
  extern __shared__ __align__(16) unsigned char given[];
  T* sh = (T*)given;                                    // [M][LD]
  __shared__ f32x4 red[2][WAVES][64];
  __shared__ float sums1[2][RB + !PRE][4], sums2[2][RB + !PRE][4];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), n16 = lane & 15, quad = lane >> 4;
  const int tiles = (a.N + 15) / 16, stride = gridDim.x, n = a.K;
  auto row = [&](int t) { return (const T*)a.w + (size_t)min(t * 16 + n16, a.N - 1) * a.K; };
  uint4 av[NP][2], bv[NP][2];
  int at[NP][2];
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
  const int half = wave >> 2, w4 = wave & 3;
  struct __align__(4 * sizeof(T)) Four { T v[4]; };
  auto place = [&](int k) { return ((int)(threadIdx.x & 255) + k * 256) * 4; };
  Four yv[RB + !PRE][NC];
  float4 xv[RB + !PRE][NC];
  float wl[NC][4], nw[NC][4];
  auto fetch = [&](int m0) {   // rows m0 + half, + 2, .., the last one again beyond it
#pragma unroll
    for (int b = 0; b < RB; b++) {
      const int m = min(m0 + 2 * b + half, a.M - 1);
#pragma unroll
      for (int k = 0; k < NC; k++) {
        const int i = place(k) < n ? place(k) : 0;
        yv[b][k] = *(const Four*)((const T*)pre.y + (size_t)m * pre.ldy + i);
        xv[b][k] = *(const float4*)(pre.x + (size_t)m * n + i);
      }
    }
  };
  // All loads go out before the first is waited for, in the order of their use (they arrive in the order they went out);
  // the weights are last
  int2 start_slot[4];
  if constexpr (CONV) {
#pragma unroll
    for (int e = 0; e < 4; e++) start_slot[e] = *(const int2*)(cv.ent + 4 * min(quad * 4 + e, a.M - 1) + 2);
  }
  float4 gw[NC], gl[NC], g2[NC];
  if constexpr (PRE) {
    fetch(0);
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = place(k) < n ? place(k) : 0;
      gw[k] = *(const float4*)(pre.w + i);
      gl[k] = pre.ls ? *(const float4*)(pre.ls + i) : make_float4(1.f, 1.f, 1.f, 1.f);
      g2[k] = pre.w2 ? *(const float4*)(pre.w2 + i) : make_float4(1.f, 1.f, 1.f, 1.f);
    }
  } else {
    const T* xp = (const T*)a.x + (size_t)min(n16, a.M - 1) * a.ldx;
#pragma unroll
    for (int i = 0; i < NP; i++)
#pragma unroll
      for (int s = 0; s < 2; s++) av[i][s] = *(const uint4*)(xp + at[i][s]);
  }
  __builtin_amdgcn_sched_barrier(0);
  ConvIn ci;
  if constexpr (CONV)   // this wavefront finishes tile number `wave` of the walk
    conv_load(cv, start_slot, min(t + wave * stride, tiles - 1) * 16 + n16, ci);
  __builtin_amdgcn_sched_barrier(0);
  const T* first = row(t);
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++) bv[i][s] = *(const uint4*)(first + at[i][s]);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (PRE) {
#pragma unroll
  for (int k = 0; k < NC; k++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const bool there = place(k) < n;
      wl[k][j] = there ? ((const float*)&gw[k])[j] * ((const float*)&gl[k])[j] : 0.0f;
      nw[k][j] = there ? ((const float*)&g2[k])[j] : 0.0f;
    }
  for (int m0 = 0; m0 < a.M; m0 += 2 * max(RB, 1)) {
    if (m0) fetch(m0);
    float x[RB + !PRE][NC][4];
#pragma unroll
    for (int b = 0; b < RB; b++) {
      if (m0 + 2 * b + half >= a.M) break;
      float ss = 0.0f;
#pragma unroll
      for (int k = 0; k < NC; k++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float v = place(k) < n ? ldf(yv[b][k].v, j) : 0.0f;
          ss += v * v;
        }
      ss = wave_sum(ss);
      if (lane == 0) sums1[half][b][w4] = ss;
    }
    meet();
#pragma unroll
    for (int b = 0; b < RB; b++) {
      const int m = m0 + 2 * b + half;
      if (m >= a.M) break;
      float ss = 0.0f, s2 = 0.0f;
#pragma unroll
      for (int u = 0; u < 4; u++) ss += sums1[half][b][u];
      const float rs = 1.0f / sqrtf(ss / (float)n + pre.eps);
#pragma unroll
      for (int k = 0; k < NC; k++) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const bool there = place(k) < n;
          x[b][k][j] = there ? ((const float*)&xv[b][k])[j] : 0.0f;
          x[b][k][j] = x[b][k][j] + (there ? ldf(yv[b][k].v, j) : 0.0f) * rs * wl[k][j];
          s2 += x[b][k][j] * x[b][k][j];
        }
        if (blockIdx.x == 0 && place(k) < n) stv<4>(pre.xo + (size_t)m * n, place(k), x[b][k]);
      }
      if (pre.w2) {
        s2 = wave_sum(s2);
        if (lane == 0) sums2[half][b][w4] = s2;
      }
    }
    if (pre.w2) meet();
#pragma unroll
    for (int b = 0; b < RB; b++) {
      const int m = m0 + 2 * b + half;
      if (m >= a.M) break;
      if (pre.w2) {
        float s2 = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; u++) s2 += sums2[half][b][u];
        const float r2 = 1.0f / sqrtf(s2 / (float)n + pre.eps);
#pragma unroll
        for (int k = 0; k < NC; k++)
#pragma unroll
          for (int j = 0; j < 4; j++) x[b][k][j] *= r2 * nw[k][j];
      }
#pragma unroll
      for (int k = 0; k < NC; k++)
        if (place(k) < n) stv<4>(sh + m * LD, place(k), x[b][k]);
    }
    meet();   // (also: the next rows' sums take the place of these)
  }
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++) av[i][s] = *(const uint4*)(sh + min(n16, a.M - 1) * LD + at[i][s]);
  }
#pragma unroll
  for (int i = 0; i < NP; i++)
#pragma unroll
    for (int s = 0; s < 2; s++)
      if (!in[i][s]) av[i][s] = make_uint4(0, 0, 0, 0);
  for (int turn = 0; t < tiles; t += stride, turn++) {
    const bool more = t + stride < tiles;
    const T* next = row(t + stride);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_s_waitcnt(0x0f70);   // see walk_k
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
    meet();
    if (wave == (turn & (WAVES - 1))) {
      acc = sums[0][lane];
#pragma unroll
      for (int w = 1; w < WAVES; w++) acc += sums[w][lane];
      const int col = t * 16 + n16;
      if (col < a.N) store_tile<T, ACT>(a, 0, col, quad, acc);
      if constexpr (CONV) {
        if (col < a.N) conv_store<T>(cv, start_slot, a.M, col, quad, ci, acc);
        const int later = t + WAVES * stride;
        if (later < tiles) conv_load(cv, start_slot, later * 16 + n16, ci);
      }
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
  if (a.g || a.logits || a.tanh_from < a.N) launch_tiles<T, true>(a, products, st);
  else launch_tiles<T, false>(a, products, st);
}

// rows that are formed here (at most 16), RB of each half's at once
template <typename T, bool ACT, bool CONV, int RB>
static int launch_norm_walk(const SkinnyArgs& a, const PreArgs& pre, const ConvArgs& cv, hipStream_t st) {
  constexpr int PIECE = 64 * 16 / (int)sizeof(T);
  const int tiles = (a.N + 15) / 16, pieces = (a.K + PIECE - 1) / PIECE;
  const dim3 g(walkers(tiles, 1, pieces)), b(512);
  const size_t shm = RB ? (size_t)a.M * (pieces * PIECE + 16 / sizeof(T)) * sizeof(T) : 0;
#define NW(NP)                                                                                          \
  {                                                                                                     \
    constexpr auto kernel = norm_walk_k<T, NP, ACT, CONV, RB>;                                          \
    static const hipError_t attr =                                                                      \
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 72 * 1024); \
    if (attr != hipSuccess) return (int)attr;                                                           \
    hipLaunchKernelGGL(kernel, g, b, shm, st, a, pre, cv);                                              \
  }
  if (pieces == 4) NW(4)
  else if (pieces == 3) NW(3)
  else if (pieces == 2) NW(2)
  else NW(1)
#undef NW
  return (int)hipGetLastError();
}
template <typename T, bool ACT, bool CONV>
static int launch_normed(const SkinnyArgs& a, const PreArgs& pre, const ConvArgs& cv, hipStream_t st) {
  if (a.M <= 2) return launch_norm_walk<T, ACT, CONV, 1>(a, pre, cv, st);
  return launch_norm_walk<T, ACT, CONV, 2>(a, pre, cv, st);
}

extern "C" {

// p2p_sm_skinny on rows that a residual pass leaves (PreArgs; x, xo fp32 [M, K] packed), with an optional convolution
// behind columns c0 .. c0 + C - 1 (cw null: none).  K is a multiple of 4 (fp32) or 8 (bf16) of at most 1024 numbers in
// fp32, 2048 in bf16.  Up to 16 rows; models send 4 at most (NORMED_ROWS in ops/seqmix.py), more than that, whose rows a
// workgroup forms in several goes, are the tests' alone.
int p2p_sm_norm_skinny(const float* x, const void* y, int ldy, const float* nw, const float* ls, const float* w2,
                       float eps, float* xo, const void* w, const void* bias, void* out, int M, int N, int K,
                       int tanh_from, int c0, int C, int taps, const float* cw, const float* cb, float* tail,
                       const int* ent, void* conv, int ldo, int conv_f32, int f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int ep = f32 ? 4 : 8;
  if (M > 16 || K < ep || K % ep || K > (f32 ? 1024 : 2048) || (size_t)w % 16 || ldy % 4 || xo == x ||
      (((size_t)x | (size_t)xo | (size_t)nw | (size_t)ls | (size_t)w2) % 16) || (size_t)y % (f32 ? 16 : 8) ||
      (cw && (taps < 1 || taps > 4 || c0 < 0 || c0 + C > N || tanh_from < N)))
    return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {nullptr, w, bias, out, 0, M, N, K, N, 0, 0, 0, tanh_from, nullptr, 0, 0, 0, 0.0f, 1.0f};
  const PreArgs pre = {x, y, ldy, nw, ls, w2, eps, xo};
  const ConvArgs cv = {c0, C, taps, cw, cb, tail, ent, conv, ldo, conv_f32};
  if (cw) SM_DISPATCH_T(f32, return (launch_normed<T, false, true>(a, pre, cv, st)));
  if (tanh_from < N) SM_DISPATCH_T(f32, return (launch_normed<T, true, false>(a, pre, cv, st)));
  SM_DISPATCH_T(f32, return (launch_normed<T, false, false>(a, pre, cv, st)));
}

// p2p_sm_skinny with that convolution behind it, K as there
int p2p_sm_skinny_conv(const void* x, int ldx, const void* w, void* out, int M, int N, int K, int c0, int C, int taps,
                       const float* cw, const float* cb, float* tail, const int* ent, void* conv, int ldo, int conv_f32,
                       int f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int ep = f32 ? 4 : 8;
  if (M > 16 || K < ep || K % ep || K > (f32 ? 1024 : 2048) || ldx % ep || (size_t)x % 16 || (size_t)w % 16 || taps < 1 ||
      taps > 4 || c0 < 0 || c0 + C > N)
    return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, nullptr, out, ldx, M, N, K, N, 0, 0, 0, N, nullptr, 0, 0, 0, 0.0f, 1.0f};
  const ConvArgs cv = {c0, C, taps, cw, cb, tail, ent, conv, ldo, conv_f32};
  SM_DISPATCH_T(f32, return (launch_norm_walk<T, false, true, 0>(a, PreArgs{}, cv, st)));
}

// x rows are ldx numbers apart and, like w, aligned to 16 bytes; y [M, N] is packed; columns from tanh_from on (N: none)
// pass a tanh
int p2p_sm_skinny(const void* x, int ldx, const void* w, const void* bias, void* y, int M, int N, int K, int tanh_from,
                  int f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int ep = f32 ? 4 : 8;
  if (M > 16 || K < ep || K % ep || ldx % ep || (size_t)x % 16 || (size_t)w % 16) return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, bias, y, ldx, M, N, K, N, 0, 0, 0, tanh_from, nullptr, 0, 0, 0, 0.0f, 1.0f};
  SM_DISPATCH_T(f32, launch_skinny<T>(a, 1, st));
  return (int)hipGetLastError();
}

// The same with fp32 logits y [M, N]: results, rounded to the type, times scale and capped (cap 0: not)
int p2p_sm_skinny_logits(const void* x, int ldx, const void* w, float* y, int M, int N, int K, float cap, float scale,
                         int f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int ep = f32 ? 4 : 8;
  if (M > 16 || K < ep || K % ep || ldx % ep || (size_t)x % 16 || (size_t)w % 16) return (int)hipErrorInvalidValue;
  const SkinnyArgs a = {x, w, nullptr, y, ldx, M, N, K, N, 0, 0, 0, N, nullptr, 0, 0, 1, cap, scale};
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
  const SkinnyArgs a = {x, w, nullptr, y, ldx, M, N, K, ldy, xb, (long)N * K, N, N, g, ldg, per_head, 0, 0.0f, 1.0f};
  launch_skinny<bf16>(a, H, st);
  return (int)hipGetLastError();
}

}  // extern "C"
