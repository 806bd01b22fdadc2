// The Mamba-2 scan over long portions in chunks of up to 64 tokens on the fp32 matrix instruction
// (v_mfma_f32_16x16x4_f32: products and sums in fp32).  Per head, with A = -exp(A_log), dt = softplus(raw +
// bias), the decays' running sum c_t = sum_{s <= t} A dt_s inside a chunk of n tokens and S the state before it:
//   local pass   L = sum_t exp(c_(n-1) - c_t) dt_t B_t x_t^T                              [N x P]
//   chain        S_next = exp(c_(n-1)) S + L over each portion's chunks, from the slot's state (or zero at
//                position 0); the last one is the slot's new state
//   output pass  y_t = exp(c_t) S^T C_t + sum_{s <= t} exp(c_t - c_s) dt_s (C_t . B_s) x_s + D x_t,  y *= silu(z)
// Every exponent is <= 0, so nothing overflows whatever the step sizes are.  One workgroup of four wavefronts per
// (chunk, head); sizes are padded to multiples of 16 with zeros in LDS, rows are laid out so that the
// lanes of a fragment read hit different banks.
//
// The walk of mamba_scan_k does the same 1 074 M state updates of a prompt of 2048 tokens (64 heads, 128 x 64 states)
// twice, token after token: 240 us each, bound by the chain per token.  The matrix form does 3.7 MFLOP per chunk and
// head, bound by LDS reads per product and by staging B and C from L2 for every head: 61 + 30 + 137 us.
#include "common.h"
using namespace sm;

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define MC 64   // tokens of a chunk

// row lengths in LDS: fragments that take 16 rows x 4 neighbours want ld = 4 mod 64, fragments that take 4
// rows x 16 neighbours ld = 16 mod 64
static __host__ __device__ __forceinline__ int ld_rows(int n) { return n + ((4 - n) & 63); }
static __host__ __device__ __forceinline__ int ld_cols(int n) { return n + ((16 - n) & 63); }

struct MambaChunkArgs {
  const float* conv;   // [R, C] = x | B | C after the convolution
  int C;
  const void* zx;
  int ldz, dtoff;
  const float *dt_bias, *A_log, *Dp;
  float *state, *cs, *decay;
  const int *vent, *cent;
  float* y;
  int H, P, N, G, NV, vec;
};

// dt and c of the chunk's tokens (zero steps beyond it) by the first wavefront
template <typename T>
__device__ __forceinline__ void chunk_steps(const MambaChunkArgs& a, const Entry& en, int h, float* sdt, float* sc) {
  if (threadIdx.x >= 64) return;
  const int t = threadIdx.x;
  float dt = 0.0f;
  if (t < en.n) dt = softplusf_(ldf((const T*)a.zx, (size_t)(en.row0 + t) * a.ldz + a.dtoff + h) + a.dt_bias[h]);
  float c = -expf(a.A_log[h]) * dt;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float v = __shfl_up(c, o, 64);
    if (t >= o) c += v;
  }
  sdt[t] = dt;
  sc[t] = c;
}

// n rows of `width` numbers of src (row stride ld) -> dst [MC][ldd] times scale(t); zeros up to `pad` columns and in
// rows n .. MC-1
template <typename F>
__device__ __forceinline__ void stage(const float* __restrict__ src, size_t ld, int n, int width, int pad, float* dst,
                                      int ldd, int vec, F scale) {
  if (vec) {   // four numbers per load
    const int w4 = pad / 4;
    for (int i = threadIdx.x; i < MC * w4; i += 256) {
      const int t = i / w4, c = i % w4 * 4;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
      if (t < n && c < width) v = *(const f32x4*)(src + (size_t)t * ld + c) * scale(t);
      *(f32x4*)(dst + t * ldd + c) = v;
    }
    return;
  }
  for (int i = threadIdx.x; i < MC * pad; i += 256) {
    const int t = i / pad, c = i % pad;
    dst[t * ldd + c] = (t < n && c < width) ? src[(size_t)t * ld + c] * scale(t) : 0.0f;
  }
}

template <typename T, int NPT>   // value size padded to NPT * 16
__global__ void __launch_bounds__(256) mamba_local_k(MambaChunkArgs a) {
  extern __shared__ __align__(16) float smem[];
  __shared__ float sdt[MC], sc[MC];
  const int c = blockIdx.x, h = blockIdx.y, N = a.N, P = a.P;
  const Entry en = load_entry(a.vent, c);
  const int NP = (N + 15) & ~15, PP = NPT * 16, LDB = ld_cols(NP), LDX = ld_cols(PP);
  float* sB = smem;
  float* sX = smem + MC * LDB;
  chunk_steps<T>(a, en, h, sdt, sc);
  __syncthreads();
  const float* row = a.conv + (size_t)en.row0 * a.C;
  const float end = sc[en.n - 1];
  stage(row + a.H * P + (h / (a.H / a.G)) * N, a.C, en.n, N, NP, sB, LDB, a.vec,
        [&](int t) { return sdt[t] * expf(end - sc[t]); });
  stage(row + h * P, a.C, en.n, P, PP, sX, LDX, a.vec, [](int) { return 1.0f; });
  if (threadIdx.x == 0) a.decay[(size_t)c * a.H + h] = expf(end);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
  const int steps = (en.n + 3) / 4;
  float* out = a.cs + ((size_t)c * a.H + h) * N * P;
  for (int nt = wave; nt * 16 < NP; nt += 4) {
    f32x4 acc[NPT];
#pragma unroll
    for (int j = 0; j < NPT; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < steps; s++) {
      const float b = sB[(4 * s + k4) * LDB + nt * 16 + i16];
#pragma unroll
      for (int j = 0; j < NPT; j++)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b, sX[(4 * s + k4) * LDX + j * 16 + i16], acc[j], 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NPT; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int n = nt * 16 + k4 * 4 + r, p = j * 16 + i16;
        if (n < N && p < P) out[(size_t)n * P + p] = acc[j][r];
      }
  }
}

// the state before chunk c replaces its local state; cent: per portion (first chunk, chunks, first position, slot)
__global__ void __launch_bounds__(256) mamba_chain_k(MambaChunkArgs a) {
  const int np = a.N * a.P, idx = blockIdx.x * 256 + threadIdx.x, h = blockIdx.y, e = blockIdx.z;
  if (idx >= np) return;
  const int c0 = a.cent[4 * e], nc = a.cent[4 * e + 1], start = a.cent[4 * e + 2], slot = a.cent[4 * e + 3];
  float* sg = a.state + ((size_t)slot * a.H + h) * np + idx;
  const size_t step = (size_t)a.H * np;
  float* q = a.cs + (size_t)c0 * step + (size_t)h * np + idx;
  const float* d = a.decay + (size_t)c0 * a.H + h;
  float cur = start > 0 ? *sg : 0.0f;
  for (int k = 0; k < nc; k += 8) {
    float loc[8], dec[8];   // eight chunks' loads in flight
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int kk = min(k + u, nc - 1);
      loc[u] = q[(size_t)kk * step];
      dec[u] = d[(size_t)kk * a.H];
    }
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (k + u < nc) {
        q[(size_t)(k + u) * step] = cur;
        cur = fmaf(dec[u], cur, loc[u]);
      }
  }
  *sg = cur;
}

template <typename T, int NPT>
__global__ void __launch_bounds__(256) mamba_out_k(MambaChunkArgs a) {
  extern __shared__ __align__(16) float smem[];
  __shared__ float sdt[MC], sc[MC];
  const int c = blockIdx.x, h = blockIdx.y, N = a.N, P = a.P, inner = a.H * P;
  const Entry en = load_entry(a.vent, c);
  const int n = en.n;
  const int NP = (N + 15) & ~15, PP = NPT * 16, LDC = ld_rows(NP), LDX = ld_cols(PP), LDW = MC + 4;
  float* sC = smem;                             // later the weights of the second product
  float* sB = smem + MC * max(LDC, LDW);        // later x
  float* sX = sB;
  float* sW = smem;                             // [MC][LDW]
  const float* row = a.conv + (size_t)en.row0 * a.C;
  const float* bc = row + inner + (h / (a.H / a.G)) * N;
  auto one = [](int) { return 1.0f; };
  chunk_steps<T>(a, en, h, sdt, sc);
  stage(bc + a.G * N, a.C, n, N, NP, sC, LDC, a.vec, one);
  stage(bc, a.C, n, N, NP, sB, LDC, a.vec, one);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
  const int r0 = wave * 16;                     // this wavefront's 16 tokens
  f32x4 w[MC / 16], acc[NPT];                   // C_t . B_s;  S^T C_t, then y
#pragma unroll
  for (int j = 0; j < MC / 16; j++) w[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NPT; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (r0 < n) {
    const float* S = a.cs + ((size_t)c * a.H + h) * N * P;
#pragma unroll 4
    for (int s = 0; s < NP / 4; s++) {
      const float q = sC[(r0 + i16) * LDC + 4 * s + k4];        // zero beyond N
      const float* Sr = S + (size_t)min(4 * s + k4, N - 1) * P;
      float b[NPT];
#pragma unroll
      for (int j = 0; j < NPT; j++) b[j] = Sr[min(j * 16 + i16, P - 1)];
#pragma unroll
      for (int j = 0; j < MC / 16; j++)
        if (j <= wave)
          w[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, sB[(j * 16 + i16) * LDC + 4 * s + k4], w[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NPT; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, b[j], acc[j], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float m = expf(sc[r0 + k4 * 4 + r]);
#pragma unroll
      for (int j = 0; j < NPT; j++) acc[j][r] *= m;
    }
  }
  __syncthreads();   // B and C have been read
  stage(row + h * P, a.C, n, P, PP, sX, LDX, a.vec, one);
#pragma unroll
  for (int j = 0; j < MC / 16; j++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int t = r0 + k4 * 4 + r, s = j * 16 + i16;
      sW[t * LDW + s] = s <= t ? w[j][r] * expf(sc[t] - sc[s]) * sdt[s] : 0.0f;
    }
  __syncthreads();
  if (r0 >= n) return;
  for (int s = 0; s < (wave + 1) * 4; s++) {
    const float q = sW[(r0 + i16) * LDW + 4 * s + k4];
#pragma unroll
    for (int j = 0; j < NPT; j++)
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(q, sX[(4 * s + k4) * LDX + j * 16 + i16], acc[j], 0, 0, 0);
  }
  const float Dh = a.Dp[h];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int t = r0 + k4 * 4 + r;
    if (t >= n) continue;
    const size_t at = (size_t)(en.row0 + t);
#pragma unroll
    for (int j = 0; j < NPT; j++) {
      const int p = j * 16 + i16;
      if (p >= P) continue;
      const float z = ldf((const T*)a.zx, at * a.ldz + h * P + p);
      a.y[at * inner + h * P + p] = (acc[j][r] + Dh * sX[t * LDX + p]) * (z * sigmoidf_(z));
    }
  }
}

template <typename T, int NPT>
static int launch_chunks(const MambaChunkArgs& a, int E, hipStream_t st) {
  const int NP = (a.N + 15) & ~15, PP = NPT * 16, lc = ld_rows(NP), lx = ld_cols(PP);
  const size_t shm1 = (size_t)MC * (ld_cols(NP) + lx) * 4;
  const size_t shm2 = (size_t)MC * ((lc > MC + 4 ? lc : MC + 4) + (lc > lx ? lc : lx)) * 4;
  static const hipError_t attr = [] {
    const hipError_t e = hipFuncSetAttribute((const void*)mamba_local_k<T, NPT>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024);
    return e != hipSuccess ? e
                           : hipFuncSetAttribute((const void*)mamba_out_k<T, NPT>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024);
  }();
  if (attr != hipSuccess) return (int)attr;
  const dim3 grid(a.NV, a.H);
  hipLaunchKernelGGL((mamba_local_k<T, NPT>), grid, dim3(256), shm1, st, a);
  hipLaunchKernelGGL(mamba_chain_k, dim3((a.N * a.P + 255) / 256, a.H, E), dim3(256), 0, st, a);
  hipLaunchKernelGGL((mamba_out_k<T, NPT>), grid, dim3(256), shm2, st, a);
  return (int)hipGetLastError();
}

extern "C" {

// vent [NV]: the portions' chunks of at most 64 tokens as entries (row0, n, 1, chunk index); tmp fp32 [NV, H, N, P];
// decay fp32 [NV, H]; cent: see mamba_chain_k
int p2p_sm_mamba_scan_chunked(const float* conv, int C, const void* zx, int ldz, int dtoff, const float* dt_bias,
                              const float* A_log, const float* Dp, float* state, float* tmp, float* decay,
                              const int* vent, int NV, const int* cent, int E, float* y, int H, int P, int N, int G,
                              int f32, hipStream_t st) {
  if (E <= 0 || NV <= 0) return 0;
  if (N < 1 || N > 256 || P < 1 || P > 256 || G < 1 || H % G) return (int)hipErrorInvalidValue;
  const int vec = C % 4 == 0 && N % 4 == 0 && P % 4 == 0 && (H * P) % 4 == 0 && (size_t)conv % 16 == 0;
  const MambaChunkArgs a = {conv, C, zx, ldz, dtoff, dt_bias, A_log, Dp, state, tmp, decay, vent, cent, y,
                            H, P, N, G, NV, vec};
#define MCH(NPT) SM_DISPATCH_T(f32, return (launch_chunks<T, NPT>(a, E, st)))
  if (P <= 32) MCH(2);
  else if (P <= 64) MCH(4);
  else if (P <= 128) MCH(8);
  else MCH(16);
#undef MCH
  return 0;
}

}  // extern "C"
