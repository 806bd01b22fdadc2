// The Mamba-2 scan over long portions in chunks of up to 64 tokens on the fp32 matrix instruction
// (v_mfma_f32_16x16x4_f32: products and sums in fp32).  Per head, with A = -exp(A_log), dt = softplus(raw +
// bias), the decays' running sum c_t = sum_{s <= t} A dt_s inside a chunk of n tokens and S the state before it:
//   local pass   L = sum_t exp(c_(n-1) - c_t) dt_t B_t x_t^T                              [N x P]
//   chain        S_next = exp(c_(n-1)) S + L over each portion's chunks, from the slot's state (or zero at
//                position 0); the last one is the slot's new state
//   output pass  y_t = exp(c_t) S^T C_t + sum_{s <= t} exp(c_t - c_s) dt_s (C_t . B_s) x_s + D x_t,  y *= silu(z)
// Every exponent is <= 0, so nothing overflows whatever the step sizes are.  The running sums are kept in 64 bits and
// differences rounded after they are taken: c grows with every token (to -64 at A = 16 and steps of 0.06), and the
// weight between two tokens must not carry the rounding of what decayed before both (off by 1e-5 with drawn steps
// at A = 16, by 5e-4 where small steps follow large ones, against 1e-7).  Sums of the output pass are taken 16 products
// at a time and added up (one chain of up to 320 roundings: 2.3e-7 off a 64-bit run).  One workgroup of four wavefronts per
// (chunk, head); sizes are padded to multiples of 16 with zeros in LDS.
//
// The walk of mamba_scan_k does the same 1 074 M state updates of a prompt of 2048 tokens (64 heads, 128 x 64 states)
// twice, token after token: 240 us each, bound by the chain per token.  The matrix form does 3.7 MFLOP per chunk and
// head: 42 + 30 + 60 us, bound by each workgroup's chain (inputs into LDS, then products) with three and four
// workgroups per CU; the chain by the states' bytes.  LDS is read four numbers at a time.  The products of B and C are formed
// once per group of heads (8 of 64 heads each here), beside the local pass, where heads share them; by every head, with B
// in LDS for it, the state's rows loaded as they are used and z and y a number at a time, the passes took 47 + 30 + 93;
// with one number per LDS read, C and the weights in LDS too, and one row's load in flight per thread while staging 61 +
// 30 + 137.
#include "attn_tile.h"
using namespace sm;

#define MC 64   // tokens of a chunk

// row length in LDS for reads of four neighbours by 16 lanes, a row each: 4 mod 64 (reads of four neighbours along a
// row take any)
static __host__ __device__ __forceinline__ int ld_rows(int n) { return n + ((4 - n) & 63); }

struct MambaChunkArgs {
  const float* conv;   // [R, C] = x | B | C after the convolution
  int C;
  const void* zx;
  int ldz, dtoff;
  const float *dt_bias, *A_log, *Dp;
  float *state, *cs, *decay, *cb;
  const int *vent, *cent;
  float* y;
  int H, P, N, G, NV, vec, vecz;   // vec: four numbers of conv at a time, vecz: of zx and y too
};

// dt and c of the chunk's tokens (zero steps beyond it) by the first wavefront: the loads, then the rest once
// other loads are under way too.  A step below -200 counts as -200: exp() of either is zero, and sums stay finite.
template <typename T>
__device__ __forceinline__ float chunk_dt(const MambaChunkArgs& a, const Entry& en, int h) {
  const int t = threadIdx.x;
  return t < en.n && t < 64 ? ldf((const T*)a.zx, (size_t)(en.row0 + t) * a.ldz + a.dtoff + h) : 0.0f;
}
__device__ __forceinline__ void chunk_steps(const MambaChunkArgs& a, const Entry& en, int h, float raw, float* sdt,
                                            double* sc) {
  if (threadIdx.x >= 64) return;
  const int t = threadIdx.x;
  const float dt = t < en.n ? softplusf_(raw + a.dt_bias[h]) : 0.0f;
  double c = fmaxf(-expf(a.A_log[h]) * dt, -200.0f);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const double v = __shfl_up(c, o, 64);
    if (t >= o) c += v;
  }
  sdt[t] = dt;
  sc[t] = c;
}

// Columns from .. from + 64 U - 1 of n rows of src (row stride ld, `width` numbers) on their way to LDS: 16 lanes take 64
// columns of a row, the loads of all of it in flight
template <int U>
struct Rows {
  f32x4 v[U][MC / 16];
  __device__ __forceinline__ void load(const float* __restrict__ src, size_t ld, int n, int width, int from) {
    const int t0 = threadIdx.x >> 4, c = from + (threadIdx.x & 15) * 4;
#pragma unroll
    for (int i = 0; i < U; i++)
#pragma unroll
      for (int u = 0; u < MC / 16; u++)
        v[i][u] = *(const f32x4*)(src + (size_t)min(t0 + u * 16, n - 1) * ld + min(c + 64 * i, width - 4));
  }
  // zeros from `width` up to `pad` columns and in rows n .. MC-1
  // (odd rows' columns ^ odd)
  __device__ __forceinline__ void store(float* dst, int ldd, int n, int width, int pad, int from, int odd = 0) const {
    const int t0 = threadIdx.x >> 4, c = from + (threadIdx.x & 15) * 4;
#pragma unroll
    for (int i = 0; i < U; i++)
      if (c + 64 * i < pad) {
#pragma unroll
        for (int u = 0; u < MC / 16; u++)
          *(f32x4*)(dst + (t0 + u * 16) * ldd + ((c + 64 * i) ^ ((t0 & 1) * odd))) =
              c + 64 * i < width && t0 + u * 16 < n ? v[i][u] : f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
};

// n rows of `width` numbers of src (row stride ld) -> dst [MC][ldd]; zeros up to `pad` (a multiple of 16, at most
// 256) columns and in rows n .. MC-1; columns below `from` (a multiple of 64) are there already
__device__ __forceinline__ void stage(const float* __restrict__ src, size_t ld, int n, int width, int pad, float* dst,
                                      int ldd, int vec, int from = 0, int odd = 0) {
  if (vec) {
#pragma unroll 1
    for (int c = from; c < pad; c += 64) {
      Rows<1> r;
      r.load(src, ld, n, width, c);
      r.store(dst, ldd, n, width, pad, c, odd);
    }
    return;
  }
  for (int i = threadIdx.x; i < MC * pad; i += 256) {
    const int t = i / pad, c = i % pad;
    dst[t * ldd + (c ^ ((t & 1) * odd))] = (t < n && c < width) ? src[(size_t)t * ld + c] : 0.0f;
  }
}

// Columns of 16 * NPT numbers as the lanes hold them: lane i16 has G = min(NPT, 4) neighbours of every 16 * G, so one
// LDS read (or store) of G numbers serves G fragments.  The same freedom on k: a fragment of four products may hold
// any four rows as long as both operands hold the same ones.
template <int NPT>
struct Cols {
  static constexpr int G = NPT < 4 ? NPT : 4;
  static __device__ __forceinline__ int at(int j, int i16) { return j / G * 16 * G + i16 * G + j % G; }
};
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <typename T>
struct __align__(4 * sizeof(T)) Four {
  T v[4];
};

// B_s . C_t of a chunk's tokens for a group of heads: this wavefront's 16 tokens t = 16 wave + i16 across, s = 16 j + 4 k4 + r
// <= t's block down (w[j][r]), which is the layout that the product with x wants its left operand in.  sB: the group's B
__device__ __forceinline__ void chunk_products(const MambaChunkArgs& a, const float* sB, int LDB, const float* Ct,
                                               f32x4 (&w)[MC / 16]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4, N = a.N;
#pragma unroll
  for (int j = 0; j < MC / 16; j++) w[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int q = 0; q < N; q += 16) {
    const int n0 = q + 4 * k4;
    f32x4 ct = {0.f, 0.f, 0.f, 0.f};            // zero beyond N
    if (a.vec) {
      if (n0 < N) ct = *(const f32x4*)(Ct + n0);
    } else {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (n0 + i < N) ct[i] = Ct[n0 + i];
    }
#pragma unroll
    for (int j = 0; j < MC / 16; j++)
      if (j <= wave) {
        const f32x4 bs = *(const f32x4*)(sB + (j * 16 + i16) * LDB + n0);
        f32x4 p = {0.f, 0.f, 0.f, 0.f};   // 16 products, then the sum
#pragma unroll
        for (int i = 0; i < 4; i++) p = __builtin_amdgcn_mfma_f32_16x16x4f32(bs[i], ct[i], p, 0, 0, 0);
        w[j] += p;
      }
  }
}

// (a.cb) a workgroup per group of heads for its products of B and C, by wavefront, block and lane: the longest, so they
// come first; then the heads'
template <typename T, int NPT>   // value size padded to NPT * 16
__global__ void __launch_bounds__(256) mamba_local_k(MambaChunkArgs a) {
  extern __shared__ __align__(16) float smem[];
  const int groups = a.cb ? a.G : 0;
  if ((int)blockIdx.y < groups) {
    const int g = blockIdx.y, N = a.N, NP = (N + 15) & ~15, LDB = ld_rows(NP);
    const Entry en = load_entry(a.vent, blockIdx.x);
    const float* bc = a.conv + (size_t)en.row0 * a.C + a.H * a.P + g * N;
    stage(bc, a.C, en.n, N, NP, smem, LDB, a.vec);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave * 16 >= en.n) return;
    f32x4 w[MC / 16];
    chunk_products(a, smem, LDB, bc + a.G * N + (size_t)min(wave * 16 + (lane & 15), en.n - 1) * a.C, w);
    f32x4* o = (f32x4*)a.cb + (((size_t)blockIdx.x * a.G + g) * 4 + wave) * (MC / 16) * 64 + lane;
#pragma unroll
    for (int j = 0; j < MC / 16; j++)
      if (j <= wave) o[j * 64] = w[j];
    return;
  }
  __shared__ float sdt[MC];
  __shared__ double sc[MC];
  typedef Cols<NPT> CP;
  const int c = blockIdx.x, h = blockIdx.y - groups, N = a.N, P = a.P;
  const Entry en = load_entry(a.vent, c);
  // two neighbours by 2 x 16 lanes along two rows: 32 columns apart in the banks
  const int NP = (N + 31) & ~31, PP = NPT * 16, LDB = NP, LDX = PP, odd = NP % 64 ? 0 : 32;
  float* sB = smem;
  float* sX = smem + MC * LDB;
  const float raw = chunk_dt<T>(a, en, h);
  const float* row = a.conv + (size_t)en.row0 * a.C;
  const float *B = row + a.H * P + (h / (a.H / a.G)) * N, *X = row + h * P;
  int from = 0;
  if (a.vec) {   // the first 128 columns of B and 64 of X in one wait for memory
    Rows<2> b;
    Rows<1> x;
    b.load(B, a.C, en.n, N, 0);
    x.load(X, a.C, en.n, P, 0);
    b.store(sB, LDB, en.n, N, NP, 0, odd);
    x.store(sX, LDX, en.n, P, PP, 0);
    from = 64;
  }
  stage(B, a.C, en.n, N, NP, sB, LDB, a.vec, 2 * from, odd);
  stage(X, a.C, en.n, P, PP, sX, LDX, a.vec, from);
  chunk_steps(a, en, h, raw, sdt, sc);
  if (threadIdx.x < 64) {   // within the first wavefront
    const double end = __shfl(sc[threadIdx.x], en.n - 1, 64);
    sdt[threadIdx.x] *= expf((float)(end - sc[threadIdx.x]));
    if (threadIdx.x == 0) a.decay[(size_t)c * a.H + h] = expf((float)end);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
  const int steps = (en.n + 3) / 4;
  float* out = a.cs + ((size_t)c * a.H + h) * N * P;
  for (int nb = wave * 32; nb < NP; nb += 128) {   // rows nb + 2 i16 and the one after it
    f32x4 acc[2][NPT];
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int j = 0; j < NPT; j++) acc[u][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int s = 0; s < steps; s++) {
      const f32x2 b = *(const f32x2*)(sB + (4 * s + k4) * LDB + ((nb + 2 * i16) ^ ((k4 & 1) * odd))) * sdt[4 * s + k4];
      float x[NPT];
#pragma unroll
      for (int j = 0; j < NPT; j++) x[j] = sX[(4 * s + k4) * LDX + CP::at(j, i16)];
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int j = 0; j < NPT; j++) acc[u][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[u], x[j], acc[u][j], 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int n = nb + 2 * (k4 * 4 + r) + u;
        if (n >= N) continue;
        float* o = out + (size_t)n * P;
        if (CP::G == 4 && a.vec) {
#pragma unroll
          for (int j = 0; j < NPT; j += 4) {
            const int p = CP::at(j, i16);
            if (p < P) *(f32x4*)(o + p) = f32x4{acc[u][j][r], acc[u][j + 1][r], acc[u][(j + 2) % NPT][r], acc[u][(j + 3) % NPT][r]};
          }
        } else {
#pragma unroll
          for (int j = 0; j < NPT; j++)
            if (CP::at(j, i16) < P) o[CP::at(j, i16)] = acc[u][j][r];
        }
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

// SHARED: the products of B and C come from a.cb
template <typename T, int NPT, bool SHARED, bool VEC>
__global__ void __launch_bounds__(256) mamba_out_k(MambaChunkArgs a) {
  extern __shared__ __align__(16) float smem[];
  __shared__ float sdt[MC];
  __shared__ double sc[MC];
  typedef Cols<NPT> CP;
  const int c = blockIdx.x, h = blockIdx.y, N = a.N, P = a.P, inner = a.H * P, g = h / (a.H / a.G);
  const Entry en = load_entry(a.vent, c);
  const int n = en.n;
  const int NP = (N + 15) & ~15, PP = NPT * 16, LDB = ld_rows(NP), LDX = PP;
  float* sX = smem;
  float* sB = smem + MC * LDX;
  const float* row = a.conv + (size_t)en.row0 * a.C;
  const float* bc = row + inner + g * N;
  const float raw = chunk_dt<T>(a, en, h);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i16 = lane & 15, k4 = lane >> 4;
  const int r0 = wave * 16;                     // this wavefront's 16 tokens
  // w[j]: see chunk_products;  acc: S^T C_t, then y, tokens r0 + 4 k4 + r down
  f32x4 w[MC / 16], acc[NPT];
#pragma unroll
  for (int j = 0; j < NPT; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float* S = a.cs + ((size_t)c * a.H + h) * N * P;
  const float* Ct = bc + a.G * N + (size_t)min(r0 + i16, n - 1) * a.C;
  // rows q .. q + 15 of the state, a lane's four of them, and their C; none behind a branch
  auto load = [&](int q, f32x4& ct, float (&st)[4][NPT]) {
    const int n0 = q + 4 * k4;
    if (VEC) ct = *(const f32x4*)(Ct + min(n0, N - 4));
    else
#pragma unroll
      for (int i = 0; i < 4; i++) ct[i] = Ct[min(n0 + i, N - 1)];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float* Sr = S + (size_t)min(n0 + i, N - 1) * P;
      if constexpr (CP::G == 4 && VEC) {
#pragma unroll
        for (int j = 0; j < NPT; j += 4) {
          const f32x4 v = *(const f32x4*)(Sr + min(CP::at(j, i16), P - 4));
#pragma unroll
          for (int u = 0; u < 4; u++) st[i][(j + u) % NPT] = v[u];
        }
      } else {
#pragma unroll
        for (int j = 0; j < NPT; j++) st[i][j] = Sr[min(CP::at(j, i16), P - 1)];
      }
    }
  };
  auto product = [&](int q, f32x4 ct, const float (&st)[4][NPT]) {
    const int n0 = q + 4 * k4;
#pragma unroll
    for (int i = 0; i < 4; i++) ct[i] = n0 + i < N ? ct[i] : 0.0f;
    f32x4 p[NPT];
#pragma unroll
    for (int j = 0; j < NPT; j++) p[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < NPT; j++) p[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ct[i], st[i][j], p[j], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < NPT; j++) acc[j] += p[j];
  };
  // the state two blocks of rows ahead of its products (which do not need LDS: they go before the barrier)
  f32x4 ct0, ct1;
  float st0[4][NPT], st1[4][NPT];
  load(0, ct0, st0);
  load(16, ct1, st1);
  if (SHARED) {
    const f32x4* o = (const f32x4*)a.cb + (((size_t)c * a.G + g) * 4 + wave) * (MC / 16) * 64 + lane;
#pragma unroll
    for (int j = 0; j < MC / 16; j++) w[j] = o[min(j, wave) * 64];
  }
  const T* zr = (const T*)a.zx + (size_t)en.row0 * a.ldz + h * P;
  constexpr bool Z4 = CP::G == 4 && VEC;
  Four<T> zv[4][NPT / 4 > 0 ? NPT / 4 : 1];
  if (Z4 && a.vecz) {
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int j = 0; j < NPT; j += 4)
        zv[r][j / 4] = *(const Four<T>*)(zr + (size_t)min(r0 + k4 * 4 + r, n - 1) * a.ldz + min(CP::at(j, i16), P - 4));
  }
  if (!SHARED) stage(bc, a.C, n, N, NP, sB, LDB, a.vec);
  stage(row + h * P, a.C, n, P, PP, sX, LDX, a.vec);
  chunk_steps(a, en, h, raw, sdt, sc);
  for (int q = 0; q < NP; q += 32) {
    product(q, ct0, st0);
    load(q + 32, ct0, st0);
    if (q + 16 < NP) product(q + 16, ct1, st1);
    load(q + 48, ct1, st1);
  }
  __syncthreads();
  if (r0 >= n) return;
  if (!SHARED) chunk_products(a, sB, LDB, Ct, w);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const float m = expf((float)sc[r0 + k4 * 4 + r]);
#pragma unroll
    for (int j = 0; j < NPT; j++) acc[j][r] *= m;
  }
  const double ce = sc[r0 + i16];
#pragma unroll
  for (int j = 0; j < MC / 16; j++) {
    if (j > wave) continue;
    f32x4 p[NPT];
    float v[4];
#pragma unroll
    for (int k = 0; k < NPT; k++) p[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int s = j * 16 + k4 * 4 + r;
      v[r] = s <= r0 + i16 ? w[j][r] * expf((float)(ce - sc[s])) * sdt[s] : 0.0f;
#pragma unroll
      for (int k = 0; k < NPT; k++)
        p[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[r], sX[s * LDX + CP::at(k, i16)], p[k], 0, 0, 0);
    }
    if (j == wave) {   // a later token of the block weighs zero, but its input need not be finite: 0 * inf is nan
      float z = 0.0f;
#pragma unroll
      for (int k = 0; k < NPT; k++) not_finite(p[k], z);
      if (__builtin_expect(__any(z != z), 0)) {
#pragma unroll
        for (int k = 0; k < NPT; k++) p[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int q = 0; q < 4; q++)
#pragma unroll
          for (int u = 0; u < 4; u++)      // token 4 q + u of the block
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const float f = __shfl(v[u], q * 16 + 4 * k4 + r, 64);
              if (4 * q + u > 4 * k4 + r) continue;
#pragma unroll
              for (int k = 0; k < NPT; k++) p[k][r] = fmaf(f, sX[(r0 + 4 * q + u) * LDX + CP::at(k, i16)], p[k][r]);
            }
      }
    }
#pragma unroll
    for (int k = 0; k < NPT; k++) acc[k] += p[k];
  }
  const float Dh = a.Dp[h];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int t = r0 + k4 * 4 + r;
    if (t >= n) continue;
    const size_t at = (size_t)(en.row0 + t);
    float* yr = a.y + at * inner + h * P;
    if (Z4 && a.vecz) {
#pragma unroll
      for (int j = 0; j < NPT; j += 4) {
        const int p = CP::at(j, i16);
        if (p >= P) continue;
        const f32x4 x = *(const f32x4*)(sX + t * LDX + p);
        f32x4 o;
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const float z = ldf(zv[r][j / 4].v, u);
          o[u] = (acc[(j + u) % NPT][r] + Dh * x[u]) * (z * sigmoidf_(z));
        }
        *(f32x4*)(yr + p) = o;
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < NPT; j++) {
      const int p = CP::at(j, i16);
      if (p < P) {
        const float z = ldf(zr + (size_t)t * a.ldz, p);
        yr[p] = (acc[j][r] + Dh * sX[t * LDX + p]) * (z * sigmoidf_(z));
      }
    }
  }
}

template <typename T, int NPT>
static int launch_chunks(const MambaChunkArgs& a, int E, hipStream_t st) {
  const int ldb = ld_rows((a.N + 15) & ~15), pp = NPT * 16;
  const size_t shm1 = (size_t)MC * max(((a.N + 31) & ~31) + pp, a.cb ? ldb : 0) * 4;
  const size_t shm2 = (size_t)MC * (pp + (a.cb ? 0 : ldb)) * 4;
  static const hipError_t attr = [] {
    const void* k[] = {(const void*)mamba_local_k<T, NPT>, (const void*)mamba_out_k<T, NPT, false, false>,
                       (const void*)mamba_out_k<T, NPT, false, true>};
    for (const void* f : k)
      if (const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 159 * 1024)) return e;
    return hipSuccess;
  }();
  if (attr != hipSuccess) return (int)attr;
  const dim3 grid(a.NV, a.H);
  hipLaunchKernelGGL((mamba_local_k<T, NPT>), dim3(a.NV, a.H + (a.cb ? a.G : 0)), dim3(256), shm1, st, a);
  hipLaunchKernelGGL(mamba_chain_k, dim3((a.N * a.P + 255) / 256, a.H, E), dim3(256), 0, st, a);
  auto out = a.cb ? a.vec ? mamba_out_k<T, NPT, true, true> : mamba_out_k<T, NPT, true, false>
                  : a.vec ? mamba_out_k<T, NPT, false, true> : mamba_out_k<T, NPT, false, false>;
  hipLaunchKernelGGL(out, grid, dim3(256), shm2, st, a);
  return (int)hipGetLastError();
}

extern "C" {

// vent [NV]: the portions' chunks of at most 64 tokens as entries (row0, n, 1, chunk index); tmp fp32 [NV, H, N, P];
// decay fp32 [NV, H]; cb: fp32 [NV, G, 64, 64], the products of B and C once per group of heads (null: by every head);
// cent: see mamba_chain_k
int p2p_sm_mamba_scan_chunked(const float* conv, int C, const void* zx, int ldz, int dtoff, const float* dt_bias,
                              const float* A_log, const float* Dp, float* state, float* tmp, float* decay,
                              float* cb, const int* vent, int NV, const int* cent, int E, float* y, int H, int P, int N,
                              int G, int f32, hipStream_t st) {
  if (E <= 0 || NV <= 0) return 0;
  if (N < 1 || N > 256 || P < 1 || P > 256 || G < 1 || H % G) return (int)hipErrorInvalidValue;
  const int vec = C % 4 == 0 && N % 4 == 0 && P % 4 == 0 && (H * P) % 4 == 0 && (size_t)conv % 16 == 0;
  const int vecz = vec && ldz % 4 == 0 && (size_t)zx % (f32 ? 16 : 8) == 0 && (size_t)y % 16 == 0;
  const MambaChunkArgs a = {conv, C, zx, ldz, dtoff, dt_bias, A_log, Dp, state, tmp, decay, cb, vent, cent, y,
                            H, P, N, G, NV, vec, vecz};
#define MCH(NPT) SM_DISPATCH_T(f32, return (launch_chunks<T, NPT>(a, E, st)))
  if (P <= 32) MCH(2);
  else if (P <= 64) MCH(4);
  else if (P <= 128) MCH(8);
  else MCH(16);
#undef MCH
  return 0;
}

}  // extern "C"
