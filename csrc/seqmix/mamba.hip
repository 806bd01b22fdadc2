// Mamba-2 (state-space duality) layer pieces.
//   conv : causal per-channel convolution over the x|B|C channels + bias + silu; the inputs
//          before a portion's first token come from the sequence's saved tail (the last
//          taps-1 raw inputs), or are zero at the start of a sequence.
//   scan : per head an N x P fp32 state, S <- exp(-exp(A_log) dt) S + dt B x^T,
//          y = S^T C + D x, y *= silu(z); dt = softplus(raw + bias).  The state sits in
//          registers (a thread holds a run of state rows of one value column); B, C, x, z,
//          dt of a few tokens go through LDS.  Long portions: mamba_chunk.hip.
//   tail : rolls the convolution tail forward after the scan.
// The convolution serves other layers too: it writes fp32 or activation-typed rows.
#include "common.h"
using namespace sm;

// roll: a portion of one token (decode) also moves its tail forward here, every thread that of
// its own channel; the tails of longer portions wait for mamba_tail_k (other rows read them).
template <typename T, typename TO>
__global__ void mamba_conv_k(const T* __restrict__ zx, int ldz, int xoff,
                             const float* __restrict__ cw, const float* __restrict__ cb,
                             float* tail, const int* __restrict__ ent,
                             const int* __restrict__ row_ent, TO* __restrict__ out, int ldo,
                             int C, int K, int roll) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  int r = blockIdx.y;
  if (c >= C) return;
  Entry en = load_entry(ent, row_ent[r]);
  int t = r - en.row0;
  float acc = cb[c];
  for (int kk = 0; kk < K; kk++) {
    int q = t - (K - 1) + kk;
    float val = 0.0f;
    if (q >= 0) val = ldf(zx, (size_t)(en.row0 + q) * ldz + xoff + c);
    else if (en.start > 0) val = tail[((size_t)en.slot * (K - 1) + (K - 1 + q)) * C + c];
    acc += cw[(size_t)c * K + kk] * val;
  }
  stf(out, (size_t)r * ldo + c, acc * sigmoidf_(acc));
  if (roll && en.n == 1) {
    float* tl = tail + (size_t)en.slot * (K - 1) * C + c;
    for (int j = 0; j < K - 1; j++)
      tl[(size_t)j * C] = j + 1 < K - 1 ? (en.start > 0 ? tl[(size_t)(j + 1) * C] : 0.0f)
                                        : ldf(zx, (size_t)r * ldz + xoff + c);
  }
}

// The same for prompts: a thread walks CR consecutive rows of its channel, so the taps are read once
// and every raw input once (its window stays in registers); all of its loads go out together.
// Rows whose window reaches before their portion take it from the tail, row by row.
#define CR 8
template <typename T, typename TO, int KT>
__global__ void mamba_conv_rows_k(const T* __restrict__ zx, int ldz, int xoff,
                                  const float* __restrict__ cw, const float* __restrict__ cb,
                                  const float* __restrict__ tail, const int* __restrict__ ent,
                                  const int* __restrict__ row_ent, TO* __restrict__ out, int ldo,
                                  int R, int C) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x, r0 = blockIdx.y * CR;
  if (c >= C) return;
  float w[KT], u[CR + KT - 1];
#pragma unroll
  for (int kk = 0; kk < KT; kk++) w[kk] = cw[(size_t)c * KT + kk];
#pragma unroll
  for (int i = 0; i < CR + KT - 1; i++)
    u[i] = ldf(zx, (size_t)min(max(r0 + i - (KT - 1), 0), R - 1) * ldz + xoff + c);
  const float b = cb[c];
#pragma unroll
  for (int i = 0; i < CR; i++) {
    const int r = r0 + i;
    if (r >= R) break;
    const Entry en = load_entry(ent, row_ent[r]);
    const int t = r - en.row0;
    float acc = b;
    if (t >= KT - 1) {
#pragma unroll
      for (int kk = 0; kk < KT; kk++) acc += w[kk] * u[i + kk];
    } else {
#pragma unroll
      for (int kk = 0; kk < KT; kk++) {
        const int q = t - (KT - 1) + kk;
        float v = u[i + kk];
        if (q < 0) v = en.start > 0 ? tail[((size_t)en.slot * (KT - 1) + (KT - 1 + q)) * C + c] : 0.0f;
        acc += w[kk] * v;
      }
    }
    stf(out, (size_t)r * ldo + c, acc * sigmoidf_(acc));
  }
}

// One thread owns NSUB consecutive state rows of one value column: thread (p, ns) holds
// S[ns * NSUB + q][p].  Per token it updates them and leaves its share of y = S^T C in LDS;
// the shares are added, D x and the gate applied, once per staged chunk of tokens.
template <typename T, int NSUB>
__global__ void __launch_bounds__(1024)
mamba_scan_k(const float* __restrict__ conv, int C, const T* __restrict__ zx, int ldz, int xoff,
             int dtoff, const float* __restrict__ dt_bias, const float* __restrict__ A_log,
             const float* __restrict__ Dp, float* __restrict__ state, float* __restrict__ tail,
             const int* __restrict__ ent, float* __restrict__ y, int H, int P, int N, int G,
             int K, int CT, int TP, int NS) {
  // a portion from its slot's state (or zero at position 0), state written back
  int e = blockIdx.x / H, h = blockIdx.x % H;
  Entry en = load_entry(ent, e);
  if (en.n <= 0) return;
  extern __shared__ __align__(16) float smem[];
  const int NPAD = NS * NSUB;
  float* sB = smem;                  // [CT][NPAD]
  float* sC = sB + CT * NPAD;        // [CT][NPAD]
  float* sx = sC + CT * NPAD;        // [CT][P]
  float* sz = sx + CT * P;           // [CT][P]
  float* sy = sz + CT * P;           // [CT][NS][P] shares of y
  float* sdt = sy + CT * NS * P;     // [CT]
  float* sdA = sdt + CT;             // [CT]
  int inner = H * P;
  int g = h / (H / G);
  const int p = threadIdx.x % TP, ns = threadIdx.x / TP;
  const bool act = p < P;
  const int n0 = ns * NSUB;
  float S[NSUB];
  float* Sg = state + ((size_t)en.slot * H + h) * N * P;
  const bool from_state = en.start > 0;
#pragma unroll
  for (int q = 0; q < NSUB; q++) {
    // loads at clamped addresses, selected afterwards: the loads stay independent of the
    // bounds tests and go out together
    float v = from_state ? Sg[(size_t)min(n0 + q, N - 1) * P + min(p, P - 1)] : 0.0f;
    S[q] = (act && n0 + q < N) ? v : 0.0f;
  }
  float A = -expf(A_log[h]), Dh = Dp[h], bias = dt_bias[h];
  for (int t0 = 0; t0 < en.n; t0 += CT) {
    int ct = min(CT, en.n - t0);
    __syncthreads();   // the previous chunk's outputs have been read
    for (int idx = threadIdx.x; idx < ct * NPAD; idx += blockDim.x) {
      int t = idx / NPAD, n = idx % NPAD;
      size_t row = (size_t)(en.row0 + t0 + t);
      float b = 0.f, c = 0.f;
      if (n < N) {
        b = conv[row * C + inner + g * N + n];
        c = conv[row * C + inner + G * N + g * N + n];
      }
      sB[idx] = b; sC[idx] = c;
    }
    for (int idx = threadIdx.x; idx < ct * P; idx += blockDim.x) {
      int t = idx / P, q = idx % P;
      size_t row = (size_t)(en.row0 + t0 + t);
      sx[idx] = conv[row * C + h * P + q];
      sz[idx] = ldf(zx, row * ldz + h * P + q);
    }
    for (int t = threadIdx.x; t < ct; t += blockDim.x) {
      size_t row = (size_t)(en.row0 + t0 + t);
      float dt = softplusf_(ldf(zx, row * ldz + dtoff + h) + bias);
      sdt[t] = dt;
      sdA[t] = expf(A * dt);
    }
    __syncthreads();
    if (act) {
      for (int t = 0; t < ct; t++) {
        float dA = sdA[t];
        float dx = sdt[t] * sx[t * P + p];
        const float* bb = sB + t * NPAD + n0;
        const float* cc = sC + t * NPAD + n0;
        float acc = 0.0f;
        // B and C come eight rows at a time, four per read: two at a time, each waited for, the reads were most of the
        // chain (31 tokens, 64 heads of 128 x 64 37.3 -> 26.1 us)
#pragma unroll
        for (int q0 = 0; q0 < NSUB; q0 += 8) {
          float b[8], c[8];
          *(float4*)b = *(const float4*)(bb + q0), *(float4*)(b + 4) = *(const float4*)(bb + q0 + 4);
          *(float4*)c = *(const float4*)(cc + q0), *(float4*)(c + 4) = *(const float4*)(cc + q0 + 4);
#pragma unroll
          for (int q = 0; q < 8; q++) {
            S[q0 + q] = dA * S[q0 + q] + dx * b[q];
            acc += S[q0 + q] * c[q];
          }
        }
        sy[(t * NS + ns) * P + p] = acc;
      }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < ct * P; idx += blockDim.x) {
      int t = idx / P, q = idx % P;
      float acc = 0.0f;
      for (int k = 0; k < NS; k++) acc += sy[(t * NS + k) * P + q];
      acc += Dh * sx[idx];
      float z = sz[idx];
      y[(size_t)(en.row0 + t0 + t) * inner + h * P + q] = acc * (z * sigmoidf_(z));
    }
  }
  if (act) {
#pragma unroll
    for (int q = 0; q < NSUB; q++)
      if (n0 + q < N) Sg[(size_t)(n0 + q) * P + p] = S[q];
  }
}

// new tail = the last K-1 raw inputs of (old tail ++ this portion): one thread per (entry,
// channel); slot j reads old slot j + n or a row of the portion, so ascending j never reads
// a slot it has already written
template <typename T>
__global__ void mamba_tail_k(const T* __restrict__ zx, int ldz, int xoff, float* __restrict__ tail,
                             const int* __restrict__ ent, int C, int K, int skip_single) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  Entry en = load_entry(ent, blockIdx.y);
  if (en.n <= 0 || (skip_single && en.n == 1)) return;
  float* tl = tail + (size_t)en.slot * (K - 1) * C;
  for (int j = 0; j < K - 1; j++) {
    int q = en.n + j - (K - 1);
    float val;
    if (q >= 0) val = ldf(zx, (size_t)(en.row0 + q) * ldz + xoff + c);
    else val = en.start > 0 ? tl[(size_t)(K - 1 + q) * C + c] : 0.0f;
    tl[(size_t)j * C + c] = val;
  }
}

template <typename T, int NSUB>
static int launch_ms(const float* conv, int C, const void* zx, int ldz, int xoff, int dtoff,
                     const float* dt_bias, const float* A_log, const float* Dp, float* state,
                     float* tail, const int* ent, int E, float* y, int H, int P, int N, int G,
                     int K, hipStream_t st) {
  int TP = ((P + 63) / 64) * 64;
  int NS = (N + NSUB - 1) / NSUB;
  int per = 2 * NS * NSUB + 2 * P + NS * P + 2;
  int CT = (48 * 1024) / (per * 4);
  if (CT > 32) CT = 32;
  if (CT < 1) CT = 1;
  size_t shm = (size_t)CT * per * 4;
  hipLaunchKernelGGL((mamba_scan_k<T, NSUB>), dim3(E * H), dim3(TP * NS), shm, st, conv, C,
                     (const T*)zx, ldz, xoff, dtoff, dt_bias, A_log, Dp, state, tail, ent, y, H,
                     P, N, G, K, CT, TP, NS);
  return (int)hipGetLastError();
}

extern "C" {

int p2p_sm_mamba_conv(const void* zx, int ldz, int xoff, const float* cw, const float* cb,
                      float* tail, const int* ent, const int* row_ent, void* out, int ldo,
                      int out_f32, int R, int C, int K, int roll, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  if (K < 1) return (int)hipErrorInvalidValue;
  dim3 g((C + 255) / 256, R), b(256);
  // portions of one token roll their tails in the other kernel, which a step of many rows
  // without the request does not need
  if (!roll && R >= 64 && (K == 4 || K == 3)) {
    g.y = (R + CR - 1) / CR;
#define CONV_ROWS(TO, KT)                                                                         \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((mamba_conv_rows_k<T, TO, KT>), g, b, 0, st, (const T*)zx, \
                                         ldz, xoff, cw, cb, tail, ent, row_ent, (TO*)out, ldo, R, C))
    if (out_f32 && K == 4) CONV_ROWS(float, 4);
    else if (out_f32) CONV_ROWS(float, 3);
    else if (K == 4) CONV_ROWS(T, 4);
    else CONV_ROWS(T, 3);
#undef CONV_ROWS
    return (int)hipGetLastError();
  }
  if (out_f32)
    SM_DISPATCH_T(f32, hipLaunchKernelGGL((mamba_conv_k<T, float>), g, b, 0, st, (const T*)zx, ldz,
                                           xoff, cw, cb, tail, ent, row_ent, (float*)out, ldo, C,
                                           K, roll));
  else
    SM_DISPATCH_T(f32, hipLaunchKernelGGL((mamba_conv_k<T, T>), g, b, 0, st, (const T*)zx, ldz,
                                           xoff, cw, cb, tail, ent, row_ent, (T*)out, ldo, C, K,
                                           roll));
  return (int)hipGetLastError();
}

int p2p_sm_mamba_scan(const float* conv, int C, const void* zx, int ldz, int xoff, int dtoff,
                      const float* dt_bias, const float* A_log, const float* Dp, float* state,
                      float* tail, const int* ent, int E, float* y, int H, int P, int N, int G,
                      int K, int f32, hipStream_t st) {
  if (E <= 0) return 0;
  if (N < 1 || N > 256 || P < 1 || P > 256 || G < 1 || H % G) return (int)hipErrorInvalidValue;
#define MS(NPV)                                                                               \
  SM_DISPATCH_T(f32, return (launch_ms<T, NPV>(conv, C, zx, ldz, xoff, dtoff, dt_bias, A_log, \
                                               Dp, state, tail, ent, E, y, H, P, N, G, K, st)))
  // state rows per thread: 32 where the block (value columns x row slices) fits 1024 threads
  int TPv = ((P + 63) / 64) * 64;
  // (value and state sizes are at most 256, so 64 rows per thread always fit)
  if (TPv * ((N + 31) / 32) <= 1024) MS(32);
  else MS(64);
#undef MS
  return 0;
}

int p2p_sm_mamba_tail(const void* zx, int ldz, int xoff, float* tail, const int* ent, int E, int C,
                      int K, int skip_single, int f32, hipStream_t st) {
  if (E <= 0 || K <= 1) return 0;
  dim3 g((C + 255) / 256, E), b(256);
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(mamba_tail_k<T>, g, b, 0, st, (const T*)zx, ldz, xoff, tail,
                                        ent, C, K, skip_single));
  return (int)hipGetLastError();
}

}  // extern "C"
