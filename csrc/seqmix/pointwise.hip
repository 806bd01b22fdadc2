// Pointwise pieces between the matrix products: tanh in place, sigmoid output gates with
// arbitrary input strides, the clamped gated feed-forward activation
//   g = min(gate, limit), u = clamp(up, -limit, limit), y = g * sigmoid(1.702 g) * (u + 1),
// the silu-gated one, silu(gate) * up, and the tanh cap of the logits.
#include "common.h"
#include "unit_act.h"
using namespace sm;

template <typename T>
__global__ void tanh_k(T* x, int ld, int n, int R) {
  int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c < n) stf(x, (size_t)r * ld + c, tanhf(ldf(x, (size_t)r * ld + c)));
}

// out[r, h * V + v] = o[h * soh + r * sor + v] * sigmoid(g[r * ldg + h * V + v]); VE channels per thread (2048 rows of
// 2048, one / four: 10.1 / 6.8 us)
template <typename T, int VE>
__global__ void sigmoid_gate_k(const T* __restrict__ o, long soh, long sor, const T* __restrict__ g,
                               int ldg, T* __restrict__ out, int ldo, int H, int V,
                               int per_head) {
  int c = (blockIdx.x * blockDim.x + threadIdx.x) * VE, r = blockIdx.y;
  if (c >= H * V) return;
  int h = c / V, v = c % V;
  float x[VE], z[VE];
  ldv<VE>(o, (size_t)h * soh + (size_t)r * sor + v, x);
  if (per_head) z[0] = ldf(g, (size_t)r * ldg + h);
  else ldv<VE>(g, (size_t)r * ldg + c, z);
#pragma unroll
  for (int j = 0; j < VE; j++) x[j] *= sigmoidf_(z[per_head ? 0 : j]);
  stv<VE>(out, (size_t)r * ldo + c, x);
}

template <typename T>
__global__ void ff_act_k(const T* __restrict__ gu, int ld, T* __restrict__ out, int ldo, int F,
                         float limit, float alpha) {
  int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= F) return;
  float g = fminf(ldf(gu, (size_t)r * ld + c), limit);
  float u = fminf(fmaxf(ldf(gu, (size_t)r * ld + F + c), -limit), limit);
  stf(out, (size_t)r * ldo + c, g * sigmoidf_(alpha * g) * (u + 1.0f));
}

// four neighbouring channels per thread (rows and widths that are multiples of 4)
template <typename T>
__global__ void ff_act4_k(const T* __restrict__ gu, int ld, T* __restrict__ out, int ldo, int F,
                          float limit, float alpha) {
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * 4, r = blockIdx.y;
  if (c >= F) return;
  struct alignas(4 * sizeof(T)) V4 { T v[4]; };
  const V4 gv = *(const V4*)(gu + (size_t)r * ld + c), uv = *(const V4*)(gu + (size_t)r * ld + F + c);
  V4 o;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float g = fminf(ldf(gv.v, i), limit), u = fminf(fmaxf(ldf(uv.v, i), -limit), limit);
    stf(o.v, i, g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * alpha * g)) *
                    (u + 1.0f));
  }
  *(V4*)(out + (size_t)r * ldo + c) = o;
}

// [gate | up] -> act(gate) * up; act: 0 silu, 1 gelu (tanh form).  Bound by memory and by the number of wavefronts:
// V = 4 neighbours per thread where rows and channels allow it (a feed-forward of Tarunex's width-2048 stack,
// prompt of 2048 rows in bf16: one channel per thread 21.1 us, four 10.9 us).
template <typename T, int V>
__global__ void __launch_bounds__(256) glu_act_k(const T* __restrict__ gu, int ld, T* __restrict__ out, int ldo,
                                                 int F, int act) {
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * V, r = blockIdx.y;
  if (c >= F) return;
  struct alignas(V * sizeof(T)) VV { T v[V]; };
  const VV gv = *(const VV*)(gu + (size_t)r * ld + c), uv = *(const VV*)(gu + (size_t)r * ld + F + c);
  VV o;
#pragma unroll
  for (int i = 0; i < V; i++) {
    const float g = ldf(gv.v, i);
    const float a = act == 1 ? gelu_tanhf_(g) : g * sigmoidf_(g);
    stf(o.v, i, a * ldf(uv.v, i));
  }
  *(VV*)(out + (size_t)r * ldo + c) = o;
}

// out[r, c] = relu(u[r, c])^2 * sigmoid(g[r]): an ungated squared-relu unit whose result is
// weighted by one gate per row (g == nullptr: no gate)
template <typename T>
__global__ void relu2_gate_k(const T* __restrict__ u, int ld, const T* __restrict__ g, int ldg,
                             T* __restrict__ out, int ldo, int F) {
  int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= F) return;
  float v = fmaxf(ldf(u, (size_t)r * ld + c), 0.0f);
  float w = g ? sigmoidf_(ldf(g, (size_t)r * ldg)) : 1.0f;
  stf(out, (size_t)r * ldo + c, v * v * w);
}

template <typename T>
__global__ void softcap_k(const T* __restrict__ y, int ld, float* __restrict__ out, int n,
                          float cap, float scale) {
  int c = blockIdx.x * blockDim.x + threadIdx.x, r = blockIdx.y;
  if (c >= n) return;
  float z = ldf(y, (size_t)r * ld + c) * scale;
  out[(size_t)r * n + c] = cap > 0.0f ? cap * tanhf(z / cap) : z;
}

// Words between page-locked host memory and device memory, past the caches (a captured step's first and last kernel: its
// metadata in, its tokens out)
__global__ void copy_words_k(const int* src, int* dst, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int v = __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(dst + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// What a step's layers derive from its entries (row0, n, start, slot), formed on the device: a copy of it from the host waits for
// all that is under way, and the layers behind it for the host (a prompt of 40 rows, two or three of them: Regesun 893 -> 827 us,
// Rasepel 880 -> 836, Tarunex 760 -> 719).  Entries of
// `least` rows and more are cut into pieces of at most `size` consecutive rows: (row, rows) to units, or (row, rows, 1, piece) to
// pieces and (first piece, pieces, start, slot) to whole; shorter ones go to rest as they are.
__global__ void __launch_bounds__(256) step_tables_k(const int4* __restrict__ ent, int E, int size, int least, int2* __restrict__ units,
                                                     int4* __restrict__ pieces, int4* __restrict__ whole, int4* __restrict__ rest) {
  __shared__ int4 s[256];
  int p0 = 0, w = 0, r = 0;   // pieces, whole and other entries so far
  for (int base = 0; base < E; base += 256) {
    __syncthreads();
    if (base + (int)threadIdx.x < E) s[threadIdx.x] = ent[base + threadIdx.x];
    __syncthreads();
    for (int i = 0; i < min(256, E - base); i++) {
      const int4 e = s[i];
      if (e.y < least) {
        if (threadIdx.x == 0) rest[r] = e;
        r++;
        continue;
      }
      const int n = (e.y + size - 1) / size;
      for (int k = threadIdx.x; k < n; k += 256) {
        const int row = e.x + k * size, rows = min(size, e.y - k * size);
        if (units) units[p0 + k] = make_int2(row, rows);
        else pieces[p0 + k] = make_int4(row, rows, 1, p0 + k);
      }
      if (!units && threadIdx.x == 0) whole[w] = make_int4(p0, n, e.z, e.w);
      p0 += n, w++;
    }
  }
}

extern "C" {

// units, or pieces, whole and rest (which may be null where no entry is shorter than `least`): see step_tables_k
int p2p_sm_step_tables(const int* ent, int E, int size, int least, int* units, int* pieces, int* whole, int* rest, hipStream_t st) {
  if (E <= 0) return 0;
  if (size < 1 || (units ? least > 0 : !pieces || !whole) || (size_t)ent % 16 || (size_t)units % 8 ||
      ((size_t)pieces | (size_t)whole | (size_t)rest) % 16)
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(step_tables_k, dim3(1), dim3(256), 0, st, (const int4*)ent, E, size, least, (int2*)units, (int4*)pieces,
                     (int4*)whole, (int4*)rest);
  return (int)hipGetLastError();
}

int p2p_sm_copy_words(const int* src, int* dst, int n, hipStream_t st) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(copy_words_k, dim3((n + 255) / 256), dim3(256), 0, st, src, dst, n);
  return (int)hipGetLastError();
}

int p2p_sm_glu_act(const void* gu, int ld, void* out, int ldo, int R, int F, int act, int f32,
                   hipStream_t st) {
  if (R <= 0) return 0;
  const size_t al = f32 ? 16 : 8;
  // above 256 channels: fewer leave most of a workgroup idle (2048 rows of 64, one / four per thread: 2.7 / 2.9 us,
  // of 300 3.8 / 3.2)
  if (F > 256 && F % 4 == 0 && ld % 4 == 0 && ldo % 4 == 0 && (size_t)gu % al == 0 && (size_t)out % al == 0)
    SM_DISPATCH_T(f32, hipLaunchKernelGGL((glu_act_k<T, 4>), dim3((F + 1023) / 1024, R), dim3(256), 0, st,
                                           (const T*)gu, ld, (T*)out, ldo, F, act));
  else
    SM_DISPATCH_T(f32, hipLaunchKernelGGL((glu_act_k<T, 1>), dim3((F + 255) / 256, R), dim3(256), 0, st,
                                           (const T*)gu, ld, (T*)out, ldo, F, act));
  return (int)hipGetLastError();
}

int p2p_sm_relu2_gate(const void* u, int ld, const void* gt, int ldg, void* out, int ldo, int R,
                      int F, int f32, hipStream_t st) {
  if (R <= 0 || F <= 0) return 0;
  dim3 g((F + 255) / 256, R), b(256);
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(relu2_gate_k<T>, g, b, 0, st, (const T*)u, ld,
                                         (const T*)gt, ldg, (T*)out, ldo, F));
  return (int)hipGetLastError();
}

int p2p_sm_softcap(const void* y, int ld, float* out, int R, int n, float cap, float scale,
                   int f32, hipStream_t st) {
  if (R <= 0 || n <= 0) return 0;
  dim3 g((n + 255) / 256, R), b(256);
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(softcap_k<T>, g, b, 0, st, (const T*)y, ld, out, n, cap,
                                         scale));
  return (int)hipGetLastError();
}

int p2p_sm_tanh(void* x, int ld, int n, int R, int f32, hipStream_t st) {
  if (R <= 0 || n <= 0) return 0;
  dim3 g((n + 255) / 256, R), b(256);
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(tanh_k<T>, g, b, 0, st, (T*)x, ld, n, R));
  return (int)hipGetLastError();
}

int p2p_sm_sigmoid_gate(const void* o, long soh, long sor, const void* gt, int ldg, void* out,
                        int ldo, int R, int H, int V, int per_head, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  const size_t al = f32 ? 16 : 8;
#define GATE(VE)                                                                                             \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((sigmoid_gate_k<T, VE>), dim3((H * V + 256 * VE - 1) / (256 * VE), R), \
                                         dim3(256), 0, st, (const T*)o, soh, sor, (const T*)gt, ldg, (T*)out, ldo, H, V, \
                                         per_head))
  if (V % 4 == 0 && soh % 4 == 0 && sor % 4 == 0 && ldo % 4 == 0 && ((size_t)o | (size_t)out) % al == 0 &&
      (per_head || (ldg % 4 == 0 && (size_t)gt % al == 0)))
    GATE(4);
  else GATE(1);
#undef GATE
  return (int)hipGetLastError();
}

int p2p_sm_ff_act(const void* gu, int ld, void* out, int ldo, int R, int F, float limit,
                  float alpha, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  const size_t al = f32 ? 16 : 8;
  if (F % 4 == 0 && ld % 4 == 0 && ldo % 4 == 0 && (size_t)gu % al == 0 && (size_t)out % al == 0) {
    SM_DISPATCH_T(f32, hipLaunchKernelGGL(ff_act4_k<T>, dim3((F + 1023) / 1024, R), dim3(256), 0, st,
                                           (const T*)gu, ld, (T*)out, ldo, F, limit, alpha));
    return (int)hipGetLastError();
  }
  dim3 g((F + 255) / 256, R), b(256);
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(ff_act_k<T>, g, b, 0, st, (const T*)gu, ld, (T*)out, ldo,
                                         F, limit, alpha));
  return (int)hipGetLastError();
}

}  // extern "C"
