// Embedding with learned positions, RMS norms over fp32 or activation-typed rows (whole
// row or equal parts, optional scatter of the rows), and the post-sublayer passes on the fp32
// residual stream: norm + layer scale + residual add, and the gated form
// x += N(y * sigmoid(g + b)) * w with the norm N taken over equal parts of the row.
#include "common.h"
using namespace sm;

// VE numbers per load (four: 8 rows of 2048 9.1 -> 4.3 us in a step, 2048 rows 15.1 -> 10.8)
template <typename T, int VE>
__global__ void embed_pos_k(const T* __restrict__ embed, const T* __restrict__ ptab,
                            const int* __restrict__ ids, const int* __restrict__ pos,
                            float* __restrict__ out, int W, int has_pos) {
  int r = blockIdx.x;
  size_t eo = (size_t)ids[r] * W, po = (size_t)pos[r] * W;
  for (int i = threadIdx.x * VE; i < W; i += blockDim.x * VE) {
    float v[VE], p[VE];
    ldv<VE>(embed, eo + i, v);
    if (has_pos) {
      ldv<VE>(ptab, po + i, p);
#pragma unroll
      for (int j = 0; j < VE; j++) v[j] += p[j];
    }
    stv<VE>(out, (size_t)r * W + i, v);
  }
}

// Row passes keep their row in registers: NC chunks of VE neighbours per thread, a workgroup of 256 threads per row.
// VE = 4 wherever the operands allow it, with the smallest NC that holds the row: these passes are bound by memory
// where there are many rows and by their chain of loads, two sums and code fetch where there are few, and one load per
// number with registers for 4096 numbers costs both.  Microseconds in bf16, one number per load -> four: post-norm
// pass of 8 rows of 2048 6.6 -> 3.8, of 2048 rows 23.6 -> 12.5 (4.0 TB/s), 4096 wide 52.3 -> 25.5; residual pass of
// 2048 rows of 2048 18.3 -> 11.0, with two outputs 15.1 -> 11.3; norm of 2048 rows in 8 parts of 128 28.5 -> 6.8.
// VE = 1, NC = 16 takes odd widths and unaligned operands, NC = 0 reads longer rows twice.
#define NV 16   // values per thread of the passes that take one number per load: rows of up to 256 * NV are read once

// one block per (row, part): out = x / sqrt(mean(x^2) + eps) * w
template <typename TI, typename TO, int VE, int NC>
__global__ void __launch_bounds__(256) rmsnorm_k(const TI* __restrict__ x, int ldx, const float* __restrict__ w,
                                                 TO* __restrict__ out, int ldo, const int* __restrict__ in_rows,
                                                 const int* __restrict__ out_rows, int n, int parts, float eps) {
  __shared__ float red[16];
  int r = blockIdx.x / parts, g = blockIdx.x % parts;
  int np = n / parts;
  int ri = in_rows ? in_rows[r] : r;
  int ro = out_rows ? out_rows[r] : r;
  const TI* xr = x + (size_t)ri * ldx + (size_t)g * np;
  const float* wp = w ? w + g * np : nullptr;
  if constexpr (NC > 0) {
    // the row and its weights are loaded once, before the reduction
    float v[NC][VE], wv[NC][VE];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) v[k][j] = 0.0f, wv[k][j] = 1.0f;
      if (i < np) {
        ldv<VE>(xr, i, v[k]);
        if (wp) ldv<VE>(wp, i, wv[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
      for (int j = 0; j < VE; j++) ss += v[k][j] * v[k][j];
    ss = block_sum(ss, red);
    if (ro < 0) return;
    float rs = 1.0f / sqrtf(ss / (float)np + eps);
    TO* o = out + (size_t)ro * ldo + (size_t)g * np;
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) v[k][j] = v[k][j] * rs * wv[k][j];
      if (i < np) stv<VE>(o, i, v[k]);
    }
    return;
  }
  float ss = 0.0f;
  for (int i = threadIdx.x; i < np; i += blockDim.x) {
    float v = ldf(xr, i);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  if (ro < 0) return;
  float rs = 1.0f / sqrtf(ss / (float)np + eps);
  TO* o = out + (size_t)ro * ldo + (size_t)g * np;
  for (int i = threadIdx.x; i < np; i += blockDim.x) {
    float v = ldf(xr, i) * rs;
    if (wp) v *= wp[i];
    stf(o, i, v);
  }
}

// x += y / sqrt(mean(y^2) + eps) * w * ls   (x fp32 residual); with h also the next sublayer's
// input from the updated row: x / sqrt(mean(x^2) + eps) * w2, or without w2 the row as it is
template <typename T, int VE, int NC>
__global__ void __launch_bounds__(256) norm_scale_add_k(float* __restrict__ x, const T* __restrict__ y, int ldy,
                                                        const float* __restrict__ w, const float* __restrict__ ls,
                                                        int n, float eps, const float* __restrict__ w2,
                                                        T* __restrict__ h, int ldh) {
  __shared__ float red[16];
  int r = blockIdx.x;
  const T* yr = y + (size_t)r * ldy;
  float* xr = x + (size_t)r * n;
  if constexpr (NC > 0) {
    // y, the weights and the residual are loaded once, before the first reduction
    float v[NC][VE], wv[NC][VE], lv[NC][VE], xv[NC][VE], nw[NC][VE];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) v[k][j] = wv[k][j] = xv[k][j] = nw[k][j] = 0.0f, lv[k][j] = 1.0f;
      if (i < n) {
        ldv<VE>(yr, i, v[k]);
        ldv<VE>(w, i, wv[k]);
        ldv<VE>(xr, i, xv[k]);
        if (ls) ldv<VE>(ls, i, lv[k]);
        if (w2) ldv<VE>(w2, i, nw[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < NC; k++)
#pragma unroll
      for (int j = 0; j < VE; j++) ss += v[k][j] * v[k][j];
    ss = block_sum(ss, red);
    float rs = 1.0f / sqrtf(ss / (float)n + eps);
    float s2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) {
        xv[k][j] = xv[k][j] + v[k][j] * rs * (wv[k][j] * lv[k][j]);
        s2 += xv[k][j] * xv[k][j];
      }
      if (i < n) stv<VE>(xr, i, xv[k]);
    }
    if (!h) return;
    if (w2) {
      s2 = block_sum(s2, red);
      float r2 = 1.0f / sqrtf(s2 / (float)n + eps);
#pragma unroll
      for (int k = 0; k < NC; k++)
#pragma unroll
        for (int j = 0; j < VE; j++) xv[k][j] *= r2 * nw[k][j];
    }
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
      if (i < n) stv<VE>(h + (size_t)r * ldh, i, xv[k]);
    }
    return;
  }
  float ss = 0.0f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    float v = ldf(yr, i);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  float rs = 1.0f / sqrtf(ss / (float)n + eps);
  float s2 = 0.0f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    float v = xr[i] + ldf(yr, i) * rs * (ls ? w[i] * ls[i] : w[i]);
    xr[i] = v;
    if (h && !w2) stf(h, (size_t)r * ldh + i, v);
    s2 += v * v;
  }
  if (!w2) return;
  s2 = block_sum(s2, red);
  float r2 = 1.0f / sqrtf(s2 / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += blockDim.x)   // each thread re-reads its own writes
    stf(h, (size_t)r * ldh + i, xr[i] * r2 * w2[i]);
}

// x += a (+ b) on the fp32 residual, the addends summed first (fp32); with w2 also the next
// layer's input h = x / sqrt(mean(x^2) + eps) * w2 from the updated row
template <typename T, int VE, int NC>
__global__ void __launch_bounds__(256) add_norm_k(float* __restrict__ x, const T* __restrict__ a, int lda,
                                                  const T* __restrict__ b, int ldb, int n, float eps,
                                                  const float* __restrict__ w2, T* __restrict__ h, int ldh) {
  __shared__ float red[16];
  int r = blockIdx.x;
  const T* ar = a + (size_t)r * lda;
  const T* br = b ? b + (size_t)r * ldb : nullptr;
  float* xr = x + (size_t)r * n;
  if constexpr (NC > 0) {
    // every load goes out before the first store (a store to x in between would hold back
    // the later loads of x)
    float xv[NC][VE], wv[NC][VE], yv[NC][VE], bv[NC][VE];
    float s2 = 0.0f;
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) xv[k][j] = wv[k][j] = yv[k][j] = bv[k][j] = 0.0f;
      if (i < n) {
        ldv<VE>(ar, i, yv[k]);
        if (br) ldv<VE>(br, i, bv[k]);
        if (w2) ldv<VE>(w2, i, wv[k]);
        ldv<VE>(xr, i, xv[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) {
        xv[k][j] += yv[k][j] + bv[k][j];
        s2 += xv[k][j] * xv[k][j];
      }
      if (i < n) stv<VE>(xr, i, xv[k]);
    }
    if (!w2) return;
    s2 = block_sum(s2, red);
    float r2 = 1.0f / sqrtf(s2 / (float)n + eps);
#pragma unroll
    for (int k = 0; k < NC; k++) {
      const int i = (threadIdx.x + k * 256) * VE;
#pragma unroll
      for (int j = 0; j < VE; j++) xv[k][j] *= r2 * wv[k][j];
      if (i < n) stv<VE>(h + (size_t)r * ldh, i, xv[k]);
    }
    return;
  }
  float s2 = 0.0f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    float y = ldf(ar, i);
    if (br) y += ldf(br, i);
    float v = xr[i] + y;
    xr[i] = v;
    s2 += v * v;
  }
  if (!w2) return;
  s2 = block_sum(s2, red);
  float r2 = 1.0f / sqrtf(s2 / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += blockDim.x)   // each thread re-reads its own writes
    stf(h, (size_t)r * ldh + i, xr[i] * r2 * w2[i]);
}

// x += a + b + rows + vec + sum_k cw[r, k] * cy[r * top + k] on the fp32 residual (each addend
// optional; a, b, cy activation typed, rows fp32 [R, n], vec fp32 [n], cw fp32 [R, top]: the
// weighted sum of a token's routed expert outputs; summed first, in fp32), then up to two normed copies of the
// updated row, h_i = x / sqrt(mean(x^2) + eps) * w_i, where w_i is a vector (ws_i = 1) or one
// number for all channels (ws_i = 0): two sublayers that read the same row through norms of
// their own get their inputs from one pass over it.
template <typename T, int VE, int NC>
__global__ void __launch_bounds__(256) add_norm2_k(float* __restrict__ x, const T* __restrict__ a, int lda,
                            const T* __restrict__ b, int ldb, const float* __restrict__ rows,
                            const float* __restrict__ vec, int n, float eps,
                            const float* __restrict__ w1, int ws1, T* __restrict__ h1, int ld1,
                            const float* __restrict__ w2, int ws2, T* __restrict__ h2, int ld2,
                            const T* __restrict__ cy, int ldcy, const float* __restrict__ cw,
                            int top) {
  __shared__ float red[16];
  int r = blockIdx.x;
  const T* cyr = cy ? cy + (size_t)r * top * ldcy : nullptr;
  const float* cwr = cy ? cw + (size_t)r * top : nullptr;
  const T* ar = a ? a + (size_t)r * lda : nullptr;
  const T* br = b ? b + (size_t)r * ldb : nullptr;
  const float* er = rows ? rows + (size_t)r * n : nullptr;
  float* xr = x + (size_t)r * n;
  const bool adds = ar || br || er || vec || cyr;
  // weights that are one number are read before the reduction
  const float g1 = (w1 && !ws1) ? w1[0] : 1.0f, g2 = (w2 && !ws2) ? w2[0] : 1.0f;
  if constexpr (NC > 0) {
    // every load goes out before the first store; each addend's loads form one batch (the
    // tests for the optional addends stay outside the unrolled loops)
    float xv[NC][VE], yv[NC][VE];
    float s2 = 0.0f;
    auto at = [&](int k) { return (int)(threadIdx.x + k * 256) * VE; };
    auto add = [&](auto* p, float w) {
      float v[NC][VE];
#pragma unroll
      for (int k = 0; k < NC; k++) ldv<VE>(p, at(k) < n ? at(k) : 0, v[k]);
#pragma unroll
      for (int k = 0; k < NC; k++)
#pragma unroll
        for (int j = 0; j < VE; j++) yv[k][j] += w * v[k][j];
    };
#pragma unroll
    for (int k = 0; k < NC; k++) {
      ldv<VE>(xr, at(k) < n ? at(k) : 0, xv[k]);
#pragma unroll
      for (int j = 0; j < VE; j++) yv[k][j] = 0.0f;
    }
    if (ar) add(ar, 1.0f);
    if (br) add(br, 1.0f);
    if (er) add(er, 1.0f);
    if (vec) add(vec, 1.0f);
    if (cyr) {
      // two experts at a time, so that a choice of two is one batch of loads
      for (int t = 0; t < top; t += 2) {
        const bool two = t + 1 < top;
        const float wa = cwr[t], wb = two ? cwr[t + 1] : 0.0f;
        const T* ya = cyr + (size_t)t * ldcy;
        const T* yb = cyr + (size_t)(two ? t + 1 : t) * ldcy;
        float va[NC][VE], vb[NC][VE];
#pragma unroll
        for (int k = 0; k < NC; k++) {
          ldv<VE>(ya, at(k) < n ? at(k) : 0, va[k]);
          ldv<VE>(yb, at(k) < n ? at(k) : 0, vb[k]);
        }
#pragma unroll
        for (int k = 0; k < NC; k++)
#pragma unroll
          for (int j = 0; j < VE; j++) yv[k][j] += wa * va[k][j] + wb * vb[k][j];
      }
    }
#pragma unroll
    for (int k = 0; k < NC; k++) {
#pragma unroll
      for (int j = 0; j < VE; j++) {
        xv[k][j] = at(k) < n ? xv[k][j] + yv[k][j] : 0.0f;
        s2 += xv[k][j] * xv[k][j];
      }
      if (adds && at(k) < n) stv<VE>(xr, at(k), xv[k]);
    }
    if (!w1) return;
    s2 = block_sum(s2, red);
    float r2 = 1.0f / sqrtf(s2 / (float)n + eps);
    auto put = [&](const float* w, int ws, float g, T* h) {
#pragma unroll
      for (int k = 0; k < NC; k++) {
        if (at(k) >= n) continue;
        float wv[VE], o[VE];
        if (ws) ldv<VE>(w, at(k), wv);
#pragma unroll
        for (int j = 0; j < VE; j++) o[j] = xv[k][j] * r2 * (ws ? wv[j] : g);
        stv<VE>(h, at(k), o);
      }
    };
    put(w1, ws1, g1, h1 + (size_t)r * ld1);
    if (w2) put(w2, ws2, g2, h2 + (size_t)r * ld2);
    return;
  }
  float s2 = 0.0f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    float y = 0.0f;
    if (ar) y += ldf(ar, i);
    if (br) y += ldf(br, i);
    if (er) y += er[i];
    if (vec) y += vec[i];
    if (cyr)
      for (int t = 0; t < top; t++) y += cwr[t] * ldf(cyr, (size_t)t * ldcy + i);
    float v = xr[i] + y;
    if (adds) xr[i] = v;
    s2 += v * v;
  }
  if (!w1) return;
  s2 = block_sum(s2, red);
  float r2 = 1.0f / sqrtf(s2 / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += blockDim.x) {   // each thread re-reads its own writes
    float v = xr[i] * r2;
    stf(h1, (size_t)r * ld1 + i, v * (ws1 ? w1[i] : g1));
    if (w2) stf(h2, (size_t)r * ld2 + i, v * (ws2 ? w2[i] : g2));
  }
}

// out[r] = embed[ids[r]] * scale as fp32, and (optionally) the same row in the activation type
template <typename T, int VE>
__global__ void embed_rows_k(const T* __restrict__ embed, const int* __restrict__ ids,
                             float* __restrict__ out, T* __restrict__ h, int ldh, int W,
                             float scale) {
  int r = blockIdx.x;
  size_t eo = (size_t)ids[r] * W;
  for (int i = threadIdx.x * VE; i < W; i += blockDim.x * VE) {
    float v[VE];
    ldv<VE>(embed, eo + i, v);
#pragma unroll
    for (int j = 0; j < VE; j++) v[j] *= scale;
    stv<VE>(out, (size_t)r * W + i, v);
    if (h) stv<VE>(h, (size_t)r * ldh + i, v);
  }
}

// one block per (row, part): x += v / sqrt(mean(v^2) + eps) * w with v = y * sigmoid(g + gb),
// the mean over the part; h (optional) receives the updated residual in the activation type
template <typename T>
__global__ void gate_norm_add_k(float* __restrict__ x, const T* __restrict__ y, int ldy,
                                const T* __restrict__ g, int ldg, const float* __restrict__ gb,
                                const float* __restrict__ w, int n, int parts, float eps,
                                T* __restrict__ h, int ldh) {
  __shared__ float red[16];
  int r = blockIdx.x / parts, p = blockIdx.x % parts;
  int np = n / parts, c0 = p * np;
  const T* yr = y + (size_t)r * ldy + c0;
  const T* gr = g + (size_t)r * ldg + c0;
  float* xr = x + (size_t)r * n + c0;
  if (np <= NV * (int)blockDim.x) {
    float v[NV], wv[NV], xv[NV];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NV; k++) {
      int i = threadIdx.x + k * blockDim.x;
      bool ok = i < np;
      float yv = ok ? ldf(yr, i) : 0.0f;
      float gv = ok ? ldf(gr, i) + gb[c0 + i] : 0.0f;
      wv[k] = ok ? w[c0 + i] : 0.0f;
      xv[k] = ok ? xr[i] : 0.0f;
      v[k] = yv * sigmoidf_(gv);
      ss += v[k] * v[k];
    }
    ss = block_sum(ss, red);
    float rs = 1.0f / sqrtf(ss / (float)np + eps);
#pragma unroll
    for (int k = 0; k < NV; k++) {
      int i = threadIdx.x + k * blockDim.x;
      if (i < np) {
        float nv = xv[k] + v[k] * rs * wv[k];
        xr[i] = nv;
        if (h) stf(h, (size_t)r * ldh + c0 + i, nv);
      }
    }
    return;
  }
  float ss = 0.0f;
  for (int i = threadIdx.x; i < np; i += blockDim.x) {
    float v = ldf(yr, i) * sigmoidf_(ldf(gr, i) + gb[c0 + i]);
    ss += v * v;
  }
  ss = block_sum(ss, red);
  float rs = 1.0f / sqrtf(ss / (float)np + eps);
  for (int i = threadIdx.x; i < np; i += blockDim.x) {
    float v = ldf(yr, i) * sigmoidf_(ldf(gr, i) + gb[c0 + i]);
    float nv = xr[i] + v * rs * w[c0 + i];
    xr[i] = nv;
    if (h) stf(h, (size_t)r * ldh + c0 + i, nv);
  }
}

// out = x / sqrt(mean(x^2) + eps) * w * sigmoid(g): the norm of a whole fp32 row (all heads of a
// recurrence together) with a gate per channel, on the way into an output projection
template <typename T, int NR>   // NR: values a thread keeps (rows of up to 256 * NR numbers are read once)
__global__ void norm_gate_k(const float* __restrict__ x, int ldx, const float* __restrict__ w,
                            const T* __restrict__ g, int ldg, T* __restrict__ out, int ldo, int n,
                            float eps) {
  __shared__ float red[16];
  const int r = blockIdx.x;
  const float* xr = x + (size_t)r * ldx;
  const T* gr = g + (size_t)r * ldg;
  T* o = out + (size_t)r * ldo;
  if (n <= NR * (int)blockDim.x) {
    float v[NR], m[NR];
    float ss = 0.0f;
#pragma unroll
    for (int k = 0; k < NR; k++) {
      int i = threadIdx.x + k * blockDim.x;
      int ic = i < n ? i : 0;
      v[k] = xr[ic];
      m[k] = w[ic] * sigmoidf_(ldf(gr, ic));
    }
#pragma unroll
    for (int k = 0; k < NR; k++) {
      if (threadIdx.x + k * blockDim.x >= (unsigned)n) v[k] = 0.0f;
      ss += v[k] * v[k];
    }
    ss = block_sum(ss, red);
    float rs = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
    for (int k = 0; k < NR; k++) {
      int i = threadIdx.x + k * blockDim.x;
      if (i < n) stf(o, i, v[k] * rs * m[k]);
    }
    return;
  }
  float ss = 0.0f;
  for (int i = threadIdx.x; i < n; i += blockDim.x) ss += xr[i] * xr[i];
  ss = block_sum(ss, red);
  float rs = 1.0f / sqrtf(ss / (float)n + eps);
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    stf(o, i, xr[i] * rs * w[i] * sigmoidf_(ldf(gr, i)));
}

// which form takes rows of n numbers (four neighbours per load if by4): chunks of four, 0: one number per load in
// registers, -1: read twice
static int row_form(int n, bool by4) {
  if (n > 256 * NV) return -1;
  if (!by4) return 0;
  return n <= 1024 ? 1 : n <= 2048 ? 2 : 4;
}
#define ROW_FORM(V, C, ...)        \
  {                                \
    constexpr int VE = V, NC = C;  \
    __VA_ARGS__;                   \
    break;                         \
  }
#define ROW_FORMS(form, ...)                    \
  do {                                          \
    switch (form) {                             \
      case 1: ROW_FORM(4, 1, __VA_ARGS__)       \
      case 2: ROW_FORM(4, 2, __VA_ARGS__)       \
      case 4: ROW_FORM(4, 4, __VA_ARGS__)       \
      case 0: ROW_FORM(1, NV, __VA_ARGS__)      \
      default: ROW_FORM(1, 0, __VA_ARGS__)      \
    }                                           \
  } while (0)

extern "C" {

int p2p_sm_norm_gate(const float* x, int ldx, const float* w, const void* g, int ldg, void* out,
                     int ldo, int R, int n, float eps, int f32, hipStream_t st) {
  if (R <= 0 || n <= 0) return 0;
#define NG(NR)                                                                                   \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((norm_gate_k<T, NR>), dim3(R), dim3(256), 0, st, x, ldx, w, \
                                         (const T*)g, ldg, (T*)out, ldo, n, eps))
  if (n <= 256 * 4) NG(4);
  else if (n <= 256 * 8) NG(8);
  else NG(16);
#undef NG
  return (int)hipGetLastError();
}

int p2p_sm_embed_rows(const void* embed, const int* ids, float* out, void* h, int ldh, int R,
                      int W, float scale, int f32, hipStream_t st) {
  if (R <= 0) return 0;
#define EMBED(VE)                                                                       \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((embed_rows_k<T, VE>), dim3(R), dim3(256), 0, st, \
                                         (const T*)embed, ids, out, (T*)h, ldh, W, scale))
  const size_t a4 = f32 ? 16 : 8;
  if (W % 4 == 0 && (size_t)embed % a4 == 0 && (size_t)out % 16 == 0 && (!h || ((size_t)h % a4 == 0 && ldh % 4 == 0)))
    EMBED(4);
  else EMBED(1);
#undef EMBED
  return (int)hipGetLastError();
}

// h (optional) has the activation type of y and g
int p2p_sm_gate_norm_add(float* x, const void* y, int ldy, const void* g, int ldg,
                         const float* gb, const float* w, int R, int n, int parts, float eps,
                         void* h, int ldh, int h_f32, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  if (parts <= 0 || n % parts || (h && h_f32 != f32)) return (int)hipErrorInvalidValue;
  // many short parts (prompts): one wavefront per (row, part), so the reduction needs no other
  // wave and more parts are in flight; few rows (decode) keep four wavefronts per part
  const int threads = (n / parts <= 1024 && R * parts >= 1024) ? 64 : 256;
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(gate_norm_add_k<T>, dim3(R * parts), dim3(threads), 0, st, x,
                                         (const T*)y, ldy, (const T*)g, ldg, gb, w, n, parts, eps,
                                         (T*)h, ldh));
  return (int)hipGetLastError();
}

int p2p_sm_embed_pos(const void* embed, const void* ptab, const int* ids, const int* pos,
                     float* out, int R, int W, int f32, hipStream_t st) {
  if (R <= 0) return 0;
#define EMBED(VE)                                                                      \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((embed_pos_k<T, VE>), dim3(R), dim3(256), 0, st, \
                                         (const T*)embed, (const T*)ptab, ids, pos, out, W, ptab != nullptr))
  if (W % 4 == 0 && ((size_t)embed | (size_t)ptab) % (f32 ? 16 : 8) == 0 && (size_t)out % 16 == 0) EMBED(4);
  else EMBED(1);
#undef EMBED
  return (int)hipGetLastError();
}

int p2p_sm_rmsnorm(const void* x, int ldx, int in_f32, const float* w, void* out, int ldo,
                   int out_f32, const int* in_rows, const int* out_rows, int R, int n, int parts,
                   float eps, hipStream_t st) {
  if (R <= 0) return 0;
  if (parts <= 0 || n % parts) return (int)hipErrorInvalidValue;
  const int np = n / parts;
  auto by4 = [](const void* p, int ld, int f32) { return ld % 4 == 0 && (size_t)p % (f32 ? 16 : 8) == 0; };
  const int ve = row_form(np, np % 4 == 0 && by4(x, ldx, in_f32) && by4(out, ldo, out_f32) && by4(w, 0, 1));
  // short parts: no more wavefronts than have a load to do (2048 rows x 8 parts of 128 with 256 / 64 threads:
  // 14.9 / 6.8 us)
  const dim3 g(R * parts), b(ve != 1 ? 256 : np <= 256 ? 64 : np <= 512 ? 128 : 256);
#define RN(TI, TO)                                                                                       \
  ROW_FORMS(ve, hipLaunchKernelGGL((rmsnorm_k<TI, TO, VE, NC>), g, b, 0, st, (const TI*)x, ldx, w,        \
                                   (TO*)out, ldo, in_rows, out_rows, n, parts, eps))
  if (in_f32 && out_f32) RN(float, float);
  else if (in_f32) RN(float, bf16);
  else if (out_f32) RN(bf16, float);
  else RN(bf16, bf16);
#undef RN
  return (int)hipGetLastError();
}

int p2p_sm_norm_scale_add(float* x, const void* y, int ldy, const float* w, const float* ls,
                          int R, int n, float eps, const float* w2, void* h, int ldh, int f32,
                          hipStream_t st) {
  if (R <= 0) return 0;
  const size_t a4 = f32 ? 16 : 8, vecs = (size_t)x | (size_t)w | (size_t)ls | (size_t)w2;
  const int ve = row_form(n, n % 4 == 0 && vecs % 16 == 0 && ((size_t)y | (size_t)h) % a4 == 0 && ldy % 4 == 0 &&
                                 ldh % 4 == 0);
  SM_DISPATCH_T(f32, ROW_FORMS(ve, hipLaunchKernelGGL((norm_scale_add_k<T, VE, NC>), dim3(R), dim3(256), 0, st, x,
                                                      (const T*)y, ldy, w, ls, n, eps, w2, (T*)h, ldh)));
  return (int)hipGetLastError();
}

int p2p_sm_add_norm2(float* x, const void* a, int lda, const void* b, int ldb, const float* rows,
                     const float* vec, int R, int n, float eps, const float* w1, int ws1, void* h1,
                     int ld1, const float* w2, int ws2, void* h2, int ld2, const void* cy, int ldcy,
                     const float* cw, int top, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  if ((w1 && !h1) || (w2 && (!h2 || !w1)) || (b && !a) || (cy && (!cw || top < 1)))
    return (int)hipErrorInvalidValue;
  const size_t a4 = f32 ? 16 : 8;
  const bool by4 = n % 4 == 0 && ((size_t)x | (size_t)rows | (size_t)vec) % 16 == 0 &&
                   (((ws1 ? (size_t)w1 : 0) | (ws2 ? (size_t)w2 : 0)) % 16) == 0 &&
                   ((size_t)a | (size_t)b | (size_t)h1 | (size_t)h2 | (size_t)cy) % a4 == 0 &&
                   (lda | ldb | ld1 | ld2 | ldcy) % 4 == 0;
#define AN2(VE, NC)                                                                                                \
  hipLaunchKernelGGL((add_norm2_k<T, VE, NC>), dim3(R), dim3(256), 0, st, x, (const T*)a, lda, (const T*)b, ldb,   \
                     rows, vec, n, eps, w1, ws1, (T*)h1, ld1, w2, ws2, (T*)h2, ld2, (const T*)cy, ldcy, cw, top)
  // rows that one number per load takes: this pass loads up to six operands, so the smallest form that holds the row
  // (2048 rows of 510 numbers with registers for 1024 / 4096: 6.6 / 10.4 us, of 1502 with 2048 / 4096: 10.0 / 14.2)
  if (!by4 && n <= 1024) SM_DISPATCH_T(f32, AN2(1, 4));
  else if (!by4 && n <= 2048) SM_DISPATCH_T(f32, AN2(1, 8));
  else SM_DISPATCH_T(f32, ROW_FORMS(row_form(n, by4), AN2(VE, NC)));
#undef AN2
  return (int)hipGetLastError();
}

int p2p_sm_add_norm(float* x, const void* a, int lda, const void* b, int ldb, int R, int n,
                    float eps, const float* w2, void* h, int ldh, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  const size_t a4 = f32 ? 16 : 8;
  const int form = row_form(n, n % 4 == 0 && ((size_t)x | (size_t)w2) % 16 == 0 && lda % 4 == 0 && ldb % 4 == 0 &&
                                   ldh % 4 == 0 && ((size_t)a | (size_t)b | (size_t)h) % a4 == 0);
  SM_DISPATCH_T(f32, ROW_FORMS(form, hipLaunchKernelGGL((add_norm_k<T, VE, NC>), dim3(R), dim3(256), 0, st, x,
                                                        (const T*)a, lda, (const T*)b, ldb, n, eps, w2, (T*)h, ldh)));
  return (int)hipGetLastError();
}

}  // extern "C"
