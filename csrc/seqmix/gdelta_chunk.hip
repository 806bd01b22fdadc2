// The generalized delta rule over long portions in chunks of up to 64 tokens on the fp32 matrix instruction
// (v_mfma_f32_16x16x4_f32: products and sums in fp32), head sizes up to 64.  Per head and token
//   S <- diag(w) S - (a * u)(u^T S) + k v^T,   o = S^T r,   u = k / sqrt(|k|^2 + 1e-6),   w = exp(-e^-1/2 sigmoid(.))
// With W(s, t) the product of the decays after token s up to t, the rows p_t = u_t^T S_(t-1) of a chunk obey
//   p_t + sum_{s<t} (u_t W(s,t-1) a_s u_s) p_s = (u_t W(-1,t-1)) S_0 + sum_{s<t} (u_t W(s,t-1) k_s) v_s,
// a unit lower triangular system: P = G S_0 + H.  What leaves the chunk is linear in S_0 as well:
//   S_end = T S_0 + L,   T = W(-1,end) - sum_s W(s,end) a_s u_s G_s,  L = sum_s W(s,end) (k_s v_s^T - a_s u_s H_s)
//   o_t   = Q_t S_0 + O_t,   Q_t = r_t W(-1,t) - sum_{s<=t} (r_t W(s,t) a_s u_s) G_s,  O_t likewise with k_s v_s, H_s
// gdelta_chunk_k forms T, L, Q, O of every (chunk, head); gdelta_chain_k walks the chunks, S <- T S + L;
// gdelta_out_k forms o = Q S_0 + O with the head norm, weight and gate.
//
// W(s, t) is taken apart into e_t / e_s, e the running product of the decays over its value after 32 tokens (a decay
// lies between 0.54 and 1, so e stays within 2^+-28).  The products are formed in 64 bits and rounded once, with the
// vector they multiply: as exponentials of a running sum in fp32 both factors were off by up to 1e-6.  Sums of products
// are taken 16 at a time and added up, which is worth half of a chain of 64 roundings.  Errors against 64 bits (64 to
// 600 tokens, decays near 1, mixed and strongest): outputs 1.6e-7, 1.4e-7, 1.4e-7, the walk 1.6e-7, 1.4e-7, 1.5e-7;
// states 1.7e-7, 1.2e-7, 0.8e-7, the walk 1.4e-7, 0.6e-7, 0.4e-7, a walk of chunks 1.7e-7, 1.2e-7, 0.9e-7.
// The system is solved in blocks of 16 rows, the blocks on the diagonal by their inverses.
// A weight of zero stands for "not before this token" in these products, and 0 * inf is nan: a chunk and head whose
// inputs are not all finite is walked token by token instead, so that tokens before such an input are what they were.
//
// A chunk and head are about 600 matrix instructions per wavefront.  The walk of gdelta_scan_k (once for L and T, once
// for the outputs) took 2 x 205 us for 2048 tokens and 32 heads of 64, and the chain 654 us of 32 dependent products on
// 32 workgroups with scalar sums; the three kernels here take 84, 31 and 21 us.  The first is bound by its workgroups' chains of
// loads, products and barriers (the products alone: 40 us).  It took 168 with six tables in LDS (104 KB: one
// workgroup per CU), 108 with four (two of them take the places of U and R in turn: 77 KB, two workgroups), 104 with a
// table of weights per wavefront instead of 16 rows of all four, 84 with no load behind a branch and one
// division in 64 bits instead of sixteen.
#include "common.h"
using namespace sm;

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GC 64               // tokens of a chunk, and the padded head size
#define GLD 68              // row length in LDS: 16 rows x 16 bytes and 4 rows x 16 numbers both spread over the banks
#define GD_DECAY_SCALE 0.6065306597126334f  // exp(-1/2)

#define MFMA4(a, b, c) __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0)

struct GdeltaArgs {
  const void *r, *k, *v, *g, *a;
  int ld;
  const void* lo;
  int ldlo;
  const float *w0, *ab, *normw;
  float* state;
  float *trn, *loc, *qq, *oo;   // scratch, [chunks, H, 64, 64] each; loc becomes the state before every chunk
  const int *vent, *cent;
  void* out;
  int ldo, H, D;
  float eps;
};

// T, L, Q and O of a chunk and head by its tokens in order, WT of them staged at a time: a thread takes 16 rows of a
// column of T and of L
template <typename T>
__device__ __forceinline__ void walk_chunk(const GdeltaArgs& p, const Entry& en, int c, int h, float* smem) {
  constexpr int WT = 32;   // six rows per token: what the four tables' LDS holds
  float *sr = smem, *sk = sr + WT * GLD, *su = sk + WT * GLD, *sa = su + WT * GLD, *sw = sa + WT * GLD, *sv = sw + WT * GLD;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, D = p.D;
  const int vc = wave * 16 + (lane & 15), i0 = (lane >> 4) * 16;
  const int col = h * D + min(lane, D - 1);
  float S[16], M[16];
#pragma unroll
  for (int q = 0; q < 16; q++) S[q] = 0.0f, M[q] = i0 + q == vc ? 1.0f : 0.0f;
  auto over_rows = [](float x) {   // the sum over a column's four threads
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
  };
  const size_t base = ((size_t)c * p.H + h) * GC * GC;
  for (int b0 = 0; b0 < en.n; b0 += WT) {
    const int nb = min(WT, en.n - b0);
    for (int t = wave; t < nb; t += 4) {
      const size_t row = (size_t)(en.row0 + b0 + t);
      const int at = t * GLD + lane;
      const bool in = lane < D;
      const float k = in ? ldf((const T*)p.k, row * p.ld + col) : 0.0f;
      const float u = k * (1.0f / sqrtf(wave_sum(k * k) + 1e-6f));
      sr[at] = in ? ldf((const T*)p.r, row * p.ld + col) : 0.0f;
      sk[at] = k;
      su[at] = u;
      sa[at] = in ? sigmoidf_(ldf((const T*)p.a, row * p.ld + col) + p.ab[col]) * u : 0.0f;
      sw[at] = in ? expf(-GD_DECAY_SCALE * sigmoidf_(ldf((const T*)p.lo, row * p.ldlo + col) + p.w0[col])) : 1.0f;
      sv[at] = in ? ldf((const T*)p.v, row * p.ld + col) : 0.0f;
    }
    __syncthreads();
    for (int t = 0; t < nb; t++) {
      const int at = t * GLD + i0;
      float ds = 0.0f, dm = 0.0f, os = 0.0f, om = 0.0f;
#pragma unroll
      for (int q = 0; q < 16; q++) {
        ds += su[at + q] * S[q];
        dm += su[at + q] * M[q];
      }
      ds = over_rows(ds);
      dm = over_rows(dm);
      const float v = sv[t * GLD + vc];
#pragma unroll
      for (int q = 0; q < 16; q++) {
        S[q] = sw[at + q] * S[q] - sa[at + q] * ds + sk[at + q] * v;
        M[q] = sw[at + q] * M[q] - sa[at + q] * dm;
        os += S[q] * sr[at + q];
        om += M[q] * sr[at + q];
      }
      os = over_rows(os);
      om = over_rows(om);
      if (i0 == 0) {
        p.oo[base + (b0 + t) * GC + vc] = os;
        p.qq[base + (b0 + t) * GC + vc] = om;
      }
    }
    __syncthreads();   // the tokens have been used
  }
#pragma unroll
  for (int q = 0; q < 16; q++) {
    p.loc[base + (i0 + q) * GC + vc] = S[q];
    p.trn[base + (i0 + q) * GC + vc] = M[q];
  }
}

template <typename T>
__global__ void __launch_bounds__(256, 2) gdelta_chunk_k(GdeltaArgs p) {
  extern __shared__ __align__(16) float smem[];
  float* sU = smem;                  // u e_(t-1), then the weights of v_s in p_t, then those of v_s in o_t
  float* sR = sU + GC * GLD;         // r e_t,     then the weights of p_s in p_t, then those of p_s in o_t
  float* sK = sR + GC * GLD;         // k / e_s
  float* sA = sK + GC * GLD;         // a u / e_s
  __shared__ double sTot[4][GC];
  __shared__ float sMid[GC], sEnd[GC];
  __shared__ __align__(16) float sD[4][16][20];   // inverses of the blocks on the diagonal
  const int c = blockIdx.x, h = blockIdx.y, D = p.D;
  const Entry en = load_entry(p.vent, c);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n16 = lane & 15, quad = lane >> 4;
  float odd = 0.0f;   // becomes nan with an input that is not finite
  // values as operands: token 16 b + quad * 4 + e, this wavefront's 16 columns
  const int vc = wave * 16 + n16;
  f32x4 V[4];
  // a lane's channel of the wavefront's 16 tokens
  {
    const int col = h * D + min(lane, D - 1);
    const bool in = lane < D;
    const float w0 = p.w0[col], ab = p.ab[col];
    // every load first and none behind a branch (which would wait for those before it)
    float kv[16], rv[16], av[16], w[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const size_t row = (size_t)(en.row0 + min(wave * 16 + q, en.n - 1));
      kv[q] = ldf((const T*)p.k, row * p.ld + col);
      rv[q] = ldf((const T*)p.r, row * p.ld + col);
      av[q] = ldf((const T*)p.a, row * p.ld + col);
      w[q] = ldf((const T*)p.lo, row * p.ldlo + col);
    }
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int e = 0; e < 4; e++)
        V[b][e] = ldf((const T*)p.v, (size_t)(en.row0 + min(b * 16 + quad * 4 + e, en.n - 1)) * p.ld + h * D + min(vc, D - 1));
    double all = 1.0;
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const bool have = in && wave * 16 + q < en.n;
      kv[q] = have ? kv[q] : 0.0f;
      rv[q] = have ? rv[q] : 0.0f;
      av[q] = sigmoidf_(av[q] + ab);
      w[q] = have ? expf(-GD_DECAY_SCALE * sigmoidf_(w[q] + w0)) : 1.0f;
      all *= w[q];
    }
    sTot[wave][lane] = all;
    __syncthreads();
    const double t0 = sTot[0][lane], t1 = sTot[1][lane], t2 = sTot[2][lane], t3 = sTot[3][lane];
    double up = wave == 0 ? 1.0 / (t0 * t1) : wave == 1 ? 1.0 / t1 : wave == 2 ? 1.0 : t2;   // before this token
    double down = 1.0 / (up * all);                                                          // after the last one
    if (wave == 0) {
      sMid[lane] = (float)(t0 * t1);
      sEnd[lane] = (float)(t2 * t3);   // to the chunk's end, from the middle
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int at = (wave * 16 + q) * GLD + lane;
      const float u = kv[q] * (1.0f / sqrtf(wave_sum(kv[q] * kv[q]) + 1e-6f));
      sU[at] = (float)(u * up);
      up *= w[q];
      sR[at] = (float)(rv[q] * up);
      av[q] *= u;
    }
#pragma unroll
    for (int q = 15; q >= 0; q--) {   // one division for the sixteen
      const int at = (wave * 16 + q) * GLD + lane;
      const float kd = (float)(kv[q] * down), ad = (float)((double)av[q] * down);
      down *= w[q];
      sK[at] = kd;
      sA[at] = ad;
      odd += 0.0f * kd + 0.0f * ad;
    }
  }
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      V[b][e] = b * 16 + quad * 4 + e < en.n && vc < D ? V[b][e] : 0.0f;
      odd += 0.0f * V[b][e];
    }
  if (__syncthreads_or(odd != 0.0f)) {
    walk_chunk<T>(p, en, c, h, smem);
    return;
  }
  // the four tables of weights, one per wavefront, its blocks of rows t and s <= t (by rows, the last wavefront had four
  // times the first one's products): U.K, U.A, R.K, R.A
  f32x4 tab[10];   // block (b, j) at b (b + 1) / 2 + j
#pragma unroll
  for (int i = 0; i < 10; i++) tab[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  {
    const float *sx = wave & 2 ? sR : sU, *sy = wave & 1 ? sA : sK;
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      f32x4 x[4], y[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        x[j] = *(const f32x4*)(sx + (j * 16 + n16) * GLD + kk * 16 + quad * 4);
        y[j] = *(const f32x4*)(sy + (j * 16 + n16) * GLD + kk * 16 + quad * 4);
      }
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int j = 0; j <= b; j++) {
          f32x4 p0 = {0.f, 0.f, 0.f, 0.f};   // sums of 16
#pragma unroll
          for (int e = 0; e < 4; e++) p0 = MFMA4(x[b][e], y[j][e], p0);
          tab[b * (b + 1) / 2 + j] += p0;
        }
    }
  }
  // G starts as U, Q as R: this wavefront's 16 columns
  f32x4 G[4], Q[4];
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int at = (b * 16 + quad * 4 + e) * GLD + vc;
      G[b][e] = sU[at];
      Q[b][e] = sR[at];
    }
  // two tables in LDS at a time, the other two in registers until these have been used
  auto put = [&](int half) {
    if (wave >> 1 != half) return;
    float* dst = wave & 1 ? sR : sU;
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int j = 0; j <= b; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int t = b * 16 + quad * 4 + e, s = j * 16 + n16;
          dst[t * GLD + s] = s < t + half ? tab[b * (b + 1) / 2 + j][e] : 0.0f;
        }
  };
  __syncthreads();   // U and R have been read
  put(0);   // U.K and U.A
  __syncthreads();
  // the inverse of this wavefront's block on the diagonal, a column per lane
  {
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      float v = i == n16 ? 1.0f : 0.0f;
#pragma unroll
      for (int q = 0; q < i; q++) v = fmaf(-sR[(wave * 16 + i) * GLD + wave * 16 + q], x[q], v);
      x[i] = v;
    }
    if (quad == 0) {
#pragma unroll
      for (int i = 0; i < 16; i++) sD[wave][i][n16] = x[i];
    }
  }
  // right side of H
  f32x4 Hm[4];
#pragma unroll
  for (int b = 0; b < 4; b++) {
    Hm[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j <= b; j++) {
      const f32x4 f = *(const f32x4*)(sU + (b * 16 + n16) * GLD + j * 16 + quad * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) Hm[b] = MFMA4(f[e], V[j][e], Hm[b]);
    }
  }
  __syncthreads();   // the inverses
#pragma unroll
  for (int b = 0; b < 4; b++) {
#pragma unroll
    for (int j = 0; j < b; j++) {
      const f32x4 f = *(const f32x4*)(sR + (b * 16 + n16) * GLD + j * 16 + quad * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        G[b] = MFMA4(-f[e], G[j][e], G[b]);
        Hm[b] = MFMA4(-f[e], Hm[j][e], Hm[b]);
      }
    }
    const f32x4 f = *(const f32x4*)&sD[b][n16][quad * 4];
    f32x4 g = {0.f, 0.f, 0.f, 0.f}, x = g;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      g = MFMA4(f[e], G[b][e], g);
      x = MFMA4(f[e], Hm[b][e], x);
    }
    G[b] = g;
    Hm[b] = x;
  }
  const size_t base = ((size_t)c * p.H + h) * GC * GC;
  const float emid = sMid[vc];
  __syncthreads();   // the system has been solved
  put(1);   // R.K and R.A
  __syncthreads();
  // outputs: Q and O
#pragma unroll
  for (int b = 0; b < 4; b++) {
    f32x4 O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j <= b; j++) {
      const f32x4 fu = *(const f32x4*)(sR + (b * 16 + n16) * GLD + j * 16 + quad * 4);
      const f32x4 fk = *(const f32x4*)(sU + (b * 16 + n16) * GLD + j * 16 + quad * 4);
      f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0, p2 = p0;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        p0 = MFMA4(-fu[e], G[j][e], p0);
        p1 = MFMA4(-fu[e], Hm[j][e], p1);
        p2 = MFMA4(fk[e], V[j][e], p2);
      }
      Q[b] += p0;
      O += p1 + p2;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const size_t at = base + (b * 16 + quad * 4 + e) * GC + vc;
      p.qq[at] = Q[b][e] * emid;
      p.oo[at] = O[e];
    }
  }
  // the end of the chunk: T and L
#pragma unroll
  for (int it = 0; it < 4; it++) {
    f32x4 tr = {0.f, 0.f, 0.f, 0.f}, lc = tr;
#pragma unroll
    for (int b = 0; b < 4; b++) {
      f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0, p2 = p0;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int at = (b * 16 + quad * 4 + e) * GLD + it * 16 + n16;
        const float ad = sA[at], kd = sK[at];
        p0 = MFMA4(ad, G[b][e], p0);
        p1 = MFMA4(kd, V[b][e], p1);
        p2 = MFMA4(-ad, Hm[b][e], p2);
      }
      tr += p0;
      lc += p1 + p2;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int i = it * 16 + quad * 4 + e;
      const float end = sEnd[i];
      p.trn[base + i * GC + vc] = (i == vc ? end * emid : 0.0f) - end * tr[e] * emid;
      p.loc[base + i * GC + vc] = end * lc[e];
    }
  }
}

// S <- T S + L over each portion's chunks, 16 columns of a head per workgroup, a wavefront per 16 rows; the state before
// a chunk replaces its L.  What a chunk needs from memory does not depend on the state: it is read three chunks
// ahead (one: 36 us for 32 chunks and heads, every chunk a wait for memory; three: 31).
__global__ void __launch_bounds__(256) gdelta_chain_k(GdeltaArgs p) {
  __shared__ float sS[2][GC][17];
  const int c0 = p.cent[4 * blockIdx.z], nc = p.cent[4 * blockIdx.z + 1], start = p.cent[4 * blockIdx.z + 2],
            slot = p.cent[4 * blockIdx.z + 3];
  const int h = blockIdx.y, D = p.D;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n16 = lane & 15, quad = lane >> 4;
  const int col = blockIdx.x * 16 + n16, row = wave * 16 + quad * 4;   // C layout: rows row .. row + 3
  float* sg = p.state + ((size_t)slot * p.H + h) * D * D;
  f32x4 cur;
#pragma unroll
  for (int e = 0; e < 4; e++)
    cur[e] = (start > 0 && row + e < D && col < D) ? sg[(size_t)(row + e) * D + col] : 0.0f;
  const size_t step = (size_t)p.H * GC * GC;
  const float* tp = p.trn + (size_t)c0 * step + (size_t)h * GC * GC + (wave * 16 + n16) * GC + quad * 4;
  float* lp = p.loc + (size_t)c0 * step + (size_t)h * GC * GC + row * GC + col;
  f32x4 T[3][4], L[3];
  auto load = [&](int c, f32x4 (&t)[4], f32x4& l) {
    c = min(c, nc - 1);   // (beyond the end: not used)
#pragma unroll
    for (int b = 0; b < 4; b++) t[b] = *(const f32x4*)(tp + c * step + b * 16);
#pragma unroll
    for (int e = 0; e < 4; e++) l[e] = lp[c * step + e * GC];
  };
#pragma unroll
  for (int u = 0; u < 3; u++) load(u, T[u], L[u]);
  for (int k = 0; k < nc; k += 3) {
#pragma unroll
    for (int u = 0; u < 3; u++) {
      const int c = k + u;
      if (c >= nc) break;
      float(*S)[17] = sS[c & 1];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        S[row + e][n16] = cur[e];
        lp[c * step + e * GC] = cur[e];
      }
      __syncthreads();
      f32x4 a[4];
      a[0] = L[u];
      a[1] = a[2] = a[3] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) a[b] = MFMA4(T[u][b][e], S[b * 16 + quad * 4 + e][n16], a[b]);
      cur = (a[0] + a[1]) + (a[2] + a[3]);
      load(c + 3, T[u], L[u]);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; e++)
    if (row + e < D && col < D) sg[(size_t)(row + e) * D + col] = cur[e];
}

// o = Q S + O, head norm, weight and gate; a wavefront per 16 tokens, column n16 * 4 + j in tile j
template <typename T>
__global__ void __launch_bounds__(256) gdelta_out_k(GdeltaArgs p) {
  const int c = blockIdx.x, h = blockIdx.y, D = p.D;
  const Entry en = load_entry(p.vent, c);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n16 = lane & 15, quad = lane >> 4;
  if (wave * 16 >= en.n) return;
  const size_t base = ((size_t)c * p.H + h) * GC * GC;
  const float* qp = p.qq + base + (wave * 16 + n16) * GC + quad * 4;
  const float* sp = p.loc + base + quad * 4 * GC + n16 * 4;
  const float* op = p.oo + base + (wave * 16 + quad * 4) * GC + n16 * 4;
  f32x4 q[4], s[4][4], o[4], acc[4], sum[4];
#pragma unroll
  for (int b = 0; b < 4; b++) q[b] = *(const f32x4*)(qp + b * 16);
#pragma unroll
  for (int b = 0; b < 4; b++)
#pragma unroll
    for (int e = 0; e < 4; e++) s[b][e] = *(const f32x4*)(sp + (b * 16 + e) * GC);
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] = *(const f32x4*)(op + e * GC);
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) acc[j][e] = o[e][j];
#pragma unroll
  for (int b = 0; b < 4; b++) {
#pragma unroll
    for (int j = 0; j < 4; j++) sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int j = 0; j < 4; j++) sum[j] = MFMA4(q[b][e], s[b][e][j], sum[j]);
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] += sum[j];
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int t = wave * 16 + quad * 4 + e;
    float ss = 0.0f;   // a column beyond D is zero, or nan after a walk
#pragma unroll
    for (int j = 0; j < 4; j++) ss += n16 * 4 + j < D ? acc[j][e] * acc[j][e] : 0.0f;
#pragma unroll
    for (int m = 8; m > 0; m >>= 1) ss += __shfl_xor(ss, m, 64);
    const float rs = 1.0f / sqrtf(ss / (float)D + p.eps);
    if (t >= en.n) continue;
    const size_t row = (size_t)(en.row0 + t);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int i = n16 * 4 + j, at = h * D + i;
      if (i < D)
        stf((T*)p.out, row * p.ldo + at, acc[j][e] * rs * p.normw[at] * sigmoidf_(ldf((const T*)p.g, row * p.ld + at)));
    }
  }
}

extern "C" {

// 1 when the kernels serve this head size
int p2p_sm_gdelta_chunk_ok(int D) { return D >= 1 && D <= GC; }

// vent [NV]: the portions' chunks of at most 64 tokens as entries (row0, n, 1, chunk index); tmp: 4 fp32 buffers of
// [NV, H, 64, 64]; cent: per portion (first chunk, chunks, first position, slot)
int p2p_sm_gdelta_chunk(const void* r, const void* k, const void* v, const void* g, const void* a, int ld,
                        const void* lo, int ldlo, const float* w0, const float* ab, const float* normw, float* state,
                        float* tmp, const int* vent, int NV, const int* cent, int E, void* out, int ldo, int H, int D,
                        float eps, int f32, hipStream_t st) {
  if (E <= 0 || NV <= 0) return 0;
  if (!p2p_sm_gdelta_chunk_ok(D)) return (int)hipErrorInvalidValue;
  const size_t sz = (size_t)NV * H * GC * GC;
  const GdeltaArgs p = {r, k, v, g, a, ld, lo, ldlo, w0, ab, normw, state, tmp, tmp + sz, tmp + 2 * sz, tmp + 3 * sz,
                        vent, cent, out, ldo, H, D, eps};
  constexpr int shm = 4 * GC * GLD * 4;
  static const hipError_t attr = [] {
    const hipError_t e = hipFuncSetAttribute((const void*)gdelta_chunk_k<float>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, shm);
    return e != hipSuccess ? e
                           : hipFuncSetAttribute((const void*)gdelta_chunk_k<bf16>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, shm);
  }();
  if (attr != hipSuccess) return (int)attr;
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(gdelta_chunk_k<T>, dim3(NV, H), dim3(256), shm, st, p));
  hipLaunchKernelGGL(gdelta_chain_k, dim3((D + 15) / 16, H, E), dim3(256), 0, st, p);
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(gdelta_out_k<T>, dim3(NV, H), dim3(256), 0, st, p));
  return (int)hipGetLastError();
}

}  // extern "C"
