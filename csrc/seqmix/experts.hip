// Mixture of experts: the router with a group-limited choice, the expert matrix products over
// the routed rows, and the weighted sum of the chosen experts' outputs.
//
// group_route_k: z = h . Wr^T in fp32, s = sigmoid(z) or softmax(z) over all experts; the
// choice is made on s plus an optional per-expert correction.  The E experts are cut into
// `groups` contiguous blocks of equal size; a block is ranked by the sum of its two best choice
// scores or by its best one; experts outside the `keep` best blocks are struck out, and the
// `top` largest remaining choice scores win (ties: the lower index).  The weights are the
// winners' s (without the correction), as they are or divided by their sum + 1e-20, times a constant.
// A token r routed to its k-th expert is slot
// r * top + k; every expert gets the list of its slots (cnt / rows).
//
// expert_gemm: for expert e and each of its slots s: out[s] = x[s / x_div] . W_e^T.  Rows are
// gathered through the slot lists, so only experts with rows read their weights.  Rows of a multiple of 16
// bytes run on the matrix cores (a 16 x 64 tile with K split over the wavefronts for decode-sized steps,
// LDS-staged tiles for prompts); odd shapes run a tiled FMA kernel.  A
// slot's result does not depend on which other slots share its tile.
#include "attn_tile.h"
using namespace sm;

// best (value, index) over the wavefront; ties go to the lower index
__device__ __forceinline__ void wave_argmax(float& v, int& i) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float ov = __shfl_xor(v, o, 64);
    int oi = __shfl_xor(i, o, 64);
    if (ov > v || (ov == v && oi < i)) {
      v = ov;
      i = oi;
    }
  }
}

// orders one wavefront's LDS writes before its later reads by other lanes
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

#define LOWEST_SCORE -3.402823466e+38f

// The choice of one row by one wavefront: ss holds its E logits (sigmoids for score 0) and becomes its scores.
// place(k, e): the row's k-th expert is e (called by lane 0).
template <typename P>
__device__ __forceinline__ void choose_experts(int r, int lane, float* ss, float* sc, float* sgs, float* stop, int E,
                                               int top, int groups, int keep, int score,
                                               const float* __restrict__ corr, int gscore, int* __restrict__ ids,
                                               float* __restrict__ wts, int renorm, float wscale, P place) {
  if (score == 1) {   // softmax over all experts
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, ss[e]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    float sum = 0.0f;
    for (int e = lane; e < E; e += 64) {
      float v = expf(ss[e] - mx);
      ss[e] = v;
      sum += v;
    }
    sum = wave_sum(sum);
    for (int e = lane; e < E; e += 64) ss[e] = ss[e] / sum;
  }
  // choice scores are above -inf, which marks what cannot be chosen (any more): a score that is not a number or
  // -inf counts as the lowest, so that every pick is an expert
  for (int e = lane; e < E; e += 64) sc[e] = fmaxf(corr ? ss[e] + corr[e] : ss[e], LOWEST_SCORE);
  wave_sync();
  const int per = E / groups;
  if (keep < groups) {
    for (int g = lane; g < groups; g += 64) {
      float b1 = -INFINITY, b2 = -INFINITY;   // top-2 of the block
      for (int i = 0; i < per; i++) {
        float v = sc[g * per + i];
        if (v > b1) { b2 = b1; b1 = v; }
        else if (v > b2) b2 = v;
      }
      sgs[g] = fmaxf(b1 + ((per > 1 && gscore == 0) ? b2 : 0.0f), LOWEST_SCORE);
    }
    wave_sync();
    // keep the best groups: pick `keep` times, then strike out the experts of the others
    for (int k = 0; k < keep; k++) {
      float bv = -INFINITY;
      int bi = 1 << 30;
      for (int g = lane; g < groups; g += 64) {
        float v = sgs[g];
        if (v > bv) { bv = v; bi = g; }     // ascending g: the first of equals stays
      }
      wave_argmax(bv, bi);
      if (lane == 0) sgs[bi] = -INFINITY;   // marks "kept"
      wave_sync();
    }
    for (int e = lane; e < E; e += 64)
      if (sgs[e / per] != -INFINITY) sc[e] = -INFINITY;
    wave_sync();
  }
  for (int k = 0; k < top; k++) {
    float bv = -INFINITY;
    int bi = 1 << 30;
    for (int e = lane; e < E; e += 64) {
      float v = sc[e];
      if (v > bv) { bv = v; bi = e; }
    }
    wave_argmax(bv, bi);
    if (lane == 0) {
      sc[bi] = -INFINITY;
      int slot = r * top + k;
      ids[slot] = bi;
      if (score == 2 || renorm) stop[k] = ss[bi];
      else wts[slot] = ss[bi] * wscale;
      place(k, bi);
    }
    wave_sync();
  }
  if (score == 2) {   // the weights become the softmax over the chosen logits
    float mx = -INFINITY;
    for (int k = lane; k < top; k += 64) mx = fmaxf(mx, stop[k]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    float sum = 0.0f;
    for (int k = lane; k < top; k += 64) sum += expf(stop[k] - mx);
    sum = wave_sum(sum);
    for (int k = lane; k < top; k += 64) wts[r * top + k] = expf(stop[k] - mx) / sum * wscale;
  } else if (renorm) {
    float sum = 0.0f;
    for (int k = lane; k < top; k += 64) sum += stop[k];
    sum = wave_sum(sum) + 1e-20f;
    for (int k = lane; k < top; k += 64) wts[r * top + k] = stop[k] / sum * wscale;
  }
}

// score: 0 sigmoid, 1 softmax over all experts, 2 the logits themselves for the choice and the
// softmax over the chosen logits as weights.  bias (optional, [E]): added to the logits.
// corr (optional, [E]): added to the scores for the choice only.  gscore: a group is ranked by 0 the sum of its two best choice scores, 1 its
// best choice score.
template <typename T>
__global__ void __launch_bounds__(256)
group_route_k(const T* __restrict__ h, int ldh, const float* __restrict__ wr, int W, int E, int top,
              int groups, int keep, int score, const float* __restrict__ corr, int gscore,
              int* __restrict__ ids, float* __restrict__ wts, int* __restrict__ cnt,
              int* __restrict__ rows, int ldr, const float* __restrict__ bias, int renorm,
              float wscale) {
  extern __shared__ float smem[];
  float* sh = smem;          // [W] the row in fp32
  float* ss = sh + W;        // [E] scores (the weights of the chosen)
  float* sc = ss + E;        // [E] choice scores; -inf marks "cannot be chosen (any more)"
  float* sgs = sc + E;       // [groups] group scores
  float* stop = sgs + groups;   // [top] the chosen logits (score 2) or scores (renorm)
  const int r = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  for (int i = threadIdx.x; i < W; i += blockDim.x) sh[i] = ldf(h, (size_t)r * ldh + i);
  __syncthreads();
  // four experts at a time per wavefront: their weight loads are independent and go out together
  for (int e0 = wave * 4; e0 < E; e0 += nw * 4) {
    const float* w0 = wr + (size_t)e0 * W;
    const float* w1 = wr + (size_t)min(e0 + 1, E - 1) * W;
    const float* w2 = wr + (size_t)min(e0 + 2, E - 1) * W;
    const float* w3 = wr + (size_t)min(e0 + 3, E - 1) * W;
    float d0 = 0.0f, d1 = 0.0f, d2 = 0.0f, d3 = 0.0f;
#pragma unroll 4
    for (int i = lane; i < W; i += 64) {
      float x = sh[i];
      d0 += x * w0[i];
      d1 += x * w1[i];
      d2 += x * w2[i];
      d3 += x * w3[i];
    }
    d0 = wave_sum(d0);
    d1 = wave_sum(d1);
    d2 = wave_sum(d2);
    d3 = wave_sum(d3);
    if (lane == 0) {
      if (bias) {
        d0 += bias[e0];
        d1 += bias[min(e0 + 1, E - 1)];
        d2 += bias[min(e0 + 2, E - 1)];
        d3 += bias[min(e0 + 3, E - 1)];
      }
      ss[e0] = score ? d0 : sigmoidf_(d0);
      if (e0 + 1 < E) ss[e0 + 1] = score ? d1 : sigmoidf_(d1);
      if (e0 + 2 < E) ss[e0 + 2] = score ? d2 : sigmoidf_(d2);
      if (e0 + 3 < E) ss[e0 + 3] = score ? d3 : sigmoidf_(d3);
    }
  }
  __syncthreads();
  if (wave != 0) return;
  choose_experts(r, lane, ss, sc, sgs, stop, E, top, groups, keep, score, corr, gscore, ids, wts, renorm, wscale,
                 [&](int k, int e) { rows[(size_t)e * ldr + atomicAdd(&cnt[e], 1)] = r * top + k; });
}

// The same, a workgroup for 16 rows, a wavefront each for the choice, and the experts' slot counts go up by one
// atomic per workgroup and expert instead of one per slot (4096 of them on eight addresses took most of the
// 57 us that 2048 rows of 2048 numbers needed).
// NB > 0, up to 16 NB experts: the logits of all rows on the fp32 matrix instruction, W cut among the wavefronts, 16 bytes of
// a row per load and four of them in flight; the wavefronts' sums meet in LDS.  With a wavefront per row walking W for four
// experts at a time (NB = 0: many experts, or rows that 16-byte loads do not fit) the chain of one row's loads and sums was
// what was left: 2048 rows of 2048 numbers, 8 experts 18.3 -> 10.9 us.
template <typename T, int NB>
__global__ void __launch_bounds__(1024)
group_route_rows_k(const T* __restrict__ h, int ldh, const float* __restrict__ wr, int R, int W, int E, int top,
                   int groups, int keep, int score, const float* __restrict__ corr, int gscore, int* __restrict__ ids,
                   float* __restrict__ wts, int* __restrict__ cnt, int* __restrict__ rows, int ldr,
                   const float* __restrict__ bias, int renorm, float wscale) {
  extern __shared__ float smem[];
  float* ss = smem;                      // [16][E]
  float* sc = ss + 16 * E;               // [16][E]
  float* sgs = sc + 16 * E;              // [16][groups]
  float* stop = sgs + 16 * groups;       // [16][top]
  int* scnt = (int*)(stop + 16 * top);   // [E] slots of this workgroup, then the place of its first
  int* spick = scnt + E;                 // [16][top] expert
  int* sat = spick + 16 * top;           // [16][top] place among the workgroup's
  __shared__ f32x4 part[NB > 0 ? 16 : 1][NB > 0 ? NB : 1][64];
  const int lane = threadIdx.x & 63, m = threadIdx.x >> 6, r = blockIdx.x * 16 + m;
  for (int e = threadIdx.x; e < E; e += 1024) scnt[e] = 0;
  if constexpr (NB > 0) {
    constexpr int EP = 16 / sizeof(T), CH = 4 * EP, U = 4;   // numbers per load, per chunk of a wavefront; chunks at once
    const int wave = uniform(m), n16 = lane & 15, quad = lane >> 4;
    const T* x = h + (size_t)min((int)blockIdx.x * 16 + n16, R - 1) * ldh;
    f32x4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * CH; k0 < W; k0 += U * 16 * CH) {
      uint4 xv[U];
      f32x4 wv[U][NB][EP / 4];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int k = k0 + u * 16 * CH + quad * EP, kk = k < W ? k : 0;   // W is a multiple of EP; past it: struck out below
        xv[u] = *(const uint4*)(x + kk);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int q = 0; q < EP / 4; q++)
            wv[u][b][q] = *(const f32x4*)(wr + (size_t)min(b * 16 + n16, E - 1) * W + kk + q * 4);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const bool in = k0 + u * 16 * CH + quad * EP < W;
        if (k0 + u * 16 * CH >= W) break;
#pragma unroll
        for (int i = 0; i < EP; i++) {
          const float xi = in ? ldf((const T*)&xv[u], i) : 0.0f;
#pragma unroll
          for (int b = 0; b < NB; b++)
            acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(xi, in ? wv[u][b][i / 4][i % 4] : 0.0f, acc[b], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int b = 0; b < NB; b++) part[wave][b][lane] = acc[b];
    __syncthreads();
    // row quad * 4 + i, expert b * 16 + n16 of lane quad * 16 + n16
    for (int at = threadIdx.x; at < 16 * 16 * NB; at += 1024) {
      const int row = at / (16 * NB), e = at % (16 * NB);
      if (e >= E) continue;
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < 16; w++) v += part[w][e / 16][row / 4 * 16 + e % 16][row % 4];
      if (bias) v += bias[e];
      ss[row * E + e] = score ? v : sigmoidf_(v);
    }
  } else {
    const T* x = h + (size_t)min(r, R - 1) * ldh;
    for (int e0 = 0; e0 < E; e0 += 4) {
      const float* w[4];
      float d[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        w[u] = wr + (size_t)min(e0 + u, E - 1) * W;
        d[u] = 0.0f;
      }
#pragma unroll 4
      for (int i = lane; i < W; i += 64) {
        const float xv = ldf(x, i);
#pragma unroll
        for (int u = 0; u < 4; u++) d[u] += xv * w[u][i];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float v = wave_sum(d[u]);
        if (lane == 0 && e0 + u < E) {
          if (bias) v += bias[e0 + u];
          ss[m * E + e0 + u] = score ? v : sigmoidf_(v);
        }
      }
    }
  }
  __syncthreads();   // scnt is clear
  if (r < R)
    choose_experts(r, lane, ss + m * E, sc + m * E, sgs + m * groups, stop + m * top, E, top, groups, keep, score, corr,
                   gscore, ids, wts, renorm, wscale, [&](int k, int e) {
                     spick[m * top + k] = e;
                     sat[m * top + k] = atomicAdd(&scnt[e], 1);
                   });
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 1024) {
    const int n = scnt[e];
    if (n) scnt[e] = atomicAdd(&cnt[e], n);
  }
  __syncthreads();
  const int slots = min(16, R - (int)blockIdx.x * 16) * top;
  for (int i = threadIdx.x; i < slots; i += 1024) {
    const int e = spick[i];
    rows[(size_t)e * ldr + scnt[e] + sat[i]] = blockIdx.x * 16 * top + i;
  }
}

// The grid is sized for the most row tiles the experts can have together (total slots / BM + E,
// since every expert wastes at most one partial tile), one-dimensional, and workgroups go to
// the 8 XCDs round-robin: block L runs on XCD L % 8.  A block counts the row tiles that exist,
// deals them to the XCDs in contiguous runs of equal length (XCD j takes row tiles
// j*pr .. j*pr+pr-1 and all column tiles, so its L2 holds the gathered rows of few experts and
// streams only those experts' weights), and finds its expert and first slot by walking the
// counts.  Blocks beyond the tiles that exist leave at once.
__device__ __forceinline__ bool find_tile(const int* __restrict__ cnt, int E, int BM,
                                          int row_tiles_pad, int& e, int& m0, int& nt) {
  // every wavefront does this for itself, 64 experts at a time: one vector load of the counts,
  // sums and prefix sums by lane shuffles (a scalar walk over the counts costs a dependent
  // load per expert, which a decode-sized launch cannot hide)
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int base = 0; base < E; base += 64) {
    int i = base + lane;
    int n = i < E ? (cnt[i] + BM - 1) / BM : 0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    total += n;
  }
  const int j = blockIdx.x & 7, s = blockIdx.x >> 3, pm = row_tiles_pad >> 3;
  const int pr = (total + 7) >> 3, li = s % pm;
  nt = s / pm;
  const int t = j * pr + li;
  if (li >= pr || t >= total) return false;
  int acc = 0, fe = -1, fm = 0;
  for (int base = 0; base < E && fe < 0; base += 64) {
    int i = base + lane;
    int n = i < E ? (cnt[i] + BM - 1) / BM : 0;
    int incl = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    int excl = acc + incl - n;
    bool hit = n > 0 && t >= excl && t < excl + n;
    unsigned long long mask = __ballot(hit);
    if (mask) {
      int src = __ffsll((long long)mask) - 1;
      fe = base + src;
      fm = (t - __shfl(excl, src, 64)) * BM;
    }
    acc += __shfl(incl, 63, 64);
  }
  // the same for every lane: keep them in scalar registers
  e = __builtin_amdgcn_readfirstlane(fe);
  m0 = __builtin_amdgcn_readfirstlane(fm);
  return e >= 0;
}

// Epilogue with the experts' activation (epi = 1): the weight rows of the first product are
// stored as 16 gate rows, their 16 up rows, the next 16 gate rows, ..., so a thread that holds
// output column c of a 16-column tile holds the matching up value in the next tile, and
//   y = min(g, limit) * sigmoid(alpha * min(g, limit)) * (clamp(u, -limit, limit) + 1)
// is written to column (tile / 2) * 16 + c of an output half as wide.
__device__ __forceinline__ float expert_act(float g, float u, float limit, float alpha) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoidf_(alpha * g) * (u + 1.0f);
}

// epi = 3: the same layout with y = g * sigmoid(g) * u
__device__ __forceinline__ float glu_epi(float g, float u, int epi, float limit, float alpha) {
  return epi == 3 ? g * sigmoidf_(g) * u : expert_act(g, u, limit, alpha);
}

// epi = 2: an ungated unit, every product passes relu(.)^2; epi = 0: the products themselves
__device__ __forceinline__ float plain_epi(float v, int epi) {
  if (epi == 2) {
    v = fmaxf(v, 0.0f);
    v *= v;
  }
  return v;
}

// one step of an accumulator: a 16-byte fragment of 16 slots' rows times one of 16 weight rows
template <typename T>
__device__ __forceinline__ f32x4 mfma_piece(uint4 a, uint4 b, f32x4 c) {
  if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int i = 0; i < 4; i++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], c, 0, 0, 0);
    return c;
  }
}

// Few slots per expert (decode-sized steps), on the matrix cores: a block takes 16 slots x
// 64 output columns of one expert and its four wavefronts split K among themselves, so the
// chain of dependent loads is a quarter as long; each wavefront walks its share in steps of 32
// with one A fragment (the gathered rows) and four B fragments (16 weight rows each), DEPTH steps'
// fragments in flight while the current products run; the four partial tiles are added through LDS.  fp32 takes half
// the K per step (a fragment is 16 bytes of a row) and four products.
// Four steps where a wavefront's share is longer than 8, two (76 instead of 116 registers) where it is shorter: rows
// of 512 numbers, 1024 columns, 128 experts of 40 slots, four / two steps 83 / 68 us, rows of 2048 with 64 experts of 16
// slots and 2048 columns 160 / 163.
template <typename T, int DEPTH>
__global__ void __launch_bounds__(256)
expert_gemm_mfma_k(const T* __restrict__ x, int ldx, int x_div, const T* __restrict__ w,
                   const int* __restrict__ cnt, const int* __restrict__ rows, int ldr,
                   T* __restrict__ out, int ldo, int N, int K, int E, int TMP, int epi, float limit, float alpha) {
  constexpr int EP = 16 / sizeof(T), KS = 4 * EP;   // numbers per fragment, per step
  __shared__ f32x4 red[3][4][64];
  int e, m0, nt;
  if (!find_tile(cnt, E, 16, TMP, e, m0, nt)) return;
  const int c = cnt[e], n0 = nt * 64;
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), n16 = lane & 15, quad = lane >> 4;
  const int mi = m0 + n16;
  const int slot = mi < c ? rows[(size_t)e * ldr + mi] : -1;
  const int kq = ((K + 4 * KS - 1) / (4 * KS)) * KS;   // K per wavefront, a multiple of the step
  const int kb = wave * kq, ke = min(K, kb + kq);
  // rows that do not exist (a slot or column beyond the last) are others, their products are dropped; past
  // the wavefront's share of K both operands are zero
  const T* xa = x + (size_t)(max(slot, 0) / x_div) * ldx;
  const T* wb[4];
#pragma unroll
  for (int t = 0; t < 4; t++) wb[t] = w + ((size_t)e * N + min(n0 + t * 16 + n16, N - 1)) * K;
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const uint4 zero = make_uint4(0, 0, 0, 0);
  uint4 av[DEPTH], bv[DEPTH][4];
  auto load = [&](int k, uint4& a, uint4 (&b)[4]) {
    const bool in = k + quad * EP < ke;            // K is a multiple of EP
    const int at = in ? k + quad * EP : 0;         // else the row's start, which is there whatever K is
    a = *(const uint4*)(xa + at);
#pragma unroll
    for (int t = 0; t < 4; t++) b[t] = *(const uint4*)(wb[t] + at);
    if (!in) {
      a = zero;
#pragma unroll
      for (int t = 0; t < 4; t++) b[t] = zero;
    }
  };
#pragma unroll
  for (int d = 0; d < DEPTH; d++) load(kb + d * KS, av[d], bv[d]);
  for (int k0 = kb; k0 < ke; k0 += DEPTH * KS) {
#pragma unroll
    for (int d = 0; d < DEPTH; d++) {
      if (k0 + d * KS < ke) {   // what a place held before must not meet zeros: it need not be finite
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = mfma_piece<T>(av[d], bv[d][t], acc[t]);
      }
      if (k0 + (DEPTH + d) * KS < ke) load(k0 + (DEPTH + d) * KS, av[d], bv[d]);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < 4; t++) red[wave - 1][t][lane] = acc[t];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int t = 0; t < 4; t++)
#pragma unroll
    for (int u = 0; u < 3; u++) acc[t] += red[u][t][lane];
  // accumulator layout: row quad*4 + i of the 16 slots, column n16 of each tile
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int so = __shfl(slot, quad * 4 + i, 64);
    if (so < 0) continue;
    if (epi == 1 || epi == 3) {
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        int n = n0 + t * 16;
        if (n + 16 + n16 < N)
          stf(out, (size_t)so * ldo + n / 2 + n16, glu_epi(acc[t][i], acc[t + 1][i], epi, limit, alpha));
      }
      continue;
    }
#pragma unroll
    for (int t = 0; t < 4; t++) {
      int n = n0 + t * 16 + n16;
      if (n < N) stf(out, (size_t)so * ldo + n, plain_epi(acc[t][i], epi));
    }
  }
}

// Many slots per expert (prompts): a block of 2 x 2 wavefronts takes BM slots x BN columns and walks K in
// steps of 128 bytes per row (64 bf16, 32 fp32).  The gathered rows and the weight rows of a step are copied
// straight into LDS (attn_tile.h) while the step before is multiplied; their 16-byte pieces are permuted
// so that a fragment's 16 rows spread over all banks.  A wavefront owns BM/2 x BN/2; 16-slot tiles
// beyond the expert's count are skipped.  bf16: one v_mfma_f32_16x16x32_bf16 per pair of 16-byte fragments;
// fp32: four v_mfma_f32_16x16x4_f32, component by component.
//
// Bound by LDS reads and the copies' latency (two or three blocks per CU) and by the last round of the CUs.  8 experts,
// 4096 slots, width 2048, gate and up of 1024: 49 us (700 TFLOP/s) and 28 us for the two products (160 rows; 50 and 29 with one
// number per store) against 229 and
// 117 with register staging, one step at a time; 1212 slots at width 1024: 10.7 and 8.7 us (64 x 64 tiles) against 53
// and 29; fp32, 1012 slots, width 1024 and 512: 37 and 21 us against 185 and 94 on vector instructions.
template <typename T, int BM, int BN>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 8)))
expert_gemm_tile_k(const T* __restrict__ x, int ldx, int x_div, const T* __restrict__ w,
                   const int* __restrict__ cnt, const int* __restrict__ rows, int ldr, T* __restrict__ out, int ldo,
                   int N, int K, int E, int TMP, int epi, float limit, float alpha, int wide) {
  constexpr int EP = 16 / sizeof(T), KS = 8 * EP;          // numbers per piece, per step
  constexpr int FM = BM / 32, FN = BN / 32;                // 16 x 16 tiles of a wavefront
  constexpr int STAGE = (BM + BN) * 128;
  extern __shared__ __align__(16) unsigned char tile[];    // [2][BM rows | BN rows] of 128 bytes
  __shared__ int sslot[BM];
  int e, m0, nt;
  if (!find_tile(cnt, E, BM, TMP, e, m0, nt)) return;
  const int c = cnt[e], n0 = nt * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), n16 = lane & 15, quad = lane >> 4;
  if (tid < BM) sslot[tid] = m0 + tid < c ? rows[(size_t)e * ldr + m0 + tid] : -1;
  __syncthreads();
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const int nmt = max(0, min(FM, (c - (m0 + wm) + 15) / 16));
  // thread t copies pieces t, t + 256, ..; rows that do not exist are the tile's first, their products are dropped
  const int sw = ((tid >> 4) & 7), c8 = ((tid & 7) ^ sw) * EP;   // row r = tid / 8 (+ 32 i) has pieces ^ (r / 2 % 8)
  const T* pa[BM / 32];
  const T* pb[BN / 32];
#pragma unroll
  for (int i = 0; i < BM / 32; i++) {
    const int sl = sslot[(tid >> 3) + 32 * i];
    pa[i] = x + (size_t)((sl >= 0 ? sl : sslot[0]) / x_div) * ldx;
  }
#pragma unroll
  for (int i = 0; i < BN / 32; i++) pb[i] = w + ((size_t)e * N + min(n0 + (tid >> 3) + 32 * i, N - 1)) * K;
  const unsigned lds0 = lds_address(tile) + wave * 1024;
  auto copy_step = [&](int k0, int st) {
    const int k = k0 + c8 < K ? k0 + c8 : 0;   // past the end: any numbers, struck out below
    const unsigned dst = lds0 + st * STAGE;
#pragma unroll
    for (int i = 0; i < BM / 32; i++) copy_lds16(pa[i] + k, dst + i * 4096);
#pragma unroll
    for (int i = 0; i < BN / 32; i++) copy_lds16(pb[i] + k, dst + BM * 128 + i * 4096);
  };
  f32x4 acc[FM][FN];
#pragma unroll
  for (int a = 0; a < FM; a++)
#pragma unroll
    for (int b = 0; b < FN; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  copy_step(0, 0);
  int st = 0;
  for (int k0 = 0; k0 < K; k0 += KS, st ^= 1) {
    tile_wait();
    __syncthreads();   // the step has landed, the other stage is free
    if (k0 + KS < K) copy_step(k0 + KS, st ^ 1);
    const unsigned char* sA = tile + st * STAGE + (wm + n16) * 128;
    const unsigned char* sB = tile + st * STAGE + BM * 128 + (wn + n16) * 128;
    uint4 af[2][FM], bf[2][FN];
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      const int at = ((kk * 4 + quad) ^ ((n16 >> 1) & 7)) * 16;
#pragma unroll
      for (int b = 0; b < FN; b++) bf[kk][b] = *(const uint4*)(sB + b * 2048 + at);
#pragma unroll
      for (int a = 0; a < FM; a++) af[kk][a] = *(const uint4*)(sA + a * 2048 + at);
    }
    if (k0 + KS > K) {   // the last step of a K that is no multiple: zeros past its end
#pragma unroll
      for (int kk = 0; kk < 2; kk++)
        if (k0 + (kk * 4 + quad) * EP >= K) {
#pragma unroll
          for (int a = 0; a < FM; a++) af[kk][a] = make_uint4(0, 0, 0, 0);
#pragma unroll
          for (int b = 0; b < FN; b++) bf[kk][b] = make_uint4(0, 0, 0, 0);
        }
    }
#pragma unroll
    for (int kk = 0; kk < 2; kk++)
#pragma unroll
      for (int a = 0; a < FM; a++)
        if (a < nmt) {
#pragma unroll
          for (int b = 0; b < FN; b++) acc[a][b] = mfma_piece<T>(bf[kk][b], af[kk][a], acc[a][b]);   // (see the stores)
        }
  }
  // The weight rows are the products' left operand, so a lane ends with four neighbouring columns of one slot: one store for
  // them, and little code behind the products (it is run once per tile, from memory).
#pragma unroll
  for (int a = 0; a < FM; a++) {
    if (a >= nmt) continue;
    const int so = sslot[wm + a * 16 + n16];
    if (so < 0) continue;
    T* o = out + (size_t)so * ldo;
    auto put = [&](int n, int end, const float (&v)[4]) {
      if (wide && n + 3 < end) {
        stv<4>(o, n, v);
        return;
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (n + i < end) stf(o, n + i, v[i]);
    };
    if (epi == 1 || epi == 3) {
#pragma unroll
      for (int b = 0; b < FN; b += 2) {
        const int n = n0 + wn + b * 16;            // (N is a multiple of 32)
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = glu_epi(acc[a][b][i], acc[a][b + 1][i], epi, limit, alpha);
        put(n / 2 + quad * 4, N / 2, v);
      }
      continue;
    }
#pragma unroll
    for (int b = 0; b < FN; b++) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = plain_epi(acc[a][b][i], epi);
      put(n0 + wn + b * 16 + quad * 4, N, v);
    }
  }
}

// The height of a prompt's expert tiles.  Tokens are taken to be routed at random: an expert has slots / E rows, give or take
// the root of that.  Fitted to sweeps of 540 to 8192 slots over 4, 8, 16, 32 and 64 experts of width 768 to 4096, evenly
// routed and skewed by a factor of 20; times below in us, all on one card.
struct TileHeight {
  int E, N, K, slots;
  double mean() const { return (double)slots / E; }
  int of(double n, int bm) const { return (int)ceil((n < 1 ? 1 : n) / bm); }
  // row tiles of all experts, when one has `dev` standard deviations more rows than the mean, and in the mean
  int most(int bm, double dev) const { return E * of(mean() + dev * sqrt(mean()), bm); }
  double middle(int bm, double dev) const {
    const double d = dev * sqrt(mean());
    return E * (of(mean() - d, bm) + 2 * of(mean(), bm) + of(mean() + d, bm)) / 4.0;
  }

  // Products bound, so a CU's time is the tiles it is given, never less than two deep (a lone block waits for memory):
  // 117 : 215 for a tile of 32 and of 64 rows.  The small tile fills the chip sooner (8 experts, gate and up, 64 -> 32 rows:
  // width 1024, 600 slots 40 -> 26, 1600 slots 62 -> 48; width 2048, 1800 slots 212 -> 183), the large one
  // needs 0.92 of the time per row where both do (width 2048, 700 slots 87 with 32 rows, 76 with 64, 4096 slots 356 and
  // 350).  Of 424 sizes 48 end above the faster one by more than 5 %, 1.09 at most with 8
  // experts of equal width, 1.25 with 32.
  double units(int bm) const {
    const int cols = (N + 63) / 64, pm = (((slots + bm - 1) / bm + E + 7) & ~7) / 8;
    // Two row tiles to an XCD at most: known exactly.  Blocks without a tile leave at once, and the hardware deals blocks to
    // its four shader engines in turn, so with pm row tiles launched the ones that exist count up to the next multiple of
    // gcd(pm, 4) (1024 columns x 64 on 4 experts: 512 blocks on half of the CUs, 161 us for 87).
    const int g = pm % 4 == 0 ? 4 : pm % 2 == 0 ? 2 : 1;
    const int pr = ((most(bm, 2) + 7) / 8 + g - 1) / g * g;
    if (pr <= 2 && cols * pr <= 64) return 2;
    const double x = middle(bm, 1.3) * cols / 256;
    return x >= 5 ? x + 0.4 : x + 0.3 <= 2 ? 2 : ceil(x + 0.3);
  }
  int f32() const { return 117 * units(32) < 215 * units(64) ? 32 : 64; }

  // us of a bf16 tile's rounds, or of reading each row tile's weights once through the caches at 8 TB/s
  double time(int bm, double tiles) const {
    const int cols = bm == 64 ? (N + 63) / 64 : (N + 127) / 128;
    const int n = (int)ceil(ceil(tiles / 8) * cols / 32);   // blocks to a CU: row tiles are dealt to 8 XCDs of 32 CUs
    static const float small[9] = {0, 10.3f, 11, 14, 18, 25.5f, 27, 30, 32.5f};
    const double k = K / 1024.0;
    const double work = bm == 64 ? (n <= 8 ? small[n] : 4.0 * n + 1) * k
                                 : (bm + 36) * 0.115 * (1.08 * (n / 2) + 0.92 * (n % 2)) * k;   // two blocks share a CU
    const double read = ceil(tiles) * N * K * 2 / 8e6;
    return work > read ? work : read;
  }
  // 64 x 64, or 128 x 128 once that gives one and a half blocks to a CU; 96 or 160 rows (or the other of the two) only where
  // they win by a twentieth with two standard deviations more rows than the mean, so that one crowded expert does not cost a
  // round.  8 experts, 64 / 96 / 128 / 160 rows: width 2048, gate and up, 4096 slots 67 / 54 / 65 / 45 (760 TFLOP/s), 2800
  // slots 51 / 53 / 39 / 43, 1800 slots 44 / 29 / 36 / 40, 1012 slots 25 / 28 / 34 / 35; width 1024, 4096 slots 25.9 / 18.6 /
  // 22.8 / 25.8; width 4096, down, 900 slots 48 / 62 / 38 / 39.  With 8
  // experts of equal width 4 of 136 sizes end above the pick of those two by more than 3 % (1.12), elsewhere 32 of 424 (1.36:
  // 4 experts of width 4096, 1200 slots).  (One workgroup of eight wavefronts per CU that
  // reads ahead, as the prompts' products have it, gave nothing here: 128 x 256 76 us, two rounds, where 128 x 128 had 69.)
  int bf16() const {
    const int old = (long)((slots + 127) / 128 + E) * ((N + 127) / 128) >= 384 ? 128 : 64;
    int best = 64;
    double t = time(64, most(64, 2));
    for (int bm : {96, 128, 160}) {
      const double u = time(bm, most(bm, 2));
      if (u < t) best = bm, t = u;
    }
    const double mid = middle(old, 1);
    return t < 0.95 * time(old, ceil(mid < 1 ? 1 : mid)) ? best : old;
  }
};

template <typename T, int BM, int BN>
static int launch_expert_tile(const void* x, int ldx, int x_div, const void* w, const int* cnt, const int* rows, int ldr,
                              void* out, int ldo, int E, int N, int K, int slots, int epi, float limit, float alpha,
                              hipStream_t st) {
  const int tmp = (((slots + BM - 1) / BM + E) + 7) & ~7;
  const size_t shm = (size_t)2 * (BM + BN) * 128;
  if (shm > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)expert_gemm_tile_k<T, BM, BN>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL((expert_gemm_tile_k<T, BM, BN>), dim3(tmp * ((N + BN - 1) / BN)), dim3(256), shm, st, (const T*)x,
                     ldx, x_div, (const T*)w, cnt, rows, ldr, (T*)out, ldo, N, K, E, tmp, epi, limit, alpha,
                     ldo % 4 == 0 && (size_t)out % (4 * sizeof(T)) == 0);
  return (int)hipGetLastError();
}

// any type, any shape: 32 slots x 64 columns per block, K staged through LDS 32 at a time
#define EG_KT 32
template <typename T>
__global__ void __launch_bounds__(256)
expert_gemm_fma_k(const T* __restrict__ x, int ldx, int x_div, const T* __restrict__ w,
                  const int* __restrict__ cnt, const int* __restrict__ rows, int ldr,
                  T* __restrict__ out, int ldo, int N, int K, int E, int TMP, int epi, float limit, float alpha) {
  __shared__ float sx[32][EG_KT + 1];
  __shared__ float sw[64][EG_KT + 1];
  __shared__ int sslot[32];
  int e, m0, nt;
  if (!find_tile(cnt, E, 32, TMP, e, m0, nt)) return;
  const int c = cnt[e], n0 = nt * 64;
  const int tid = threadIdx.x;
  if (tid < 32) sslot[tid] = m0 + tid < c ? rows[(size_t)e * ldr + m0 + tid] : -1;
  __syncthreads();
  // thread (ty, tx): slots ty*2 .. ty*2+1, columns tx + 16*u
  const int tx = tid & 15, ty = tid >> 4;
  float acc[2][4];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int u = 0; u < 4; u++) acc[a][u] = 0.0f;
  for (int k0 = 0; k0 < K; k0 += EG_KT) {
    for (int idx = tid; idx < 32 * EG_KT; idx += 256) {
      int m = idx / EG_KT, k = idx % EG_KT;
      int s = sslot[m];
      sx[m][k] = (s >= 0 && k0 + k < K) ? ldf(x, (size_t)(s / x_div) * ldx + k0 + k) : 0.0f;
    }
    for (int idx = tid; idx < 64 * EG_KT; idx += 256) {
      int n = idx / EG_KT, k = idx % EG_KT;
      sw[n][k] = (n0 + n < N && k0 + k < K) ? ldf(w, ((size_t)e * N + n0 + n) * K + k0 + k) : 0.0f;
    }
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < EG_KT; k++) {
      float xa = sx[ty * 2][k], xb = sx[ty * 2 + 1][k];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        float wv = sw[tx + 16 * u][k];
        acc[0][u] += xa * wv;
        acc[1][u] += xb * wv;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < 2; a++) {
    int s = sslot[ty * 2 + a];
    if (s < 0) continue;
    if (epi == 1 || epi == 3) {
#pragma unroll
      for (int u = 0; u < 4; u += 2) {
        int n = n0 + 16 * u;
        if (n + 16 + tx < N)
          stf(out, (size_t)s * ldo + n / 2 + tx,
              glu_epi(acc[a][u], acc[a][u + 1], epi, limit, alpha));
      }
      continue;
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      int n = n0 + tx + 16 * u;
      if (n < N) stf(out, (size_t)s * ldo + n, plain_epi(acc[a][u], epi));
    }
  }
}

// out[r] = sum_k wts[r, k] * y[r * top + k]; a slot whose expert index is >= n_real (ids given)
// stands for an expert that hands its input back: its term is wts * x[r]
// VE channels per thread (2048 rows of 2048, two experts each, one / four: 12.8 / 7.4 us)
template <typename T, int VE>
__global__ void expert_combine_k(const T* __restrict__ y, int ldy, const float* __restrict__ wts,
                                 T* __restrict__ out, int ldo, int top, int n,
                                 const int* __restrict__ ids, int n_real, const T* __restrict__ x,
                                 int ldx) {
  int c = (blockIdx.x * blockDim.x + threadIdx.x) * VE, r = blockIdx.y;
  if (c >= n) return;
  float s[VE];
#pragma unroll
  for (int j = 0; j < VE; j++) s[j] = 0.0f;
  for (int k = 0; k < top; k++) {
    bool same = ids && ids[r * top + k] >= n_real;
    float v[VE];
    ldv<VE>(same ? x : y, same ? (size_t)r * ldx + c : (size_t)(r * top + k) * ldy + c, v);
#pragma unroll
    for (int j = 0; j < VE; j++) s[j] += wts[r * top + k] * v[j];
  }
  stv<VE>(out, (size_t)r * ldo + c, s);
}

extern "C" {

// cnt must be zero on entry
int p2p_sm_group_route(const void* h, int ldh, const float* wr, int R, int W, int E, int top,
                       int groups, int keep, int score, const float* corr, int gscore, int* ids,
                       float* wts, int* cnt, int* rows, int ldr, const float* bias, int renorm,
                       float wscale, int f32, hipStream_t st) {
  if (R <= 0) return 0;
  if (E < 1 || groups < 1 || E % groups || keep < 1 || keep > groups || top < 1 ||
      top > keep * (E / groups) || ldr < R * top)
    return (int)hipErrorInvalidValue;
  size_t shm = (size_t)(W + 2 * E + groups + top) * 4;
  if (shm > 64 * 1024) return (int)hipErrorInvalidValue;
  const size_t many = (size_t)(16 * (2 * E + groups + 3 * top) + E) * 4;
#define ROUTE_ROWS(NB)                                                                                          \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((group_route_rows_k<T, NB>), dim3((R + 15) / 16), dim3(1024), many, st, \
                                         (const T*)h, ldh, wr, R, W, E, top, groups, keep, score, corr, gscore, ids, wts, \
                                         cnt, rows, ldr, bias, renorm, wscale))
  // Up to 32 experts: sixteen rows' logits on the matrix instruction, from as many rows on as make one row per workgroup (below)
  // the longer chain.  A workgroup's products grow with the numbers of a row, in fp32 and above 16 experts (two products per
  // step) faster than one row's share.  us, one / sixteen: bf16, 8 experts, 1024 numbers, 100 rows 9.0 / 9.3, 200 11.2 / 9.4,
  // 700 13.5 / 9.6; 2048, 150 rows 11.1 / 11.3, 200 12.2 / 11.3, 2048 rows 19.9 / 12.3; 4096, 200 14.6 / 15.3, 256 15.8 / 15.3;
  // 32 experts, 2048, 200 13.2 / 16.6, 400 16.5 / 17.0, 700 21.0 / 16.8; fp32, 8 experts, 2048, 200 12.4 / 13.0, 300 14.7 /
  // 13.0; 4096, 300 17.1 / 18.7, 400 19.6 / 18.7; 32 experts, 2048, 400 16.1 / 18.3, 700 21.0 / 18.5.
  // The logits' sums have another order then (fp32 both): experts whose scores are as close as fp32 rounding of W products
  // may be chosen otherwise in a step of so many rows than in a smaller one.
  const int ep = f32 ? 4 : 8;
  const int from = max(200, E <= 16 ? f32 ? 90 + W / 12 : 120 + W / 26 : f32 ? 240 + W / 8 : 190 + W / 10);
  if (R >= from && E <= 32 && W % ep == 0 && ldh % ep == 0 && (size_t)h % 16 == 0 && (size_t)wr % 16 == 0) {
    if (E <= 16) ROUTE_ROWS(1);
    else ROUTE_ROWS(2);
    return (int)hipGetLastError();
  }
  // Sixteen rows per workgroup take as long as one row's E sums of W products by one wavefront, whatever R is (until
  // the chip is full); one row per workgroup takes its slots' atomics, R of them, and shares a row's sums among four
  // wavefronts.  us, one / sixteen: E * W = 8192, 256 rows 10.0 / 10.9, 606 rows 18.3 / 11.1; 16384, 606 rows 19 /
  // 17; 65536, 1024 rows 40 / 54, 2048 rows 68 / 55; 262144, 2048 rows 92 / 188
  if (R >= 256 && (size_t)R * 28 >= (size_t)E * W && many <= 48 * 1024) {
    ROUTE_ROWS(0);
    return (int)hipGetLastError();
  }
#undef ROUTE_ROWS
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(group_route_k<T>, dim3(R), dim3(256), shm, st,
                                         (const T*)h, ldh, wr, W, E, top, groups, keep, score, corr,
                                         gscore, ids, wts, cnt, rows, ldr, bias, renorm, wscale));
  return (int)hipGetLastError();
}

// total_slots: slots over all experts (rows * top; every slot is in exactly one list).
// epi = 1: w holds gate / up rows interleaved in groups of 16 (N = 2F rows, a multiple of 32)
// and out [slots, F] receives the experts' activation instead of the raw products.
// rows of a prompt's expert tiles (0: few slots, no tiles)
int p2p_sm_expert_tile(int E, int N, int K, int total_slots, int f32) {
  if (E < 1 || N < 1 || K < 1 || total_slots < 64 * E) return 0;
  const TileHeight pick{E, N, K, total_slots};
  return f32 ? pick.f32() : pick.bf16();
}

int p2p_sm_expert_gemm(const void* x, int ldx, int x_div, const void* w, const int* cnt,
                       const int* rows, int ldr, void* out, int ldo, int E, int N, int K,
                       int total_slots, int epi, float limit, float alpha, int f32,
                       hipStream_t st) {
  if (total_slots <= 0 || E <= 0) return 0;
  if (x_div < 1 || N < 1 || K < 1 || ((epi == 1 || epi == 3) && N % 32))
    return (int)hipErrorInvalidValue;
  const int ep = f32 ? 4 : 8;   // numbers per 16 bytes
  if (K % ep == 0 && ldx % ep == 0 && ((size_t)x & 15) == 0 && ((size_t)w & 15) == 0) {
    if (total_slots >= 64 * E) {   // prompts: tiles
#define ET(T, BM, BN)                                                                                        \
  return launch_expert_tile<T, BM, BN>(x, ldx, x_div, w, cnt, rows, ldr, out, ldo, E, N, K, total_slots, epi, \
                                       limit, alpha, st)
      const TileHeight pick{E, N, K, total_slots};
      if (f32) {
        if (pick.f32() == 32) ET(float, 32, 64);
        ET(float, 64, 64);
      }
      switch (pick.bf16()) {
        case 64: ET(bf16, 64, 64);
        case 96: ET(bf16, 96, 128);
        case 128: ET(bf16, 128, 128);
        default: ET(bf16, 160, 128);
      }
#undef ET
    }
    int tmp = (((total_slots + 15) / 16 + E) + 7) & ~7;
    dim3 grid(tmp * ((N + 63) / 64));
#define EM(DEPTH)                                                                                                     \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((expert_gemm_mfma_k<T, DEPTH>), grid, dim3(256), 0, st, (const T*)x, ldx, x_div, \
                                         (const T*)w, cnt, rows, ldr, (T*)out, ldo, N, K, E, tmp, epi, limit, alpha))
    if (K > 128 * ep) EM(4);   // 4 wavefronts x 8 steps of 4 pieces
    else EM(2);
#undef EM
    return (int)hipGetLastError();
  }
  int tmp = (((total_slots + 31) / 32 + E) + 7) & ~7;
  dim3 grid(tmp * ((N + 63) / 64));
  SM_DISPATCH_T(f32, hipLaunchKernelGGL(expert_gemm_fma_k<T>, grid, dim3(256), 0, st,
                                         (const T*)x, ldx, x_div, (const T*)w, cnt, rows, ldr,
                                         (T*)out, ldo, N, K, E, tmp, epi, limit, alpha));
  return (int)hipGetLastError();
}

int p2p_sm_expert_combine(const void* y, int ldy, const float* wts, void* out, int ldo, int R,
                          int top, int n, const int* ids, int n_real, const void* x, int ldx,
                          int f32, hipStream_t st) {
  if (R <= 0) return 0;
  if (ids && !x) return (int)hipErrorInvalidValue;
  const size_t al = f32 ? 16 : 8;
#define COMBINE(VE)                                                                                                  \
  SM_DISPATCH_T(f32, hipLaunchKernelGGL((expert_combine_k<T, VE>), dim3((n + 256 * VE - 1) / (256 * VE), R), dim3(256), \
                                         0, st, (const T*)y, ldy, wts, (T*)out, ldo, top, n, ids, n_real, (const T*)x, ldx))
  if (n % 4 == 0 && ldy % 4 == 0 && ldo % 4 == 0 && ((size_t)y | (size_t)out) % al == 0 &&
      (!ids || (ldx % 4 == 0 && (size_t)x % al == 0)))
    COMBINE(4);
  else COMBINE(1);
#undef COMBINE
  return (int)hipGetLastError();
}

}  // extern "C"
