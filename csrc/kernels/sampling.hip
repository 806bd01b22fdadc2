// Ollama-style stochastic sampling on the GPU: temperature -> top-k ->
// top-p -> multinomial draw, one workgroup per row, graph-capturable (all
// per-row parameters live in device memory; the random stream is a counter-based
// hash of (seed, position, token id), so a replayed graph draws fresh numbers
// every step without host state).
//
// A row of a real vocabulary (24449 to 262144 logits; row_groups() has the exceptions) takes two launches: one workgroup
// per row reads 513 KB twice and selects and sorts between 28 barriers, 28 us at 128256 logits whatever the batch (up to
// the CUs; back to back, 33 behind another kernel), and that chain, not memory, is what bounds it.  So
//   a. row_groups_kernel leaves the largest key of every 128 neighbouring logits, by as many workgroups as
//      the rows have (one read of the logits: 4.7 us for a row, launch and all, 6.1 for 32);
//   b. sample_kernel takes a bound from those maxima that at least k logits reach, reads only the groups that
//      reach it (about 45 of 1002 at k = 40) and ranks what it finds by counting: no histogram, no sort.
// Both sides give the same candidates in the same order, so the same tokens.  Back to back, k = 40: 128256 logits
// 27.7 -> 11.8 us for 1 row and 35.3 -> 18.1 for 64, 32000 logits 18.9 -> 11.9, 128256 with k = 128 28.5 -> 17.7; what is left is
// two launches' ends and the chain of the second (maxima, bound, groups, ranks, draw).
// Other rows (small vocabularies, gathered shards, and rows with more than 1024 logits at the bound: ties)
// are selected by one workgroup (1024 threads = 16 waves, the row stays L2-resident across passes):
//   1. top-k threshold by an MSB-first radix select over the order-preserving
//      32-bit keys of the fp32 logits: 4 passes of 8 bits, per-wave LDS histograms
//      (16 x 256 bins) summed, wave 0 finds the bin holding the k-th largest by a
//      shuffle suffix-scan.  The k-th largest key T is exact after 4 passes.  A
//      prefilter first bounds T from below by the k-th largest per-thread maximum,
//      so the passes run over a few hundred LDS-resident entries, not the row.
//   2. collect the k candidates: every key > T, then the keys == T with the lowest
//      ids (a second radix select over ~id, only when the k-th value is tied).
//   3. bitonic sort of the (<= 128) candidates in LDS, descending value, ascending id.
// Then, on either side:
//   4. softmax(v / temperature) over them, inclusive cumsum; keep the smallest
//      prefix whose mass reaches top_p (drop i when cum_i - p_i > top_p).
//   5. exponential race: token = argmax_i p_i / E_i with E_i ~ Exp(1) -- exactly a
//      draw from the renormalised kept distribution.
// temperature <= 0 rows are greedy (argmax, lowest id on ties, like torch).
// The same semantics as engine/sampling.py (the CPU reference and the test oracle).
#include "common.h"

namespace {

constexpr int THREADS = 1024;
constexpr int NWAVES = THREADS / 64;
constexpr int KMAX = 128;
constexpr int CAP = 4096;  // prefiltered candidates held in LDS

// Groups of a row (kernel a).  128 logits: a wave's two loads, and 1002 maxima of 128256 logits are 16 a lane of
// the wave that picks the bound.  At least 128 groups, so that any k has as many maxima; at most 32 a lane.
constexpr int GROUP = 128;
constexpr int GROUPS_MIN = KMAX, GROUPS_MAX = 2048;
constexpr int GPW = 4;          // groups per wave of kernel a: 8 loads in flight per lane
constexpr int RANKED = 1024;    // candidates ranked by counting (more: the radix select)

__device__ __forceinline__ unsigned ord_key(float v) {
  unsigned u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_float(unsigned u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

// splitmix64 finaliser: a well-mixed 64-bit hash of the draw's coordinates
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {
  z += 0x9e3779b97f4a7c15ull;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// uniform in (0, 1) from (seed, pos, token): 24 random bits, centred in their cell
__device__ __forceinline__ float uniform01(unsigned long long seed, int pos, int tok) {
  const unsigned long long h =
      mix64(seed ^ mix64(((unsigned long long)(unsigned)pos << 32) | (unsigned)tok));
  return ((float)(h >> 40) + 0.5f) * (1.0f / 16777216.0f);
}

// Key of the greedy choice: NaN below every number (they are never chosen), -0 equal to 0.
__device__ __forceinline__ unsigned greedy_key(float v) { return v != v ? 0u : ord_key(v + 0.f); }

// gmax[r][g] <- the largest key of logits [128 g, 128 g + 128) of row r; greedy rows by greedy_key.
__global__ __launch_bounds__(256) void row_groups_kernel(const float* __restrict__ logits, int ld, int V,
                                                         int NG, const float* __restrict__ temp,
                                                         unsigned* __restrict__ gmax) {
  const int r = blockIdx.y, lane = threadIdx.x & 63;
  const int g0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * GPW;
  const float* row = logits + (size_t)r * ld;
  const bool greedy = temp && !(temp[r] > 0.f);
  float x[GPW][2];
#pragma unroll
  for (int j = 0; j < GPW; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) x[j][e] = row[min((g0 + j) * GROUP + 64 * e + lane, V - 1)];
#pragma unroll
  for (int j = 0; j < GPW; ++j) {
    // a group past the end reads the last logit again and is not stored; the last group reads it again in
    // its own range, which leaves its maximum as it is
    unsigned m = greedy ? max(greedy_key(x[j][0]), greedy_key(x[j][1])) : max(ord_key(x[j][0]), ord_key(x[j][1]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    if (lane == 0 && g0 + j < NG) gmax[(size_t)r * NG + g0 + j] = m;
  }
}

// Entry sources of one row: a dense logits row (ids = column + id_off), or -- vocab-
// parallel TP -- the gathered per-shard candidates: entry i of row r is slot i % seg of
// segment i / seg (one per rank), at vals/ids[(i / seg) * seg_stride + r * seg + i % seg].
struct Src {
  const float* vals;
  const int* ids;  // null: dense row
  int ld, seg;
  long long seg_stride;
  int id_off;
};

__global__ __launch_bounds__(THREADS) void sample_kernel(
    Src src, int V, const float* __restrict__ temp,
    const int* __restrict__ topk, const float* __restrict__ topp,
    const unsigned long long* __restrict__ seeds, const int* __restrict__ pos,
    int* __restrict__ out, float* __restrict__ cand_v, int* __restrict__ cand_id,
    const unsigned* __restrict__ gmax, int NG) {
  // gmax != null (dense rows only): the row's group maxima, from row_groups_kernel
  // cand_v != null: emit mode -- write this row's top-KMAX (value, id) pairs, sorted
  // (descending value, ascending id; padding -inf / INT_MAX) instead of drawing
  const int r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const bool emit = cand_v != nullptr;
  const float* row = src.vals + (size_t)r * src.ld;
  const bool vec = !src.ids && ((src.ld | V) & 3) == 0;
  const float T = emit ? 1.f : temp[r];
  auto for_each_key = [&](const float* __restrict__, int, bool, auto&& f) {
    if (src.ids) {
      for (int i = threadIdx.x; i < V; i += THREADS) {
        const size_t o = (size_t)(i / src.seg) * src.seg_stride + (size_t)r * src.seg + i % src.seg;
        f(src.ids[o], src.vals[o]);
      }
    } else if (vec) {
      const float4* r4 = reinterpret_cast<const float4*>(row);
      for (int i = threadIdx.x; i < (V >> 2); i += THREADS) {
        const float4 x = r4[i];
        f(src.id_off + 4 * i + 0, x.x);
        f(src.id_off + 4 * i + 1, x.y);
        f(src.id_off + 4 * i + 2, x.z);
        f(src.id_off + 4 * i + 3, x.w);
      }
    } else {
      for (int i = threadIdx.x; i < V; i += THREADS) f(src.id_off + i, row[i]);
    }
  };

  __shared__ int hist[NWAVES][256];
  __shared__ float cv[KMAX];
  __shared__ int ci[KMAX];
  __shared__ int s_bin, s_kr, s_cnt, s_ngt, s_ntie, s_nc;
  __shared__ unsigned s_tmk[THREADS];  // per-thread max keys (prefilter)
  __shared__ unsigned s_ck[CAP];       // prefiltered candidates: key, id
  __shared__ int s_ci[CAP];
  __shared__ float s_bestv[NWAVES];
  __shared__ int s_besti[NWAVES];
  __shared__ unsigned short s_list[GROUPS_MAX];  // groups that reach the bound
  __shared__ int s_nl;
  __shared__ unsigned s_bound;

  if (gmax && !(T > 0.f)) {  // greedy: the first group that holds the largest key, then its first logit
    if (w == 0) {
      const unsigned* gm = gmax + (size_t)r * NG;
      unsigned bk = 0u;
      int bg = 0;
      for (int g = lane; g < NG; g += 64) {
        const unsigned u = gm[g];
        if (u > bk) { bk = u; bg = g; }
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const unsigned ok = (unsigned)__shfl_xor((int)bk, o, 64);
        const int og = __shfl_xor(bg, o, 64);
        if (ok > bk || (ok == bk && og < bg)) { bk = ok; bg = og; }
      }
      const int i0 = bg * GROUP + lane, i1 = i0 + 64;
      const unsigned u0 = i0 < V ? greedy_key(row[i0]) : 0u, u1 = i1 < V ? greedy_key(row[i1]) : 0u;
      const unsigned long long h0 = __ballot(u0 == bk), h1 = __ballot(u1 == bk);
      // bk 0: a row of NaN only
      if (lane == 0)
        out[r] = bk == 0u ? 0 : src.id_off + bg * GROUP + (h0 ? __ffsll(h0) - 1 : 63 + __ffsll(h1));
    }
    return;
  }
  if (!(T > 0.f)) {  // greedy
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    for_each_key(row, V, vec, [&](int i, float x) {
      if (x > bv || (x == bv && i < bi)) { bv = x; bi = i; }
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (lane == 0) { s_bestv[w] = bv; s_besti[w] = bi; }
    __syncthreads();
    if (tid == 0) {
      for (int i = 1; i < NWAVES; ++i)
        if (s_bestv[i] > bv || (s_bestv[i] == bv && s_besti[i] < bi)) { bv = s_bestv[i]; bi = s_besti[i]; }
      out[r] = bi == 0x7fffffff ? 0 : bi;
    }
    return;
  }

  int k = emit ? KMAX : topk[r];
  if (k <= 0 || k > KMAX) k = KMAX;
  if (k > V) k = V;

  // ---- the groups that reach a bound, ranked by counting ----
  bool ranked = false;
  if (gmax) {
    if (w == 0) {
      // The bound: the largest t found, bit by bit, that at least k of 256 maxima reach (the maximum over the
      // groups g, g + 256, ... for each of 256), and so at least k logits; it need not be the k-th, so
      // the search ends at k to k + 8.  About 45 groups pass at k = 40, 160 at k = 128.
      const unsigned* gm = gmax + (size_t)r * NG;
      unsigned gk[GROUPS_MAX / 64];
#pragma unroll
      for (int j = 0; j < GROUPS_MAX / 64; ++j)
        gk[j] = gm[min(64 * j + lane, NG - 1)];
      unsigned top[4] = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < GROUPS_MAX / 64; ++j) {
        if (64 * j + lane >= NG) gk[j] = 0u;
        top[j & 3] = max(top[j & 3], gk[j]);
      }
      unsigned t = 0u;
      for (unsigned bit = 0x80000000u; bit; bit >>= 1) {
        const unsigned c = t | bit;
        int n = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) n += __popcll(__ballot(top[j] >= c));
        if (n >= k) {
          t = c;
          if (n <= k + 8) break;
        }
      }
      int n = 0;
#pragma unroll
      for (int j = 0; j < GROUPS_MAX / 64; ++j) {
        const bool in = 64 * j + lane < NG && gk[j] >= t;
        const unsigned long long b = __ballot(in);
        if (in) s_list[n + __popcll(b & ((1ull << lane) - 1))] = (unsigned short)(64 * j + lane);
        n += __popcll(b);
      }
      if (lane == 0) { s_nl = n; s_bound = t; s_nc = 0; }
    }
    __syncthreads();
    const int nl = s_nl;
    const unsigned t = s_bound;
    constexpr int NB = 4;  // groups of a wave at a time: 8 loads in flight per lane
    for (int l0 = w; l0 < nl; l0 += NB * NWAVES) {
      float x[NB][2];
      int id[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        id[j] = (int)s_list[min(l0 + j * NWAVES, nl - 1)] * GROUP + lane;
        x[j][0] = row[min(id[j], V - 1)];
        x[j][1] = row[min(id[j] + 64, V - 1)];
      }
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int i = id[j] + 64 * e;
          const unsigned u = ord_key(x[j][e]);
          if (l0 + j * NWAVES < nl && i < V && u >= t) {
            const int sidx = atomicAdd(&s_nc, 1);
            if (sidx < RANKED) { s_ck[sidx] = u; s_ci[sidx] = src.id_off + i; }
          }
        }
    }
    __syncthreads();
    const int nc = s_nc;
    ranked = nc <= RANKED;
    if (ranked) {
      // rank of a candidate = how many come before it, four threads a candidate; ranks below k are in
      for (int c0 = 0; c0 < nc; c0 += THREADS / 4) {
        const int c = c0 + (tid >> 2);
        const unsigned u = s_ck[min(c, nc - 1)];
        const int i = s_ci[min(c, nc - 1)];
        int n = 0;
#pragma unroll 8
        for (int q = tid & 3; q < nc; q += 4) {  // both reads of every turn go out ahead of their comparison
          const unsigned uq = s_ck[q];
          const int iq = s_ci[q];
          n += (uq > u) | ((uq == u) & (iq < i));
        }
        n += __shfl_xor(n, 1, 64);
        n += __shfl_xor(n, 2, 64);
        if ((tid & 3) == 0 && c < nc && n < k) { s_tmk[n] = u; s_ci[RANKED + n] = i; }
      }
      __syncthreads();
      // ... and their order by value, where -0 and 0 are equal and the lower id comes first
      const int c = tid >> 2;
      if (c < KMAX) {
        const int cc = min(c, k - 1), i = s_ci[RANKED + cc];
        const float v = key_float(s_tmk[cc]);
        const unsigned u = ord_key(v + 0.f);
        int n = 0;
#pragma unroll 8
        for (int q = tid & 3; q < k; q += 4) {
          const unsigned uq = ord_key(key_float(s_tmk[q]) + 0.f);
          const int iq = s_ci[RANKED + q];
          n += (uq > u) | ((uq == u) & (iq < i));
        }
        n += __shfl_xor(n, 1, 64);
        n += __shfl_xor(n, 2, 64);
        if ((tid & 3) == 0) {
          if (c < k) {
            cv[n] = v;
            ci[n] = i;
          } else {
            cv[c] = -INFINITY;
            ci[c] = 0x7fffffff;
          }
        }
      }
      __syncthreads();
    }
  }
  if (!ranked) {
    // ---- 1. radix select of the k-th largest (value, -id) pair ----
    // One MSB-first 8-bit digit per pass over the keys that match the prefix so far
    // (per-wave LDS histograms; wave 0 finds the bin by a shuffle suffix-scan).  Phase
    // A selects on the value key; if the k-th value is tied with more keys than remain
    // to be taken, phase B selects among those ties on ~id (ascending ids win), so the
    // candidate set is exact and deterministic.  `each(f)` enumerates (id, key) pairs.
    auto radix_pass = [&](auto&& each, auto&& digit_of) {  // -> s_bin / s_kr / s_cnt
      for (int i = lane; i < 256; i += 64) hist[w][i] = 0;
      __syncthreads();
      each([&](int i, unsigned key) {
        unsigned d;
        if (digit_of(i, key, &d)) atomicAdd(&hist[w][d], 1);
      });
      __syncthreads();
      if (w == 0) {
        int c[4];
        int s = 0;
  #pragma unroll
        for (int j = 0; j < 4; ++j) {
          int t = 0;
  #pragma unroll
          for (int ww = 0; ww < NWAVES; ++ww) t += hist[ww][4 * lane + j];
          c[j] = t;
          s += t;
        }
        int suf = s;  // keys in bins >= 4*lane
  #pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int t = __shfl_down(suf, o, 64);
          if (lane + o < 64) suf += t;
        }
        int above = suf - s;  // keys in bins > 4*lane+3
        const int kr0 = s_kr;
        if (above < kr0 && suf >= kr0) {  // the kr-th largest lies in this lane's 4 bins
  #pragma unroll
          for (int j = 3; j >= 0; --j) {
            if (above + c[j] >= kr0) {
              s_bin = 4 * lane + j;
              s_cnt = c[j];
              s_kr = kr0 - above;
              break;
            }
            above += c[j];
          }
        }
      }
      __syncthreads();
    };
    // k-th largest (value key, ~id) among `each`'s pairs: returns (value key, ties taken,
    // id threshold: ties with ~id >= thr are in)
    auto select = [&](auto&& each, int kk, unsigned* vkey, int* kr_out, unsigned* idthr) {
      if (tid == 0) s_kr = kk;
      unsigned prefix = 0u, mask = 0u;
      for (int shift = 24; shift >= 0; shift -= 8) {
        radix_pass(each, [&](int, unsigned u, unsigned* d) {
          *d = (u >> shift) & 255u;
          return (u & mask) == prefix;
        });
        prefix |= (unsigned)s_bin << shift;
        mask |= 255u << shift;
      }
      const int kr = s_kr;
      unsigned thr = 0u;
      if (s_cnt > kr) {
        unsigned ip = 0u, im = 0u;
        for (int shift = 24; shift >= 0; shift -= 8) {
          radix_pass(each, [&](int i, unsigned u, unsigned* d) {
            const unsigned ni = ~(unsigned)i;
            *d = (ni >> shift) & 255u;
            return u == prefix && (ni & im) == ip;
          });
          ip |= (unsigned)s_bin << shift;
          im |= 255u << shift;
        }
        thr = ip;
      }
      *vkey = prefix;
      *kr_out = kr;
      *idthr = thr;
    };
    auto each_row = [&](auto&& f) {
      for_each_key(row, V, vec, [&](int i, float x) { f(i, ord_key(x)); });
    };

    // Prefilter: the k-th largest of the 1024 per-thread maxima is a key with at least
    // k row entries at or above it, so only those entries (typically a few hundred)
    // can be in the top k.  They are gathered to LDS and selected there; a row with
    // more than CAP such entries (massive ties) is selected over the whole row instead.
    float tmax = -INFINITY;
    for_each_key(row, V, vec, [&](int, float x) { tmax = fmaxf(tmax, x); });
    s_tmk[tid] = ord_key(tmax);
    unsigned t0key;
    {
      int kr_;
      unsigned thr_;
      select([&](auto&& f) { f(tid, s_tmk[tid]); }, min(k, THREADS), &t0key, &kr_, &thr_);
    }
    if (tid == 0) s_nc = 0;
    __syncthreads();
    each_row([&](int i, unsigned u) {
      if (u >= t0key) {
        const int sidx = atomicAdd(&s_nc, 1);
        if (sidx < CAP) { s_ck[sidx] = u; s_ci[sidx] = i; }
      }
    });
    __syncthreads();
    const int nc = s_nc;
    const bool small = nc <= CAP;
    auto each_cand = [&](auto&& f) {
      for (int j = tid; j < nc; j += THREADS) f(s_ci[j], s_ck[j]);
    };
    unsigned prefix, idthr;
    int kr;
    if (small)
      select(each_cand, k, &prefix, &kr, &idthr);
    else
      select(each_row, k, &prefix, &kr, &idthr);
    const int n_gt = k - kr;

    // ---- 2. collect the k candidates ----
    if (tid == 0) {
      s_ngt = 0;
      s_ntie = 0;
    }
    __syncthreads();
    auto take = [&](int i, unsigned u) {
      if (u > prefix) {
        const int sidx = atomicAdd(&s_ngt, 1);
        if (sidx < KMAX) { cv[sidx] = key_float(u); ci[sidx] = i; }
      } else if (u == prefix && ~(unsigned)i >= idthr) {
        const int sidx = atomicAdd(&s_ntie, 1);
        if (sidx < kr) { cv[n_gt + sidx] = key_float(u); ci[n_gt + sidx] = i; }
      }
    };
    if (small)
      each_cand(take);
    else
      each_row(take);
    __syncthreads();

    // ---- 3. bitonic sort (descending value, ascending id), KMAX slots padded ----
    if (tid < KMAX && tid >= k) {
      cv[tid] = -INFINITY;
      ci[tid] = 0x7fffffff;
    }
    __syncthreads();
    for (int size = 2; size <= KMAX; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        if (tid < KMAX) {
          const int j = tid ^ stride;
          if (j > tid) {
            const bool desc = (tid & size) == 0;  // descending overall
            const float a = cv[tid], b = cv[j];
            const int ia = ci[tid], ib = ci[j];
            // "a before b" in the final (descending value, ascending id) order
            const bool a_first = a > b || (a == b && ia < ib);
            if (desc != a_first) {
              cv[tid] = b; cv[j] = a;
              ci[tid] = ib; ci[j] = ia;
            }
          }
        }
        __syncthreads();
      }
    }
  }

  if (emit) {
    if (tid < KMAX) {
      cand_v[(size_t)r * KMAX + tid] = cv[tid];
      cand_id[(size_t)r * KMAX + tid] = ci[tid];
    }
    return;
  }

  // ---- 4 + 5. softmax / top-p / exponential race, wave 0 (2 slots per lane) ----
  if (w == 0) {
    const float vmax = cv[0];
    const float invT = 1.f / T;
    float p[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = 2 * lane + j;
      p[j] = i < k ? __expf((cv[i] - vmax) * invT) : 0.f;
    }
    const float tot = wave_sum(p[0] + p[1]);
    p[0] /= tot;
    p[1] /= tot;
    // inclusive prefix sum over slots 0..127 (lane-major: slot 2*lane + j)
    float ls = p[0] + p[1];
    float inc = ls;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const float t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    const float base = inc - ls;  // mass of slots before 2*lane
    const float cum0 = base + p[0], cum1 = cum0 + p[1];
    const float top_p = topp[r];
    const bool keep0 = 2 * lane < k && (cum0 - p[0]) <= top_p;
    const bool keep1 = 2 * lane + 1 < k && (cum1 - p[1]) <= top_p;
    const unsigned long long seed = seeds[r];
    const int ps = pos[r];
    float best = -1.f;
    int bid = 0x7fffffff;
    if (keep0) {
      best = p[0] / -__logf(uniform01(seed, ps, ci[2 * lane]));
      bid = ci[2 * lane];
    }
    if (keep1) {
      const float sc = p[1] / -__logf(uniform01(seed, ps, ci[2 * lane + 1]));
      if (sc > best) { best = sc; bid = ci[2 * lane + 1]; }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bid, o, 64);
      if (ob > best || (ob == best && oi < bid)) { best = ob; bid = oi; }
    }
    if (lane == 0) out[r] = bid == 0x7fffffff ? ci[0] : bid;
  }
}

}  // namespace

// Group maxima a row of V logits needs in the workspace of the two calls below; 0: none (one workgroup per row).
P2P_API int p2p_sample_groups(int V) {
  const int ng = (V + GROUP - 1) / GROUP;
  return ng >= GROUPS_MIN && ng <= GROUPS_MAX ? ng : 0;
}

static int row_groups(const float* logits, int ld, int B, int V, const float* temp, unsigned* ws, int* ng,
                      hipStream_t st) {
  *ng = ws ? p2p_sample_groups(V) : 0;
  // Below 192 groups k = 128 finds logits in most of them, and the launch of kernel a is not won back (16384 logits, one
  // workgroup per row / two launches: k = 128 18.2 / 26.4 us, but k = 40 17.6 / 11.7).  For many rows, which fill the CUs by
  // themselves, both are level at the worst k (32000 logits, 256 rows: k = 128 23.6 / 24.0, 40 23.1 / 18.5, 1 22.5 / 15.7;
  // greedy rows 8.6 / 11.8, which only come beside sampled ones: a step of greedy rows takes its argmax).
  if (*ng < 192) *ng = 0;
  if (*ng == 0) return 0;
  const int wgs = (*ng + 4 * GPW - 1) / (4 * GPW);
  for (int r = 0; r < B; r += 65535)  // grid.y
    hipLaunchKernelGGL(row_groups_kernel, dim3(wgs, min(B - r, 65535)), dim3(256), 0, st,
                       logits + (size_t)r * ld, ld, V, *ng, temp ? temp + r : nullptr, ws + (size_t)r * *ng);
  return (int)hipGetLastError();
}

// ids[r] <- a draw from row r of logits [B, V] (row stride ld) with per-row
// temperature (<= 0: greedy), top_k (<= 0 or > 128: 128), top_p, and a random
// stream keyed by (seeds[r], pos[r], token id).  ws: B * p2p_sample_groups(V) words (or null).
P2P_API int p2p_sample(const float* logits, int ld, int B, int V, const float* temp,
                       const int* topk, const float* topp, const unsigned long long* seeds,
                       const int* pos, int* ids, unsigned* ws, hipStream_t st) {
  if (B <= 0 || V <= 0 || ld < V) return (int)hipErrorInvalidValue;
  int ng = 0;
  const int e = row_groups(logits, ld, B, V, temp, ws, &ng, st);
  if (e) return e;
  Src src{logits, nullptr, ld, 0, 0, 0};
  hipLaunchKernelGGL(sample_kernel, dim3(B), dim3(THREADS), 0, st, src, V, temp, topk, topp,
                     seeds, pos, ids, (float*)nullptr, (int*)nullptr, ng ? ws : (const unsigned*)nullptr, ng);
  return (int)hipGetLastError();
}

// Vocab-parallel sampling, step 1 (every TP rank, its logits shard [B, V] at columns
// id_off ..): the shard's top-128 (value, global id) pairs per row, sorted, into
// cand_v / cand_id [B][128].  The global top-k (k <= 128, the sampler's cap) of a row is
// contained in the union of the shards' sets, ties included (lowest ids first).
P2P_API int p2p_topk_candidates(const float* logits, int ld, int B, int V, int id_off,
                                float* cand_v, int* cand_id, unsigned* ws, hipStream_t st) {
  if (B <= 0 || V <= 0 || ld < V || !cand_v || !cand_id) return (int)hipErrorInvalidValue;
  int ng = 0;
  const int e = row_groups(logits, ld, B, V, nullptr, ws, &ng, st);
  if (e) return e;
  Src src{logits, nullptr, ld, 0, 0, id_off};
  hipLaunchKernelGGL(sample_kernel, dim3(B), dim3(THREADS), 0, st, src, V, (const float*)nullptr,
                     (const int*)nullptr, (const float*)nullptr,
                     (const unsigned long long*)nullptr, (const int*)nullptr, (int*)nullptr,
                     cand_v, cand_id, ng ? ws : (const unsigned*)nullptr, ng);
  return (int)hipGetLastError();
}

// Step 2 (after the all-gather of every rank's candidates, rank-major [W][B][128]):
// the same draw as p2p_sample over the full vocabulary row -- identical token for
// the same (seed, position), since only ids in the union can be drawn.
P2P_API int p2p_sample_candidates(const float* cand_v, const int* cand_id, int W, int B,
                                  const float* temp, const int* topk, const float* topp,
                                  const unsigned long long* seeds, const int* pos, int* ids,
                                  hipStream_t st) {
  if (B <= 0 || W <= 0) return (int)hipErrorInvalidValue;
  Src src{cand_v, cand_id, 0, KMAX, (long long)B * KMAX, 0};
  hipLaunchKernelGGL(sample_kernel, dim3(B), dim3(THREADS), 0, st, src, W * KMAX, temp, topk,
                     topp, seeds, pos, ids, (float*)nullptr, (int*)nullptr, (const unsigned*)nullptr, 0);
  return (int)hipGetLastError();
}
