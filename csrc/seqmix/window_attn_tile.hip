// Grouped-query window attention for prompts: the same inputs, options and outputs as
// window_attn_mfma_k (bf16 activations, fp32 scores / softmax / sums), with key tiles that four
// wavefronts share.
//
// window_attn_mfma_k gives every wavefront its own 16 (row, head) pairs and its own walk over the
// keys: a key tile is loaded from the cache once per 16 pairs, by the wavefront that waits for it.
// Here a workgroup owns 64 pairs of one key/value head -- 64 / HS consecutive rows x HS head slots,
// 16 pairs per wavefront -- and walks the union of their windows KT keys at a time; the tile's keys
// and values come through LDS (attn_tile.h), copied while the tile before is used, so a key row
// is read once per 64 pairs and the wait for it is hidden by the products and the other workgroups
// of the CU.  Per tile and wavefront:
//   S^T[KT keys x 16 pairs] = K . Q^T     (K rows from LDS, Q in registers)
//   online softmax in the accumulator layout; tiles in which no pair's maximum moves need no exchange between lanes
//   and no rescaling.  The largest weight is one, which bf16 holds exactly, and the sum is that of the rounded weights:
//   with a maximum that lagged by up to 2^8 and the sum of the unrounded ones, results were up to 18 % further off a
//   64-bit run than window_attn_mfma_k's where few keys dominate (scores of deviation 3.4: 1.96e-3 against 1.74e-3, now
//   1.72e-3; 2048 rows 48 -> 56 us)
//   O[16 pairs x V] += P . V              (V read transposed from the same row-major tile)
//
// All operands of a product are read before it starts (two wavefronts per SIMD leave the registers for
// it), the values while the weights are formed.
//
// What bounds it: with plain scores the LDS reads (a wavefront reads the whole tile for 16 pairs) and
// the copies, then the exponentials; with capped and penalised scores the exponentials and logarithms.
// 2048 rows, 16 heads on 4, D = V = 128: 56 us (300 TFLOP/s) against 276 us for window_attn_mfma_k; a window of 256 20
// against 58; 32 heads on 8, D = V = 64: 62 against 264.  (Such windows alone are prompt_attn_k's now, 42 us; blocks, kept
// tokens, two maps and other sizes are this kernel's.)
//
// Grid: one dimension, (row group, key/value head, head block) with the last row groups first (they
// see the most keys), key/value heads innermost so that an XCD's workgroups share few heads; y:
// runs of a window that is cut (portions of few rows far into a sequence), merged by the kernels
// of window_attn_mfma.hip.  Pages are a multiple of KT tokens.
#include "attn_tile.h"
#include "window_attn.h"
using namespace sm;

#define LOG2E_ 1.4426950408889634f
#define NO_KEY_YET -1e30f   // running maximum of a pair that has seen no key

template <int NK, int NV2, int KEYS, int MAPS, int KT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MAPS * (NK + NV2) < 32 ? 2 : 1, MAPS * (NK + NV2) < 32 ? 2 : 1)))
window_attn_tile_k(WindowArgs a) {
  constexpr bool BLK = KEYS == KEYS_BLOCKS, KEPT = KEYS == KEYS_KEPT;
  constexpr int DP = NK * 32, VP = NV2 * 32, NT = NV2 * 2, NS = KT / 16;
  constexpr int PK = MAPS * DP / 8, PV = VP / 8;          // 16-byte pieces per key and value row
  constexpr int MK = PK < 16 ? PK - 1 : 15, MV = PV < 16 ? PV - 1 : 15;
  constexpr int STAGE = KT * (PK + PV) * 8;               // bf16 per stage
  extern __shared__ __align__(16) unsigned short lds[];   // [2][KT keys | KT values]
  __shared__ int srow[2][BLK ? KT : 1];                   // pool rows of a tile of blocks
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), n16 = lane & 15, quad = lane >> 4;
  const int HG = a.H / a.G, hblocks = (HG + a.HS - 1) / a.HS, gh = a.G * hblocks;
  const int at = folded_block(), unit = a.U - 1 - at / gh, gb = at % gh;
  const int r0 = a.units[2 * unit], nr = a.units[2 * unit + 1];
  const int g = gb / hblocks, hb0 = (gb % hblocks) * a.HS;
  const int D = a.D, V = a.V, page = a.page, win = a.win;
  const int ldpool = a.G * (MAPS * D + V);
  const int koff = g * MAPS * D, voff = a.G * MAPS * D + g * V;
  // this lane's pair (as a column of S^T and a row of P)
  const int prow = (wave * 16 + n16) / a.HS, phs = hb0 + n16 % a.HS;
  const bool pvalid = prow < nr && phs < HG;
  const int ph = g * HG + min(phs, HG - 1);
  const int ppos = pvalid ? a.pos[r0 + prow] : -1;
  const bool wlive = (wave * 16) / a.HS < nr;             // this wavefront has rows
  const int* pages = a.bt + (size_t)a.row_ent[r0] * a.max_pages;
  const int p_lo = a.pos[r0], p_hi = a.pos[r0 + nr - 1];
  // Tiles: `heads` tiles of what stands before the windows -- blocks 0 .. nb-1, or the kept tokens 0 ..
  // nb-1 -- then the tokens of the windows from a multiple of KT on, so that a tile of tokens lies in one page.
  const int w_lo = max(0, p_lo - win + 1);
  int nb = 0, pnb = 0, SB = 1;
  if constexpr (BLK) {
    nb = max(0, p_hi - win + 1) / a.P;
    pnb = pvalid ? max(0, ppos - win + 1) / a.P : 0;      // blocks this lane's row sees
    SB = (page + a.P - 1) / a.P;
  }
  if constexpr (KEPT) nb = min(a.keep, w_lo);
  const int heads = (nb + KT - 1) / KT, t_lo = w_lo / KT;
  int i_lo = 0, i_hi = heads + p_hi / KT - t_lo;          // first and last tile
  if (a.splits > 1) {                                     // this workgroup's run of them
    const int per = (i_hi + a.splits) / a.splits;
    i_lo = blockIdx.y * per;
    i_hi = min(i_hi, i_lo + per - 1);
  }
  // first place of a tile: block or token number
  auto place = [&](int i) { return ((BLK || KEPT) && i < heads ? i : i - heads + t_lo) * KT; };
  auto block_row = [&](int j) {                           // of the pool of blocks; past the last: the last
    const int t = min(j, nb - 1) * a.P + a.P - 1;
    return pages[t / page] * SB + (t % page) / a.P;
  };

  // Copies of a tile: thread t takes 16-byte pieces t, t + 256, .. of its rows, as long as there are any (32 rows of
  // four pieces are two wavefronts' work).  Channels beyond D and V (which meet zero queries, or columns that
  // are not written) are some channels of the same row.
  constexpr int CK = (KT * PK + 255) / 256, CV = (KT * PV + 255) / 256;
  static_assert(KT * PK % 64 == 0 && KT * PV % 64 == 0, "a copy is a whole wavefront's");
  auto mine = [&](int c, int pieces) { return pieces % 256 == 0 || c * 256 + wave * 64 < pieces; };
  int ok_[CK], ov_[CV];                                   // byte offsets within a page's rows
#pragma unroll
  for (int i = 0; i < CK; i++) {
    const int p = i * 256 + tid, r = p / PK, lc = (p % PK) ^ swz(r, MK);
    const int u = lc / (DP / 8), c8 = (lc % (DP / 8)) * 8;
    ok_[i] = (r * ldpool + koff + u * D + (c8 < D ? c8 : 0)) * 2;
  }
#pragma unroll
  for (int i = 0; i < CV; i++) {
    const int p = i * 256 + tid, r = p / PV, c8 = ((p % PV) ^ swz(r, MV)) * 8;
    ov_[i] = (r * ldpool + voff + (c8 < V ? c8 : 0)) * 2;
  }
  const unsigned lds0 = lds_address(lds);
  auto copy_tile = [&](int i, int st, int row0) {         // row0: the pool row of a tile of tokens
    const unsigned base = lds0 + st * STAGE * 2 + wave * 1024, vbase = base + KT * PK * 16;
    if (BLK && i < heads) {
#pragma unroll
      for (int c = 0; c < CK; c++) {
        if (!mine(c, KT * PK)) continue;
        const int r = (c * 256 + tid) / PK;
        copy_lds16((const char*)a.blk + ((size_t)srow[st][r] - r) * ldpool * 2 + ok_[c],
                   base + c * 4096);
      }
#pragma unroll
      for (int c = 0; c < CV; c++) {
        if (!mine(c, KT * PV)) continue;
        const int r = (c * 256 + tid) / PV;
        copy_lds16((const char*)a.blk + ((size_t)srow[st][r] - r) * ldpool * 2 + ov_[c],
                   vbase + c * 4096);
      }
      return;
    }
    const char* src = (const char*)a.pool + (size_t)row0 * ldpool * 2;
    // a tile that reaches over the windows' ends takes their last (first) row again there: what else
    // the page holds (an earlier owner's tokens) meets weights of zero, but must not be infinite
    const int j0 = place(i), lo = KEPT && i < heads ? 0 : w_lo - j0, hi = (KEPT && i < heads ? nb - 1 : p_hi) - j0;
    if (lo > 0 || hi < KT - 1) {
#pragma unroll
      for (int c = 0; c < CK; c++) {
        if (!mine(c, KT * PK)) continue;
        const int r = (c * 256 + tid) / PK;
        copy_lds16_at(src, ok_[c] + (min(max(r, lo), hi) - r) * ldpool * 2, base + c * 4096);
      }
#pragma unroll
      for (int c = 0; c < CV; c++) {
        if (!mine(c, KT * PV)) continue;
        const int r = (c * 256 + tid) / PV;
        copy_lds16_at(src, ov_[c] + (min(max(r, lo), hi) - r) * ldpool * 2,
                      vbase + c * 4096);
      }
      return;
    }
#pragma unroll
    for (int c = 0; c < CK; c++)
      if (mine(c, KT * PK)) copy_lds16_at(src, ok_[c], base + c * 4096);
#pragma unroll
    for (int c = 0; c < CV; c++)
      if (mine(c, KT * PV)) copy_lds16_at(src, ov_[c], vbase + c * 4096);
  };
  auto token_page = [&](int i) { return BLK && i < heads ? 0 : pages[place(i) / page]; };
  auto token_row = [&](int i, int pg) {                   // the pool row of a tile's first token
    return __builtin_amdgcn_readfirstlane(pg) * page + place(i) % page;
  };

  // queries in registers (zero rows for unused pairs, zero columns beyond D)
  bf16x8 qf[MAPS][NK];
#pragma unroll
  for (int u = 0; u < MAPS; u++)
#pragma unroll
    for (int kk = 0; kk < NK; kk++) {
      const int c8 = kk * 32 + quad * 8;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (pvalid && c8 < D) v = *(const uint4*)(a.q + (size_t)(r0 + prow) * a.ldq + (size_t)(ph * MAPS + u) * D + c8);
      qf[u][kk] = __builtin_bit_cast(bf16x8, v);
    }
  // a score in powers of two: scale log2(e) s, or capped cap log2(e) tanh(scale s / cap), with tanh(x) =
  // 1 - 2 / (e^2x + 1) on the hardware's units (inf for large x -> 1, 0 for small -> -1)
  const float sl2 = a.scale * LOG2E_;
  const float cap2 = a.cap * LOG2E_, capx = a.cap > 0.0f ? 2.0f * sl2 / a.cap : 0.0f;
  const float pr1 = (pvalid && a.r1) ? a.r1[ph] : 0.0f, pr2 = (pvalid && a.r1) ? a.r2[ph] : 0.0f;
  float m_run[MAPS], l_part[MAPS];                // maxima in powers of two
  f32x4 acc[MAPS][NT];
#pragma unroll
  for (int u = 0; u < MAPS; u++) {
    m_run[u] = pvalid ? NO_KEY_YET : 0.0f;
    l_part[u] = 0.0f;
#pragma unroll
    for (int t = 0; t < NT; t++) acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  int next_page = 0;
  if (i_lo <= i_hi) {
    if constexpr (BLK) {
      if (tid < KT && i_lo < heads) {
        srow[0][tid] = block_row(place(i_lo) + tid);
        srow[1][tid] = block_row(place(i_lo + 1) + tid);
      }
      __syncthreads();
    }
    copy_tile(i_lo, 0, token_row(i_lo, token_page(i_lo)));
    if (i_lo < i_hi) next_page = token_page(i_lo + 1);
  }

  int st = 0;
  for (int i = i_lo; i <= i_hi; i++, st ^= 1) {
    tile_wait();
    __syncthreads();   // the tile has landed, the other stage is free
    // (the page of the tile after that is looked up now and not touched before the next wait: its use
    // would wait for the copies too)
    if (i < i_hi) copy_tile(i + 1, st ^ 1, token_row(i + 1, next_page));
    int nrow = 0;
    if (i + 2 <= i_hi) {
      next_page = token_page(i + 2);
      if (BLK && i + 2 < heads && tid < KT) nrow = block_row(place(i + 2) + tid);
    }
    if (wlive) {
      const unsigned short* sK = lds + st * STAGE;
      const unsigned short* sV = sK + KT * PK * 8;
      const bool head = (BLK || KEPT) && i < heads;
      const int j0 = place(i);
      // some place of the tile is out of some row's sight (the same for the whole workgroup)
      const bool cut = head ? (BLK ? (j0 + KT) * a.P > p_lo - win + 1 : j0 + KT > nb)
                            : j0 + KT - 1 > p_lo || j0 <= p_hi - win;
      const int jl = j0 + quad * 4;                // this lane's places: jl + sub * 16 + i
      f32x8 pw[MAPS][NS / 2];
      bf16x8 pf[MAPS][NS / 2];
      bf16x8 vf[NT][NS / 2];
#pragma unroll
      for (int u = 0; u < MAPS; u++) {
        f32x4 s[NS];
        bf16x8 kf[NS][NK];   // all of the map's operands, so that the reads are in flight together
#pragma unroll
        for (int kk = 0; kk < NK; kk++)
#pragma unroll
          for (int sub = 0; sub < NS; sub++) {
            const int r = sub * 16 + n16, piece = (u * (DP / 8) + kk * 4 + quad) ^ swz(r, MK);
            kf[sub][kk] = __builtin_bit_cast(bf16x8, *(const uint4*)(sK + (r * PK + piece) * 8));
          }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int sub = 0; sub < NS; sub++) s[sub] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < NK; kk++)
#pragma unroll
          for (int sub = 0; sub < NS; sub++)
            s[sub] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[sub][kk], qf[u][kk], s[sub], 0, 0, 0);
        if (u == MAPS - 1) {   // the values are on their way while the weights are formed
#pragma unroll
          for (int t = 0; t < NT; t++)
#pragma unroll
            for (int hf = 0; hf < NS / 2; hf++) vf[t][hf] = read_keys_by_channel<PV>(sV, hf * 32, t * 16, lane);
          __builtin_amdgcn_sched_barrier(0);
        }
        // scores in powers of two, less the running maximum
        const bool fresh = m_run[u] == NO_KEY_YET;
        const float base = fresh ? 0.0f : m_run[u];
        if (a.cap > 0.0f) {
          const float top = cap2 - base;
#pragma unroll
          for (int sub = 0; sub < NS; sub++)
#pragma unroll
            for (int e = 0; e < 4; e++)
              s[sub][e] = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(exp2_(s[sub][e] * capx) + 1.0f), top);
        } else {
#pragma unroll
          for (int sub = 0; sub < NS; sub++)
#pragma unroll
            for (int e = 0; e < 4; e++) s[sub][e] = fmaf(s[sub][e], sl2, -base);
        }
        if (a.r1) {   // r1 ln(1 + r2 d) in powers of two; keys behind the row are struck out below
          const float x0 = fmaf(pr2, (float)(ppos - jl), 1.0f);
#pragma unroll
          for (int sub = 0; sub < NS; sub++)
#pragma unroll
            for (int e = 0; e < 4; e++)
              s[sub][e] = fmaf(-pr1, __builtin_amdgcn_logf(fmaf(pr2, -(float)(sub * 16 + e), x0)), s[sub][e]);
        }
        if (cut) {
          // visible places as a range [from, to) of this lane's, all others struck out
          int from = ppos - win + 1 - jl, to = ppos + 1 - jl;
          if (head) {
            from = 0;
            to = (BLK ? pnb : nb) - jl;
          }
#pragma unroll
          for (int sub = 0; sub < NS; sub++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
              const int k = sub * 16 + e;
              bool ok = k >= from && k < to;
              // a later row of the group: its window has passed kept tokens that the first row's had not
              if (KEPT && !head) ok = ok || (k < to && jl + k >= nb && jl + k < a.keep);
              if (!ok) s[sub][e] = -INFINITY;
            }
        }
        float tmax = -INFINITY;
#pragma unroll
        for (int sub = 0; sub < NS; sub++)
#pragma unroll
          for (int e = 0; e < 4; e++) tmax = fmaxf(tmax, s[sub][e]);
        if (__any(tmax > (fresh ? -INFINITY : 0.0f))) {
          tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
          tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
          const bool none = fresh && tmax == -INFINITY;
          const float up = none ? 0.0f : fresh ? tmax : fmaxf(tmax, 0.0f);
          const float alpha = fresh ? 1.0f : exp2_(-up);   // a fresh pair's sums are zero
          m_run[u] = none ? NO_KEY_YET : base + up;
          l_part[u] *= alpha;
#pragma unroll
          for (int sub = 0; sub < NS; sub++) s[sub] -= up;
          // the accumulators hold pairs quad * 4 + i: fetch their factors
          float al[4];
#pragma unroll
          for (int e = 0; e < 4; e++) al[e] = __shfl(alpha, quad * 4 + e, 64);
#pragma unroll
          for (int t = 0; t < NT; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[u][t][e] *= al[e];
        }
        float psum = 0.0f;   // of the weights as the product has them
#pragma unroll
        for (int sub = 0; sub < NS; sub++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            pw[u][sub >> 1][(sub & 1) * 4 + e] = exp2_(s[sub][e]);   // 0 for places out of sight
          }
#pragma unroll
        for (int hf = 0; hf < NS / 2; hf++) {
          pf[u][hf] = to_bf16(pw[u][hf]);
#pragma unroll
          for (int e = 0; e < 8; e++) psum += (float)pf[u][hf][e];
        }
        l_part[u] += psum;
      }
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int hf = 0; hf < NS / 2; hf++)
#pragma unroll
          for (int u = 0; u < MAPS; u++)
            acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[u][hf], vf[t][hf], acc[u][t], 0, 0, 0);
    }
    if (BLK && i + 2 < heads && i + 2 <= i_hi && tid < KT) srow[st][tid] = nrow;   // read after the next barrier
  }
  if (!wlive) return;
  float z = 0.0f;
#pragma unroll
  for (int u = 0; u < MAPS; u++)
#pragma unroll
    for (int t = 0; t < NT; t++) not_finite(acc[u][t], z);
  if (__builtin_expect(__any(z != z), 0)) {   // see not_finite()
#pragma unroll 1
    for (int m = wave * 16; m < wave * 16 + 16; m++) {
      const int row = r0 + m / a.HS, hs = hb0 + m % a.HS, h = g * HG + hs;
      if (m / a.HS >= nr || hs >= HG) continue;
      const int p = a.pos[row], blocks = BLK ? max(0, p - win + 1) / a.P : 0;
      PairSums<(VP + 63) / 64> sums[MAPS];
#pragma unroll
      for (int u = 0; u < MAPS; u++) sums[u].begin(a.sink ? a.sink[h] : 0.0f, MAPS == 1 && a.sink && blockIdx.y == 0);
#pragma unroll 1
      for (int x = i_lo * KT; x < (i_hi + 1) * KT; x++) {
        const int i = x / KT, j = place(i) + x % KT;
        const bool head = (BLK || KEPT) && i < heads;
        if (!(head ? j < (BLK ? blocks : nb) : j <= p && (j > p - win || (KEPT && j >= nb && j < a.keep)))) continue;
        const bf16* kr = BLK && head ? a.blk + (size_t)block_row(j) * ldpool
                                     : a.pool + ((size_t)pages[j / page] * page + j % page) * ldpool;
#pragma unroll
        for (int u = 0; u < MAPS; u++) {
          float s = wave_dot(a.q + (size_t)row * a.ldq + (size_t)(h * MAPS + u) * D, kr + koff + u * D, D) * a.scale;
          if (a.cap > 0.0f) s = a.cap * tanhf(s / a.cap);
          if (a.r1) s -= a.r1[h] * log1pf(a.r2[h] * (float)(p - j));
          sums[u].add(s, kr + voff, V);
        }
      }
      if (a.splits > 1) {
        float* rec = a.part + (((size_t)unit * gh + gb) * a.splits + blockIdx.y) * MAPS * 64 * (VP + 2) + m * (VP + 2);
#pragma unroll
        for (int u = 0; u < MAPS; u++, rec += 64 * (VP + 2)) {
#pragma unroll
          for (int t = 0; t < (VP + 63) / 64; t++)
            if (t * 64 + lane < V) rec[t * 64 + lane] = sums[u].o[t];
          if (lane == 0) rec[VP] = sums[u].m, rec[VP + 1] = sums[u].l;
        }
        continue;
      }
      float ss = 0.0f, f = sums[0].l != 0.0f ? 1.0f / sums[0].l : 0.0f;
      if constexpr (MAPS == 2) {
        const float f1 = sums[1].l != 0.0f ? a.lam / sums[1].l : 0.0f;
#pragma unroll
        for (int t = 0; t < (VP + 63) / 64; t++) {
          sums[0].o[t] = sums[0].o[t] * f - sums[1].o[t] * f1;
          ss += sums[0].o[t] * sums[0].o[t];
        }
        f = 1.0f / sqrtf(wave_sum(ss) / (float)V + a.eps);
      }
      f *= a.out_scale;
      const bf16* gr = a.gate + (size_t)row * a.ldg + (size_t)h * (a.gate_pc ? V : 1);
#pragma unroll
      for (int t = 0; t < (VP + 63) / 64; t++) {
        const int c = t * 64 + lane;
        if (c >= V) continue;
        const float gv = a.gate ? sigmoidf_(__bfloat162float(gr[a.gate_pc ? c : 0])) : 1.0f;
        a.out[(size_t)row * a.ldo + (size_t)h * V + c] = __float2bfloat16(sums[0].o[t] * f * gv);
      }
    }
    return;
  }
  float l[MAPS];
#pragma unroll
  for (int u = 0; u < MAPS; u++) {
    l[u] = l_part[u] + __shfl_xor(l_part[u], 16, 64);
    l[u] += __shfl_xor(l[u], 32, 64);
    m_run[u] *= 1.0f / LOG2E_;   // natural from here on
  }
  // The sink joins the finished sums (of the first run of a window that is cut).  Scores are taken less the running
  // maximum before it moves: one that began with a sink far below them would swallow their low bits.
  float sf = 1.0f;               // rescales the sums of this lane's pair
  int pair = lane & 15;
  again(pair);                   // (its row and head are not kept in registers until here)
  if (MAPS == 1 && a.sink && blockIdx.y == 0 && (wave * 16 + pair) / a.HS < nr && hb0 + pair % a.HS < HG) {
    const float sink = a.sink[g * HG + hb0 + pair % a.HS], m = fmaxf(m_run[0], sink);
    sf = expf(m_run[0] - m);
    l[0] = l[0] * sf + expf(sink - m);
    m_run[0] = m;
  }
  if (a.splits > 1) {
    // partial record of this run: [map][64 pairs][VP + 2] = unnormalised sums, running max (natural), sum
    float* rec = a.part + (((size_t)unit * gh + gb) * a.splits + blockIdx.y) * MAPS * 64 * (VP + 2) +
                 (size_t)wave * 16 * (VP + 2);
#pragma unroll
    for (int u = 0; u < MAPS; u++, rec += 64 * (VP + 2)) {
      if (quad == 0) {
        rec[n16 * (VP + 2) + VP] = m_run[u];
        rec[n16 * (VP + 2) + VP + 1] = l[u];
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float f = MAPS == 1 ? __shfl(sf, quad * 4 + i, 64) : 1.0f;
#pragma unroll
        for (int t = 0; t < NT; t++) rec[(quad * 4 + i) * (VP + 2) + t * 16 + n16] = acc[u][t][i] * f;
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int m = wave * 16 + quad * 4 + i, mr = m / a.HS, ms = hb0 + m % a.HS;
    const float l0 = __shfl(l[0], quad * 4 + i, 64);
    const float i0 = l0 != 0.0f ? (MAPS == 1 ? __shfl(sf, quad * 4 + i, 64) : 1.0f) / l0 : 0.0f;
    if constexpr (MAPS == 2) {
      const float l1 = __shfl(l[1], quad * 4 + i, 64);
      const float i1 = l1 > 0.0f ? a.lam / l1 : 0.0f;
      float ss = 0.0f;
#pragma unroll
      for (int t = 0; t < NT; t++) {   // columns beyond V hold what the clamped channels gave
        const float o = t * 16 + n16 < V ? acc[0][t][i] * i0 - acc[1][t][i] * i1 : 0.0f;
        acc[0][t][i] = o;
        ss += o * o;
      }
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);   // the pair's 16 lanes
      const float rs = a.out_scale / sqrtf(ss / (float)V + a.eps);
      if (mr < nr && ms < HG) {
        bf16* o = a.out + (size_t)(r0 + mr) * a.ldo + (size_t)(g * HG + ms) * V;
#pragma unroll
        for (int t = 0; t < NT; t++)
          if (t * 16 + n16 < V) o[t * 16 + n16] = __float2bfloat16(acc[0][t][i] * rs);
      }
    } else if (mr < nr && ms < HG) {
      bf16* o = a.out + (size_t)(r0 + mr) * a.ldo + (size_t)(g * HG + ms) * V;
      float gv = i0 * a.out_scale;
      const bf16* gr = a.gate + (size_t)(r0 + mr) * a.ldg + (size_t)(g * HG + ms) * (a.gate_pc ? V : 1);
      if (a.gate && !a.gate_pc) gv *= sigmoidf_(__bfloat162float(*gr));
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const int c = t * 16 + n16;
        if (c < V) {
          float v = acc[0][t][i] * gv;
          if (a.gate && a.gate_pc) v *= sigmoidf_(__bfloat162float(gr[c]));
          o[c] = __float2bfloat16(v);
        }
      }
    }
  }
}

template <int NK, int NV2, int KEYS, int MAPS>
static int launch_tile(const WindowArgs& a, hipStream_t st) {
  // 64 keys per tile while two stages leave room for two workgroups per CU, else 32
  // (window_attn_tile() has checked that pages are a multiple of 64 tokens)
  constexpr int KT = (MAPS * NK + NV2) * 32 * 2 * 64 * 2 <= 64 * 1024 ? 64 : 32;
  const int HG = a.H / a.G, hblocks = (HG + a.HS - 1) / a.HS;
  const size_t shm = (size_t)2 * KT * (MAPS * NK + NV2) * 32 * 2;
  if (shm > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)window_attn_tile_k<NK, NV2, KEYS, MAPS, KT>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL((window_attn_tile_k<NK, NV2, KEYS, MAPS, KT>), dim3(a.U * a.G * hblocks, a.splits),
                     dim3(256), shm, st, a);
  return (int)hipGetLastError();
}

template <int NK, int NV2>
static int launch_keys(const WindowArgs& a, int maps, hipStream_t st) {
  if (maps == 2) return launch_tile<NK, NV2, KEYS_KEPT, 2>(a, st);
  if (a.blk) return launch_tile<NK, NV2, KEYS_BLOCKS, 1>(a, st);
  if (a.keep) return launch_tile<NK, NV2, KEYS_KEPT, 1>(a, st);
  // windows alone, with keys and values of 33 to 128 numbers: prompt_attn.hip (its figures)
  if constexpr (NK >= 2 && NK <= 4 && NV2 >= 2 && NV2 <= 4) return prompt_attn_paged(a, st);
  else return launch_tile<NK, NV2, KEYS_WINDOW, 1>(a, st);
}

template <int NK>
static int launch_values(const WindowArgs& a, int maps, hipStream_t st) {
  switch (window_pad32(a.V)) {
    case 1: return launch_keys<NK, 1>(a, maps, st);
    case 2: return launch_keys<NK, 2>(a, maps, st);
    case 4: return launch_keys<NK, 4>(a, maps, st);
    default: return launch_keys<NK, 8>(a, maps, st);
  }
}

int window_attn_tile(const WindowArgs& a, int maps, hipStream_t st) {
  if (a.page < 64 || a.page % 64) return (int)hipErrorInvalidValue;
  switch (window_pad32(a.D)) {
    case 1: return launch_values<1>(a, maps, st);
    case 2: return launch_values<2>(a, maps, st);
    case 4: return launch_values<4>(a, maps, st);
    default: return launch_values<8>(a, maps, st);
  }
}
