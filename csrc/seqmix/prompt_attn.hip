// Attention of prompts on wavefronts of 32 (row, head) pairs: bf16 activations, fp32 scores, softmax and sums.
//
// Two sources of keys and values:
//   PAGED   the paged pool of window_attn_tile_k, whose inputs, options and outputs these are (a window of tokens, one map;
//           blocks, kept tokens, two maps and other sizes stay there)
//   FORMED  keys and values that a layer of cached latents formed for this step (kv, one row per token, all heads' keys and then
//           their values), beside a rotated key part that all heads share and the pool holds (RP channels).  Prompts take
//           this form: a pair meets D + Rd + V numbers of a key instead of twice the latent (16 heads of 128 + 64, latents of 448:
//           320 for 960), for one product that forms each key once.
//
// A workgroup owns 64 pairs of one key/value head (64 / HS consecutive rows x HS head slots) and walks the union of their
// windows 64 keys at a time; a tile is copied to LDS while the one before is used (attn_tile.h).  Its four wavefronts are 2
// halves of the pairs x 2 halves of a tile's keys, each with a maximum, sums and weights of its own that meet at the end.
//   S^T[32 keys x 32 pairs] = K . Q^T           (v_mfma_f32_32x32x16_bf16; K rows from LDS, Q in registers)
//   online softmax, one pair per lane (two lanes share a pair): the largest weight is one and the sum is that of the rounded
//   weights, as in window_attn_tile_k
//   O^T[V x 32 pairs] += V^T . P^T              (V read transposed from the row-major tile; P in registers as S^T left it)
// A lane keeps to one pair throughout, so factors need no exchange.
//
// Why 32 x 32: a tile's reads from LDS serve 32 pairs.  With 16 x 16 x 32 products they serve 16, and LDS, which gives 128 bytes a
// cycle, is busy for twice the time that the products take.  Why the keys are cut: two wavefronts per SIMD without reading a
// tile more often.
//
// What bounds it: a tile's chain (copy, 12 + 8 products, 16 scores per lane), about 1 us of which a third is the matrix cores,
// through the longest window's tiles; wavefronts issue some 400 instructions a tile.  128 pairs with eight wavefronts (57 us
// where this takes 48), with their halves out of step (59), and the next tile's first product under this one's exponentials (55)
// gave nothing: the wavefronts' issue is what is full.
// 2048 rows, us: FORMED, 16 heads of 128 + 64 and 128, 48 where latent_attn_tile_k takes 150; PAGED, 16 heads of 128 on 4, 42
// (window_attn_tile_k 53), capped and penalised 56 (65), 16 heads of 64 28 (38); 1201 + 361 + 841 rows 30 (36), 38 (44), 20 (27).
#include <type_traits>

#include "attn_tile.h"
#include "window_attn.h"
using namespace sm;

#define LOG2E_ 1.4426950408889634f
#define NO_KEY_YET -1e30f   // running maximum of a pair that has seen no key

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// What place of a row holds piece p: p ^ this.  Keys are read 16 rows x one piece, values 4 rows x 4 pieces: 16 places of 16
// bytes are all the banks.
template <int PIECES>
__device__ __forceinline__ int key_swz(int r) { return PIECES == 8 ? (r >> 1) & 7 : r & 15; }
template <int PIECES>
__device__ __forceinline__ int value_swz(int r) {
  return PIECES == 8 ? ((r >> 1) & 1) << 2 | ((r >> 2) & 3) : (r & 3) << 2 | ((r >> 2) & 3);
}

// four numbers to neighbouring channels
__device__ __forceinline__ void store4(bf16* o, const float* v, bool whole) {
  if (whole) {
    bf16 b[4];
#pragma unroll
    for (int j = 0; j < 4; j++) b[j] = __float2bfloat16(v[j]);
    *(uint2*)o = __builtin_bit_cast(uint2, b);
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++) o[j] = __float2bfloat16(v[j]);
  }
}

template <int DP, int RP, int VP, bool FORMED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) prompt_attn_k(PromptArgs p) {
  const WindowArgs& a = p.w;
  constexpr int KT = 64, PK = DP / 8, PR = RP / 8, PV = VP / 8, NK = DP / 16, NR = RP / 16, NC = VP / 32, NQ = NK + NR;
  constexpr int KB = KT * PK * 16, RB = KT * PR * 16, STAGE = KB + RB + KT * PV * 16;   // bytes
  static_assert(2 * STAGE >= 64 * VP * 2 + 256 * 12, "what the halves of the keys exchange");
  static_assert(PV == 8 || PV == 16, "eight keys on, a value's piece moves by 2 places");
  // (what only the paged form has)
  const bool capped = !FORMED && a.cap > 0.0f, fading = !FORMED && a.r1, cut = !FORMED && a.splits > 1;
  extern __shared__ __align__(16) char lds[];   // [2][keys | rotated parts | values]
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), n32 = lane & 31, hi = lane >> 5;
  const int rh = wave & 1, kh = wave >> 1;      // half of the pairs, half of a tile's keys
  const int HG = a.H / a.G, hblocks = (HG + a.HS - 1) / a.HS, gh = a.G * hblocks;
  const int at = folded_block(), unit = a.U - 1 - at / gh, gb = at % gh;
  const int r0 = a.units[2 * unit], nr = a.units[2 * unit + 1];
  const int g = gb / hblocks, hb0 = (gb % hblocks) * a.HS;
  const int D = a.D, V = a.V, page = a.page, win = a.win;
  const int ldkv = FORMED ? p.ldkv : a.G * (D + V), koff = g * D, voff = a.G * D + g * V;
  // this lane's pair (HS is a power of two)
  const int hs_bits = __builtin_ctz(a.HS);
  auto row_of = [&](int n) { return (rh * 32 + n) >> hs_bits; };
  auto slot_of = [&](int n) { return hb0 + (n & (a.HS - 1)); };
  const int prow = row_of(n32), ph = g * HG + min(slot_of(n32), HG - 1);
  const bool pvalid = prow < nr && slot_of(n32) < HG;
  const int ppos = pvalid ? a.pos[r0 + prow] : -1;
  const int first = row_of(0), last = min(nr, row_of(31) + 1) - 1;   // this wavefront's rows
  const bool wlive = first < nr;
  const int ent = a.row_ent[r0];
  const int* pages = a.bt + (size_t)ent * a.max_pages;
  const int p_lo = a.pos[r0], p_hi = p_lo + nr - 1, w_lo = max(0, p_lo - win + 1);
  const int q_lo = p_lo + first, q_hi = p_lo + last;   // positions of this wavefront's rows
  const int t_lo = w_lo / KT;
  int i_lo = 0, i_hi = p_hi / KT - t_lo;
  if (cut) {                                     // this workgroup's run of tiles
    const int per = (i_hi + a.splits) / a.splits;
    i_lo = blockIdx.y * per;
    i_hi = min(i_hi, i_lo + per - 1);
  }
  const long kbase = FORMED ? p.kbase[(size_t)ent * p.kstride] : 0;   // key j is row kbase + j of kv

  // Copies of a tile: thread t takes 16-byte pieces t, t + 256, .. of its keys, rotated parts and values.  Channels beyond D,
  // Rd and V (which meet zero queries, or are not written) are some channels of the same row.  A tile that reaches over the
  // windows' ends takes their last (first) row again there: what else stands there (an earlier owner's tokens, another
  // prompt's) meets weights of zero, but must not be infinite.
  const unsigned lds0 = lds_address(lds) + wave * 1024;
  constexpr bool PAGES = !FORMED || RP > 0;
  // (a tile lies in one page; tiles are walked in order, so the page's number and the place in it are counted, not divided)
  int pi = (t_lo + i_lo) * KT / page, po = (t_lo + i_lo) * KT % page;
  auto look_up = [&]() {                         // the row of the pool that the next tile begins with, as page and place
    const int2 at_ = make_int2(PAGES ? pages[pi] : 0, po);
    po += KT;
    if (po == page) po = 0, pi++;
    return at_;
  };
  const char* kv0 = FORMED ? (const char*)(p.kv + kbase * ldkv) : (const char*)a.pool;
  const int ld2 = ldkv * 2, ldr2 = p.ldr * 2;
  // lanes' offsets in a tile whose rows are all in sight: of the first copy, and from one to the next
  const int rk = tid / PK, ck = ((tid % PK) ^ key_swz<PK>(rk)) * 8, kcol = (koff + (ck < D ? ck : 0)) * 2, at_k = rk * ld2 + kcol;
  const int rv = tid / PV, cv = ((tid % PV) ^ value_swz<PV>(rv)) * 8, vcol = (voff + (cv < V ? cv : 0)) * 2, at_v = rv * ld2 + vcol;
  const int rr = RP ? tid / max(PR, 1) : 0, cr = RP ? ((tid % max(PR, 1)) ^ key_swz<8>(rr)) * 8 : 0;
  const int rcol = (cr < p.Rd ? cr : 0) * 2, at_r = rr * ldr2 + rcol;
  auto copy_rows = [&](auto pieces, auto on, const char* src, unsigned dst, auto&& at) {
    constexpr int N = KT * pieces / 256, ON = on;
    static_assert(N == 2 || N == 4, "8 or 16 pieces");
    copy_lds16_on<ON>(src, at(0), dst);
    copy_lds16_on<ON + 4096>(src, at(1), dst);
    if constexpr (N > 2) {
      copy_lds16_on<ON + 8192>(src, at(2), dst);
      copy_lds16_on<ON + 12288>(src, at(3), dst);
    }
  };
  auto copy_tile = [&](int i, int st, int2 where) {
    const int j0 = (t_lo + i) * KT;
    const unsigned dst = lds0 + st * STAGE;
    const long prow = PAGES ? (long)uniform(where.x) * page + where.y : 0;
    const char* src = kv0 + (FORMED ? (long)j0 : prow) * ld2;
    const char* rot = (const char*)(a.pool + p.rot0) + prow * ldr2;
    constexpr std::integral_constant<int, PK> pk;
    constexpr std::integral_constant<int, PV> pv;
    constexpr std::integral_constant<int, RP ? PR : 8> pr;
    constexpr std::integral_constant<int, 0> on_k;
    constexpr std::integral_constant<int, KB> on_r;
    constexpr std::integral_constant<int, KB + RB> on_v;
    if (j0 >= w_lo && j0 + KT - 1 <= p_hi) {
      copy_rows(pk, on_k, src, dst, [&](int c) { return at_k + c * (256 / PK * ld2); });
      if constexpr (RP > 0) copy_rows(pr, on_r, rot, dst, [&](int c) { return at_r + c * (32 * ldr2); });
      copy_rows(pv, on_v, src, dst, [&](int c) { return at_v + c * (256 / PV * ld2); });
    } else {
      auto row = [&](int r) { return min(max(j0 + r, w_lo), p_hi) - j0; };
      copy_rows(pk, on_k, src, dst, [&](int c) { return row(rk + c * (256 / PK)) * ld2 + kcol; });
      if constexpr (RP > 0) copy_rows(pr, on_r, rot, dst, [&](int c) { return row(rr + c * 32) * ldr2 + rcol; });
      copy_rows(pv, on_v, src, dst, [&](int c) { return row(rv + c * (256 / PV)) * ld2 + vcol; });
    }
  };

  // queries in registers (zero for unused pairs and beyond D and Rd)
  bf16x8 qf[NQ];
#pragma unroll
  for (int kk = 0; kk < NQ; kk++) {
    const bool rot = kk >= NK;
    const int c8 = (rot ? kk - NK : kk) * 16 + hi * 8;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (pvalid && c8 < (rot ? p.Rd : D))
      v = rot ? *(const uint4*)(p.qrot + (size_t)(r0 + prow) * p.ldqr + (size_t)ph * p.Rd + c8)
              : *(const uint4*)(a.q + (size_t)(r0 + prow) * a.ldq + (size_t)ph * p.qhs + c8);
    qf[kk] = __builtin_bit_cast(bf16x8, v);
  }
  // a score in powers of two: scale log2(e) s, or capped (see window_attn_tile_k)
  const float sl2 = a.scale * LOG2E_;
  const float cap2 = a.cap * LOG2E_, capx = capped ? 2.0f * sl2 / a.cap : 0.0f;
  const float pr1 = (pvalid && fading) ? a.r1[ph] : 0.0f, pr2 = (pvalid && fading) ? a.r2[ph] : 0.0f;
  float m_run = pvalid ? NO_KEY_YET : 0.0f, l_part = 0.0f;   // maximum in powers of two
  const f32x16 zero = {};
  f32x16 acc[NC];
#pragma unroll
  for (int t = 0; t < NC; t++) acc[t] = zero;

  // LDS reads: this lane's row of keys, its rows and channels of values
  const int kr = kh * 32 + n32, k_at = kr * (PK * 16) + ((key_swz<PK>(kr) ^ hi) << 4);
  const int r_at = RP ? KB + kr * (PR * 16) + ((key_swz<8>(kr) ^ hi) << 4) : 0;
  const int vk = kh * 32 + hi * 4 + ((lane & 15) >> 2), vp = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
  const int v_at = KB + RB + vk * (PV * 16) + ((vp ^ value_swz<PV>(vk)) << 4) + (lane & 1) * 8;
#pragma unroll
  for (int kk = 0; kk < NQ; kk++) asm volatile("" : "+v"(qf[kk]));   // (waited for here and not in the loop)

  int2 next = make_int2(0, 0);
  if (i_lo <= i_hi) {
    copy_tile(i_lo, 0, look_up());
    if (i_lo < i_hi) next = look_up();
  }
  const int l0 = lds_address(lds);               // (a multiple of what is xored to addresses)
  for (int i = i_lo, st = 0; i <= i_hi; i++, st ^= 1) {
    tile_wait();
    __syncthreads();   // the tile has landed, the other stage is free
    // (a page is looked up a tile ahead, and used before the copies begin: the compiler waits for all that is under way where
    // it takes the number)
    next.x = uniform(next.x);
    if (i < i_hi) copy_tile(i + 1, st ^ 1, next);
    if (i + 2 <= i_hi) next = look_up();
    const int j0 = (t_lo + i) * KT + kh * 32;   // this wavefront's keys
    int kst = l0 + k_at + st * STAGE, rst = l0 + r_at + st * STAGE, vst = l0 + v_at + st * STAGE;
    again(kst);                                  // (a place for each read would take the registers of the sums)
    again(rst);
    again(vst);
    auto read_key = [&](int kk) {
      typedef __attribute__((address_space(3))) const bf16x8* lds_t;
      return *(lds_t)(kk < NK ? kst ^ (kk << 5) : rst ^ ((kk - NK) << 5));
    };
    // values v = h * NC + t: channels 32 t .., keys 16 h + 8 (e / 4) + 4 hi + e % 4 in slot e
    auto read_value = [&](int v) {
      typedef __attribute__((address_space(3))) s16x4* lds_t;
      s16x4 part[2];
#pragma unroll
      for (int e = 0; e < 2; e++)                // eight keys on: place ^ 2; sixteen: the same place
        part[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_t)((vst ^ ((v % NC * 4) << 4 ^ e << 5)) + (e * 8 + (v / NC) * 16) * (PV * 16)));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7));
    };
    f32x16 s;
    {
      bf16x8 kf[NQ];
#pragma unroll
      for (int kk = 0; kk < NQ; kk++) kf[kk] = read_key(kk);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < NQ; kk++) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kk], qf[kk], kk ? s : zero, 0, 0, 0);
    }
    // the values are on their way while the weights are formed
    bf16x8 vf[NC * 2];
#pragma unroll
    for (int v = 0; v < NC * 2; v++) vf[v] = read_value(v);
    __builtin_amdgcn_sched_barrier(0);
    // scores; plain ones are put into powers of two once the maximum is known
    float f = sl2;
    if (capped) {
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(exp2_(s[e] * capx) + 1.0f), cap2);
      f = 1.0f;
    } else if (!(sl2 > 0.0f)) {                  // (the maximum of the scores is that of the products only for scales above 0)
#pragma unroll
      for (int e = 0; e < 16; e++) s[e] *= sl2;
      f = 1.0f;
    }
    const int jl = j0 + hi * 4;                  // this lane's keys: jl + 8 (e / 4) + e % 4
    if (fading) {   // r1 ln(1 + r2 d) in powers of two; keys behind the row are struck out below
      const float x0 = fmaf(pr2, (float)(ppos - jl), 1.0f);
#pragma unroll
      for (int e = 0; e < 16; e++)
        s[e] = fmaf(-pr1, __builtin_amdgcn_logf(fmaf(pr2, -(float)((e >> 2) * 8 + (e & 3)), x0)), s[e] * f);
      f = 1.0f;
    }
    if (j0 + 31 > q_lo || j0 <= q_hi - win) {    // some key is out of some row's sight
      const int from = ppos - win + 1 - jl, to = ppos + 1 - jl;
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int k = (e >> 2) * 8 + (e & 3);
        if (k < from || k >= to) s[e] = -INFINITY;
      }
    }
    float tmax = -INFINITY;
#pragma unroll
    for (int e = 0; e < 16; e++) tmax = fmaxf(tmax, s[e]);
    tmax *= f;                                   // (f > 0)
    if (__any(tmax > m_run)) {
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float up = fmaxf(m_run, tmax), alpha = exp2_(m_run - up);   // (a fresh pair's sums are zero)
      m_run = up;
      l_part *= alpha;
#pragma unroll
      for (int t = 0; t < NC; t++) acc[t] *= alpha;
    }
    const float less = -m_run;
    bf16x8 pf[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
      f32x8 pw;
#pragma unroll
      for (int e = 0; e < 8; e++) pw[e] = exp2_(fmaf(s[h * 8 + e], f, less));   // 0 for keys out of sight
      pf[h] = to_bf16(pw);
      const bf16x2 one = {(__bf16)1.0f, (__bf16)1.0f};   // the sum of the weights as the product has them
      l_part = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[h], pf[h], 0, 1), one, l_part, false);
      l_part = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[h], pf[h], 2, 3), one, l_part, false);
      l_part = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[h], pf[h], 4, 5), one, l_part, false);
      l_part = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[h], pf[h], 6, 7), one, l_part, false);
#pragma unroll
      for (int t = 0; t < NC; t++) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[h * NC + t], pf[h], acc[t], 0, 0, 0);
    }
  }
  // The halves of the keys meet: each wavefront finishes half of the channels and hands the other half over, rescaled to the
  // common maximum.
  __syncthreads();   // the stages are free
  float* sx = (float*)lds;                       // what is handed over: [rh][number][lane]
  float* sm_ = sx + 2 * 64 * VP / 4;             // [wave][32] maxima
  float* sl = sm_ + 128;                         // [wave][32] sums
  int* sbad = (int*)(sl + 128);
  float l = l_part + __shfl_xor(l_part, 32, 64);
  if (hi == 0) sm_[wave * 32 + n32] = m_run, sl[wave * 32 + n32] = l;
  __syncthreads();
  const int other = wave ^ 2;
  const float mo = sm_[other * 32 + n32], m_all = fmaxf(m_run, mo), f_own = exp2_(m_run - m_all);
  l = l * f_own + sl[other * 32 + n32] * exp2_(mo - m_all);
#pragma unroll
  for (int t = 0; t < NC; t++) acc[t] *= f_own;
  constexpr int HC = NC / 2;
  f32x16 fin[HC];
#pragma unroll
  for (int half = 0; half < 2; half++) {         // channels of half `half` are finished by the wavefronts with kh == half
    __syncthreads();
    if (kh != half)
#pragma unroll
      for (int t = 0; t < HC; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) sx[((rh * HC + t) * 16 + e) * 64 + lane] = acc[half * HC + t][e];
    __syncthreads();
    if (kh == half)
#pragma unroll
      for (int t = 0; t < HC; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) fin[t][e] = acc[half * HC + t][e] + sx[((rh * HC + t) * 16 + e) * 64 + lane];
  }
  float z = 0.0f;
#pragma unroll
  for (int t = 0; t < HC; t++)
#pragma unroll
    for (int e = 0; e < 16; e++) z = fmaf(fin[t][e], 0.0f, z);
  const bool bad = __any(z != z);
  if (lane == 0) sbad[wave] = bad;
  __syncthreads();
  if (!wlive) return;
  if (__builtin_expect(uniform(sbad[wave] | sbad[other]), 0)) {   // see not_finite(); the pairs are shared by the two wavefronts
#pragma unroll 1
    for (int m = rh * 32 + kh * 16; m < rh * 32 + kh * 16 + 16; m++) {
      const int row = r0 + m / a.HS, hs = hb0 + m % a.HS, h = g * HG + hs;
      if (m / a.HS >= nr || hs >= HG) continue;
      const int pos = a.pos[row];
      PairSums<(VP + 63) / 64> sums;
      sums.begin(a.sink ? a.sink[h] : 0.0f, a.sink && blockIdx.y == 0);
#pragma unroll 1
      for (int j = max((t_lo + i_lo) * KT, max(0, pos - win + 1)); j <= min(pos, (t_lo + i_hi) * KT + KT - 1); j++) {
        const long prow0 = PAGES ? (long)pages[j / page] * page + j % page : 0;
        const bf16* kv = FORMED ? p.kv + (kbase + j) * ldkv : a.pool + prow0 * ldkv;
        float s = wave_dot(a.q + (size_t)row * a.ldq + (size_t)h * p.qhs, kv + koff, D);
        if (RP) s += wave_dot(p.qrot + (size_t)row * p.ldqr + (size_t)h * p.Rd, a.pool + prow0 * p.ldr + p.rot0, p.Rd);
        s *= a.scale;
        if (capped) s = a.cap * tanhf(s / a.cap);
        if (fading) s -= a.r1[h] * log1pf(a.r2[h] * (float)(pos - j));
        sums.add(s, kv + voff, V);
      }
      float* rec = a.part + (((size_t)unit * gh + gb) * a.splits + blockIdx.y) * PROMPT_PAIRS * (VP + 2) + m * (VP + 2);
      const float f = (sums.l != 0.0f ? 1.0f / sums.l : 0.0f) * a.out_scale;
      const bf16* gr = a.gate + (size_t)row * a.ldg + (size_t)h * (a.gate_pc ? V : 1);
#pragma unroll
      for (int t = 0; t < (VP + 63) / 64; t++) {
        const int c = t * 64 + lane;
        if (c >= V) continue;
        if (cut) {
          rec[c] = sums.o[t];
          continue;
        }
        const float gv = a.gate ? sigmoidf_(__bfloat162float(gr[a.gate_pc ? c : 0])) : 1.0f;
        a.out[(size_t)row * a.ldo + (size_t)h * V + c] = __float2bfloat16(sums.o[t] * f * gv);
      }
      if (cut && lane == 0) rec[VP] = sums.m, rec[VP + 1] = sums.l;
    }
    return;
  }
  int n = lane & 31;
  again(n);                                      // (the pair's row and head are not kept in registers until here)
  const int orow = row_of(n), oh = g * HG + slot_of(n);
  if (orow >= nr || slot_of(n) >= HG) return;
  float m_nat = m_all * (1.0f / LOG2E_), sf = 1.0f;   // natural from here on
  // the sink joins the finished sums (of the first run of a window that is cut), see window_attn_tile_k
  if (a.sink && blockIdx.y == 0) {
    const float sink = a.sink[oh], m = fmaxf(m_nat, sink);
    sf = expf(m_nat - m);
    l = l * sf + expf(sink - m);
    m_nat = m;
  }
  const int c0 = kh * (VP / 2) + hi * 4;         // this lane's channels: c0 + 32 t + 8 e4 + 0 .. 3
  if (cut) {
    // partial record of this run: [pairs][VP + 2] = unnormalised sums, running max (natural), sum
    float* rec = a.part + ((((size_t)unit * gh + gb) * a.splits + blockIdx.y) * PROMPT_PAIRS + rh * 32 + n) * (VP + 2);
    if (hi == 0 && kh == 0) rec[VP] = m_nat, rec[VP + 1] = l;
#pragma unroll
    for (int t = 0; t < HC; t++)
#pragma unroll
      for (int e = 0; e < 16; e++) rec[c0 + t * 32 + (e >> 2) * 8 + (e & 3)] = fin[t][e] * sf;
    return;
  }
  bf16* o = a.out + (size_t)(r0 + orow) * a.ldo + (size_t)oh * V;
  const bf16* gr = a.gate + (size_t)(r0 + orow) * a.ldg + (size_t)oh * (a.gate_pc ? V : 1);
  float f = (l != 0.0f ? sf / l : 0.0f) * a.out_scale;
  if (a.gate && !a.gate_pc) f *= sigmoidf_(__bfloat162float(*gr));
#pragma unroll
  for (int t = 0; t < HC; t++)
#pragma unroll
    for (int e4 = 0; e4 < 4; e4++) {
      const int c = c0 + t * 32 + e4 * 8;
      if (c >= V) continue;                      // (V is a multiple of eight)
      float v[4], gv[4] = {1.0f, 1.0f, 1.0f, 1.0f};
      if (a.gate && a.gate_pc) {
        if (p.gate_wide) ldv<4>(gr, c, gv);
        else
#pragma unroll
          for (int j = 0; j < 4; j++) gv[j] = __bfloat162float(gr[c + j]);
#pragma unroll
        for (int j = 0; j < 4; j++) gv[j] = sigmoidf_(gv[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = fin[t][e4 * 4 + j] * (f * gv[j]);
      store4(o + c, v, p.out_wide);
    }
}

template <int DP, int RP, int VP, bool FORMED>
static int launch_prompt(PromptArgs p, hipStream_t st) {
  const WindowArgs& a = p.w;
  p.gate_wide = a.gate && a.ldg % 4 == 0 && (uintptr_t)a.gate % 8 == 0;
  p.out_wide = a.ldo % 4 == 0 && (uintptr_t)a.out % 8 == 0;
  const int HG = a.H / a.G, hblocks = (HG + a.HS - 1) / a.HS;
  constexpr size_t shm = (size_t)2 * 64 * (DP + RP + VP) * 2;
  const auto k = prompt_attn_k<DP, RP, VP, FORMED>;
  if (const hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm))
    return (int)e;
  hipLaunchKernelGGL(k, dim3(a.U * a.G * hblocks, a.splits), dim3(256), shm, st, p);
  return (int)hipGetLastError();
}

template <int RP, bool FORMED>
static int launch_sizes(const PromptArgs& p, hipStream_t st) {
  const bool d = p.w.D > 64, v = p.w.V > 64;
  return d ? (v ? launch_prompt<128, RP, 128, FORMED>(p, st) : launch_prompt<128, RP, 64, FORMED>(p, st))
           : (v ? launch_prompt<64, RP, 128, FORMED>(p, st) : launch_prompt<64, RP, 64, FORMED>(p, st));
}

int prompt_attn_paged(const WindowArgs& w, hipStream_t st) {
  PromptArgs p = {};
  p.w = w;
  p.qhs = w.D;
  return launch_sizes<0, false>(p, st);
}

extern "C" {

// Keys and values formed for the step: kv [tokens, H * D keys | H * V values], key j of entry e at row kbase[e * kstride] + j;
// pool (with Rd > 0): rows of ldr numbers by page, the shared rotated key part at number rot0 of each.
int p2p_sm_formed_attn(const void* q, int ldq, int qhs, const void* qrot, int ldqr, const void* kv, int ldkv, const int* kbase, int kstride,
                       const void* pool, int ldr, int rot0, int Rd, const int* bt, int max_pages, const int* row_ent,
                       const int* pos, const int* units, int U, const float* sink, float scale, int win, void* out, int ldo,
                       int H, int D, int V, int page, float out_scale, const void* gate, int ldg, int gate_pc,
                       hipStream_t st) {
  if (U <= 0) return 0;
  if (H < 1 || D < 8 || D > 128 || D % 8 || V < 8 || V > 128 || V % 8 || Rd < 0 || Rd > 64 || Rd % 8 || win < 1 || ldq % 8 ||
      qhs % 8 || ldkv % 8 || (Rd && (ldqr % 8 || ldr % 8 || rot0 % 8 || page < 64 || page % 64)))
    return (int)hipErrorInvalidValue;
  PromptArgs p = {};
  p.w = {(const bf16*)q, ldq, (const bf16*)pool, bt, max_pages, row_ent, pos, units, U, sink, scale, win, (bf16*)out, ldo, H, H,
         D, V, page, 1, 1, nullptr, out_scale, 0.0f, nullptr, nullptr, (const bf16*)gate, ldg, gate_pc, nullptr, 1, 0, 0.0f, 0.0f};
  p.qhs = qhs;
  p.qrot = (const bf16*)qrot;
  p.ldqr = ldqr;
  p.kv = (const bf16*)kv;
  p.ldkv = ldkv;
  p.kbase = kbase;
  p.kstride = kstride;
  p.ldr = ldr;
  p.rot0 = rot0;
  p.Rd = Rd;
  return Rd ? launch_sizes<64, true>(p, st) : launch_sizes<0, true>(p, st);
}

}  // extern "C"
