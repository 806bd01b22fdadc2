// Grouped expert GEMM for prompts: out[slot] = epi(X[slot / x_div] . W_e^T) over the slots routed to each expert.
//
// Every expert's weights are read, and few rows share them: 700 rows of a model with 8 experts of 4096 x 14336 and 2 per
// row are 175 slots per expert, 2.8 GB of weights (580 us at a copy's rate) for 490 GFLOP.  So
//  * an expert's rows sit in ONE row tile where 320 hold them (more are cut into tiles of equal height, not into full
//    ones and a rest; from 256 on where the tiles then still take one round of the CUs), and products of 16-row fragments past the last row are left out: fragment g of a tile belongs to
//    wave row g % 4, so whatever the height is the waves have the same number of them, but for one;
//  * the column tiles are narrow (128: 1792 tiles of 28672 columns for 8 experts, seven for every CU, and 256 of 4096);
//  * what bounds the stream is the bytes in flight per CU, so the weights' ring is as deep as LDS allows and deeper than
//    the rows' (which come from L2): counted waits are in order per wavefront, so four wavefronts copy rows and four
//    copy weights.  How LDS is shared follows the tallest tile of the launch (Rings).
// Workgroups stay, one per CU: each walks tiles of neighbouring numbers on its XCD and copies the first stages of its next
// tile while it stores the finished one.  Tiles of one expert are neighbours (its gathered rows stay in the XCD's
// L2), and the row tiles of one column tile follow each other (its weights are in the L2 for the second).
//
// Gate and up (28672 x 4096, with the rows' scales) / down (4096 x 14336) of 8 experts, 2 per row, even routing, us,
// 128 x 128 tiles with one launch dimension per expert / this: 65 rows 366 / 318 and 220 / 156, 400 rows 1180 / 367 and
// 583 / 187, 700 rows 678 / 425 and 541 / 226 (a model's uneven routing: 500 and 245 now), 1024 rows 1223 / 640 and
// 630 / 315; 59 to 400 rows per expert 772 / 616 and 539 / 524.  Up to about 200 rows the weight stream (5.9 TB/s) is the
// bound.  Above that a CU takes in some 40 KB/us, rows from the L2 and weights together, which is not what its copies reach
// (95 to 100 KB/us in whole lines, and these are whole lines): what it waits for is not established.  Half a stage read ahead
// of its products measured the same, two stages in flight for rows and weights alike (every wavefront copying both) 5 to 40 % slower; copies issued before the reads
// instead of between the products 2 to 5 % slower from 400 rows on, but for tiles of more than 256 rows (down 365
// against 323 us at 1024 rows).
#pragma once
#include "prefill_gemm.h"

namespace pgemm {

constexpr int MOE_WM = 4;            // wave rows: a tile of NL fragment rows per wave has NL * 64 rows
constexpr int MOE_NL = 5;
constexpr int MOE_ROWS = MOE_NL * 64;

// Row tiles of an expert.  Tiles of more than 256 rows have two stages of rows in flight, which only pays for weights that
// would be read again: where tiles of 256 rows take one round of the CUs all the same (experts of 4096 x 14336 that a rank
// has one or two of), the smaller ones are the faster (down, us: one expert, 320 rows 254 / 149, two of 320 and 330 262 /
// 161; 128 x 128 tiles had 199 and 224)
__device__ __forceinline__ int moe_row_tiles(int cnt, bool tall) {
  return tall ? (cnt + MOE_ROWS - 1) / MOE_ROWS : (cnt + 255) / 256;
}

// LDS stages of 64 numbers of K: rows NL * 8 KiB, weights 16 KiB; 160 KiB together
template <int NL>
struct Rings {
  static constexpr int A = NL == 5 ? 2 : 3;
  static constexpr int B = NL == 1 ? 8 : NL == 2 ? 7 : NL == 4 ? 4 : 5;
  static_assert(A * NL * 8 + B * 16 <= 160, "LDS");
};

// waits until at most `pending` stages of L copies each of this wavefront are in flight
template <int L, int MAX>
__device__ __forceinline__ void wait_stages(int pending) {
  if constexpr (MAX > 0) {
    if (pending < MAX) return wait_stages<L, MAX - 1>(pending);
  }
  wait_vmcnt<MAX * L>();
}

template <int N, int I = 0>
__device__ __forceinline__ void moe_read_a(unsigned at, bf16x8 (&f)[N]) {
  f[I] = ldsp::lds_rd_at<I * 8192>(at);
  if constexpr (I + 1 < N) moe_read_a<N, I + 1>(at, f);
}
template <int EPI, int KS>
__device__ __forceinline__ void moe_read_b(unsigned at, bf16x8 (&f)[4]) {
  constexpr int UP = EPI == EPI_SILU ? 4 : 2;
  f[0] = ldsp::lds_rd_at<KS * 1024>(at);
  f[1] = ldsp::lds_rd_at<2048 + KS * 1024>(at);
  f[2] = ldsp::lds_rd_at<UP * 2048 + KS * 1024>(at);
  f[3] = ldsp::lds_rd_at<(UP + 1) * 2048 + KS * 1024>(at);
}

// EPI_SILU / EPI_STORE; rows' rstd (ea.rstd_in, per row of X) and weights (ea.row_w, per slot) are applied at the end
template <int EPI, int NL>
__device__ __forceinline__ void moe_gemm_body(bf16x8* lds, const bf16x8* __restrict__ Wt, const bf16* __restrict__ X,
                                              int ldx, int M, int K, int n_tiles, int up_off, bf16* __restrict__ out,
                                              int ldo, const EpiArgs& ea, bool tall, int idx, int last, int step) {
  constexpr int WM = MOE_WM, FN = 4, SA = Rings<NL>::A, SB = Rings<NL>::B;
  constexpr int ASTAGE = NL * 512, BSTAGE = 1024;      // bf16x8
  constexpr int LA = 2 * NL, LB = 4;                   // copies per stage of a wavefront that has them
  static_assert(EPI == EPI_SILU || EPI == EPI_STORE, "epilogue");
  bf16x8* ldsb = lds + SA * ASTAGE;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w >> 1, wn = w & 1, r = lane & 15, q = lane >> 4;
  const bool rows_wave = w < 4;
  const int S = K >> 5, n = K / BK, E = ea.n_experts;

  struct Tile {
    int e, nt, m0, rows;   // expert, column tile, first slot of the list, slots
  };
  auto locate = [&](int i) {
    Tile t{0, 0, 0, 0};
    int before = 0;
    for (int b = 0; b < E; b += 64) {
      const int cnt = b + lane < E ? min(ea.moe_cnt[b + lane], M) : 0;
      const int c = moe_row_tiles(cnt, tall);
      int incl = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      const unsigned long long hit = __ballot((before + incl) * n_tiles > i);
      if (hit) {
        const int src = __ffsll(hit) - 1, tm = __shfl(c, src, 64), all = __shfl(cnt, src, 64);
        const int at = i - (before + __shfl(incl, src, 64) - tm) * n_tiles;
        const int h = ((all + 15) / 16 + tm - 1) / tm * 16;
        t.e = b + src;
        t.nt = at / tm;
        t.m0 = (at % tm) * h;
        t.rows = min(h, all - t.m0);
        break;
      }
      before += __shfl(incl, 63, 64);
    }
    t.e = __builtin_amdgcn_readfirstlane(t.e);
    t.nt = __builtin_amdgcn_readfirstlane(t.nt);
    t.m0 = __builtin_amdgcn_readfirstlane(t.m0);
    t.rows = __builtin_amdgcn_readfirstlane(t.rows);
    return t;
  };

  const char* src[LA > LB ? LA : LB];   // this lane's part of stage 0 of each of its copies
  auto sources = [&](const Tile& t) {
    if (rows_wave) {
      // an instruction takes 8 rows x 128 bytes; chunk p of LDS row R holds the row's chunk p ^ (R & 7), so that
      // the 16 rows of a fragment are read without bank conflicts.  Rows past the last repeat it.
      const int* slots = ea.moe_rows + (size_t)t.e * ea.rows_stride + t.m0;
#pragma unroll
      for (int i = 0; i < LA; ++i) {
        const int R = 8 * (w + 4 * i) + (lane >> 3);
        const int s = slots[min(R, t.rows - 1)];
        src[i] = (const char*)(X + (size_t)(s / ea.x_div) * ldx + 8 * ((lane & 7) ^ (R & 7)));
      }
    } else {
      const bf16x8* we = Wt + (size_t)t.e * ea.w_stride;
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const int blk = w - 4 + 4 * i, gi = blk >> 1;   // column group of the tile; gate groups, then up groups
        const int g = EPI == EPI_SILU ? (gi < 4 ? t.nt * 4 + gi : t.nt * 4 + (gi - 4) + up_off) : t.nt * 8 + gi;
        src[i] = (const char*)(we + ((size_t)g * S + (blk & 1)) * 64 + lane);
      }
    }
  };
  const unsigned lds_a = __builtin_amdgcn_readfirstlane(ldsp::lds_off(lds)) + (w & 3) * 1024, lds_b = lds_a + SA * ASTAGE * 16;
  auto copy_a = [&](int i, int kt) {
    ldsp::dma_lds16(src[i] + kt * (BK * 2), lds_a + (kt % SA) * (ASTAGE * 16) + i * 4096);
  };
  auto copy_b = [&](int i, int kt) {
    ldsp::dma_lds16(src[i] + (size_t)kt * 2048, lds_b + (kt % SB) * (BSTAGE * 16) + i * 4096);
  };
  auto issue_a = [&](int kt) {
#pragma unroll
    for (int i = 0; i < LA; ++i) copy_a(i, kt);
  };
  auto issue_b = [&](int kt) {
#pragma unroll
    for (int i = 0; i < LB; ++i) copy_b(i, kt);
  };
  auto prologue = [&]() {
    if (rows_wave) {
      for (int t = 0; t < min(SA - 1, n); ++t) issue_a(t);
    } else {
      for (int t = 0; t < min(SB - 1, n); ++t) issue_b(t);
    }
  };

  // LDS byte addresses: rows (per half of a stage, fragment row i 8 KiB further), weights (column group c 2 KiB further)
  const unsigned fa0 = ldsp::lds_off(lds) + (wm * 16 + r) * 128 + (q ^ (r & 7)) * 16;
  const unsigned fa1 = ldsp::lds_off(lds) + (wm * 16 + r) * 128 + ((4 + q) ^ (r & 7)) * 16;
  constexpr int CW = EPI == EPI_SILU ? 2 : 4;   // neighbouring column groups of a wave; SwiGLU: two more, 4 further
  const unsigned fb = ldsp::lds_off(ldsb) + wn * CW * 2048 + lane * 16;

  f32x4 acc[NL][FN];
  // all stages of a wave that has LIVE fragment rows
  auto walk = [&](auto live) {
    constexpr int LIVE = decltype(live)::value;
    constexpr bool BETWEEN = LIVE > 0 && NL < 5;   // copies go out between products; a ring of two stages wants them first
    for (int t = 0; t < n; ++t) {
      if (rows_wave) wait_stages<LA, SA - 2>(n - 1 - t);   // this wavefront's copies of stage t have landed
      else wait_stages<LB, SB - 2>(n - 1 - t);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();                        // ... and every other's; the stage before is used up
      const int ahead = t + (rows_wave ? SA : SB) - 1;     // the stage this wavefront copies next
      if constexpr (!BETWEEN) {
        if (ahead < n) {
          if (rows_wave) issue_a(ahead);
          else issue_b(ahead);
        }
      }
      if constexpr (LIVE > 0) {
        const unsigned sa = (t % SA) * (ASTAGE * 16), sb = fb + (t % SB) * (BSTAGE * 16);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          bf16x8 af[LIVE], bfr[FN];
          const unsigned at = sa + (ks ? fa1 : fa0);
          if (ks == 0) moe_read_b<EPI, 0>(sb, bfr);
          else moe_read_b<EPI, 1>(sb, bfr);
          moe_read_a(at, af);
          ldsp::lds_wait(af, bfr);
          __builtin_amdgcn_s_setprio(1);
#pragma unroll
          for (int i = 0; i < LIVE; ++i) {
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
            if (BETWEEN && ks == 0) {
              __builtin_amdgcn_sched_barrier(0);
              if (ahead < n) {
                if (rows_wave) {
#pragma unroll
                  for (int c = i * LA / LIVE; c < (i + 1) * LA / LIVE; ++c) copy_a(c, ahead);
                } else {
#pragma unroll
                  for (int c = i * LB / LIVE; c < (i + 1) * LB / LIVE; ++c) copy_b(c, ahead);
                }
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          }
          __builtin_amdgcn_s_setprio(0);
        }
      }
    }
  };

  Tile cur = locate(idx);
  sources(cur);
  prologue();
  while (true) {
#pragma unroll
    for (int i = 0; i < NL; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the rows' slots and scales arrive with the first stages
    int slot[NL][4];
    float scale[NL][4];
    {
      const int* slots = ea.moe_rows + (size_t)cur.e * ea.rows_stride + cur.m0;
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int m = (WM * i + wm) * 16 + 4 * q + jj;
          slot[i][jj] = m < cur.rows ? slots[m] : -1;
        }
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int s = max(slot[i][jj], 0);
          scale[i][jj] = ea.rstd_in ? ea.rstd_in[s / ea.x_div] : 1.f;
          if (ea.row_w) scale[i][jj] *= ea.row_w[s];
        }
    }
    const int live = ((cur.rows + 15) / 16 - wm + WM - 1) / WM;   // 0 .. NL
    switch (live) {
      case 0: walk(std::integral_constant<int, 0>{}); break;
      case 1: walk(std::integral_constant<int, 1>{}); break;
      case 2: walk(std::integral_constant<int, NL < 2 ? NL : 2>{}); break;
      case 3: walk(std::integral_constant<int, NL < 3 ? NL : 3>{}); break;
      case 4: walk(std::integral_constant<int, NL < 4 ? NL : 4>{}); break;
      default: walk(std::integral_constant<int, NL>{}); break;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();   // the stages are free
    const int nt = cur.nt;
    idx += step;
    const bool more = idx < last;
    if (more) {
      cur = locate(idx);
      sources(cur);
      prologue();
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) {
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        if (slot[i][jj] < 0) continue;
        const float sc = scale[i][jj];
        bf16* o = out + (size_t)slot[i][jj] * ldo + r;
        if constexpr (EPI == EPI_SILU) {
#pragma unroll
          for (int j = 0; j < 2; ++j)
            o[(nt * 4 + wn * 2 + j) * 16] = f2bf(silu(acc[i][j][jj] * sc) * (acc[i][j + 2][jj] * sc));
        } else {
#pragma unroll
          for (int j = 0; j < FN; ++j) o[(nt * 8 + wn * 4 + j) * 16] = f2bf(acc[i][j][jj] * sc);
        }
      }
    }
    if (!more) return;
  }
}

template <int EPI>
__global__ __launch_bounds__(NT) void moe_gemm_kernel(const bf16x8* __restrict__ Wt, const bf16* __restrict__ X,
                                                      int ldx, int M, int K, int n_tiles, int up_off,
                                                      bf16* __restrict__ out, int ldo, EpiArgs ea) {
  __shared__ __attribute__((aligned(16))) bf16x8 lds[160 * 64];
  const int lane = threadIdx.x & 63;
  // row tiles in all and the 16-row fragments of the tallest, cut at 256 rows and at MOE_ROWS
  int total[2] = {0, 0}, high[2] = {0, 0};
  for (int b = 0; b < ea.n_experts; b += 64) {
    const int cnt = b + lane < ea.n_experts ? min(ea.moe_cnt[b + lane], M) : 0;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      int c = moe_row_tiles(cnt, t), h = c ? ((cnt + 15) / 16 + c - 1) / c : 0;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        c += __shfl_xor(c, o, 64);
        h = max(h, __shfl_xor(h, o, 64));
      }
      total[t] += c;
      high[t] = max(high[t], h);
    }
  }
  const bool tall = __builtin_amdgcn_readfirstlane(total[0]) * n_tiles > (int)gridDim.x;
  const int tiles = __builtin_amdgcn_readfirstlane(tall ? total[1] : total[0]) * n_tiles;
  const int nl = (__builtin_amdgcn_readfirstlane(tall ? high[1] : high[0]) + MOE_WM - 1) / MOE_WM;
  // an XCD's workgroups share a contiguous run of tiles
  const int xcd = blockIdx.x & 7, step = gridDim.x >> 3;
  const int last = (int)((long long)(xcd + 1) * tiles / 8);
  const int idx = (int)((long long)xcd * tiles / 8) + (blockIdx.x >> 3);
  if (idx >= last) return;
  switch (nl) {
    case 1: return moe_gemm_body<EPI, 1>(lds, Wt, X, ldx, M, K, n_tiles, up_off, out, ldo, ea, tall, idx, last, step);
    case 2: return moe_gemm_body<EPI, 2>(lds, Wt, X, ldx, M, K, n_tiles, up_off, out, ldo, ea, tall, idx, last, step);
    case 3: return moe_gemm_body<EPI, 3>(lds, Wt, X, ldx, M, K, n_tiles, up_off, out, ldo, ea, tall, idx, last, step);
    case 4: return moe_gemm_body<EPI, 4>(lds, Wt, X, ldx, M, K, n_tiles, up_off, out, ldo, ea, tall, idx, last, step);
    default: return moe_gemm_body<EPI, MOE_NL>(lds, Wt, X, ldx, M, K, n_tiles, up_off, out, ldo, ea, tall, idx, last, step);
  }
}

template <int EPI>
int launch_moe_gemm(const void* Wt, const void* X, int ldx, int M, int K, int N, void* out, int ldo,
                    const EpiArgs& ea, hipStream_t st) {
  const int cus = cu_count();
  hipLaunchKernelGGL((moe_gemm_kernel<EPI>), dim3(cus > 8 ? cus / 8 * 8 : 8), dim3(NT), 0, st, (const bf16x8*)Wt,
                     (const bf16*)X, ldx, M, K, N / 128, EPI == EPI_SILU ? N / 32 : 0, (bf16*)out, ldo, ea);
  return (int)hipGetLastError();
}

}  // namespace pgemm
