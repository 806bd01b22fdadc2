// Prefill GEMM v2: MFMA GEMM with direct global->LDS (LDS-DMA) staging.
//
//   out[m, n] = epilogue( rstd[m] * sum_k X[m, k] * W[n, k] )   (gemm_epilogue.h)
//
// Tiles BM x BN x 64 (launch_tile has the shapes, pick_tile the choice): 512 threads = 8 waves in a 2 (M) x 4 (N)
// grid, wave tile (BM/2) x (BN/4) of v_mfma_f32_16x16x32_bf16 accumulators.
// Both operands are staged with `global_load_lds_dwordx4` (one wave-instruction
// = 1 KiB), so no VGPRs or VALU are spent on staging, and read by conflict-free
// ds_read_b128:
//   * W is fragment-major in HBM already (ops.tile_weight): a block is one MFMA
//     fragment, 1 KiB contiguous;
//   * X is row-major: a block is 8 rows x 128 bytes, whole lines (a CU takes those
//     in at 95 to 100 KB/us, the 16 rows x 64 bytes of a fragment at 58), 16-byte
//     piece p of row R at p ^ (R & 7).
// LDS holds two to five stages of (BM+BN) x 64 bf16 (stages_for, launch_pairs): later
// stages are in flight while the MFMAs consume stage kt; one barrier per
// k-tile.  Blocks sharing a weight n-tile are consecutive after the XCD remap.
// NORM: the waves of column 0 also square the A fragments they read; a lane
// sees 8 of every 32 k of one row, 3 shuffles finish the row's sum.
#pragma once
#include <algorithm>

#include "gemm_epilogue.h"
#include "lds_pipe.h"

// The split-K fault word of the current device (tiled_gemm.hip): one int per device,
// allocated with the first split-K workspace and never moved, so a captured graph, the
// Python check (ops.gemm.tiled_split_fault) and the native loop (EngineLoop::set_aux_fault)
// all see the same word.  nullptr while a capture is in progress and it does not exist yet.
extern "C" int* p2p_split_fault_word_ptr(hipStream_t st);

namespace pgemm {

constexpr int BK = 64;
constexpr int NT = 512;
typedef int v4i __attribute__((ext_vector_type(4)));

typedef __attribute__((address_space(3))) void* lds_ptr_t;

struct SplitArgs {
  int splitk;          // K slices per output tile (1 = no split)
  f32x4* slab;         // [tiles][splitk][FM*FN][NT] partial accumulators
  float* ss_slab;      // [tiles][splitk][BM] partial row sums of squares
  unsigned* counters;  // [tiles], zeroed before the launch
  // parallel reduction (every slice reduces its part of the tile's fragment rows; all slices of a
  // tile must be resident together -- the host enables it only for grids <= the CU count):
  unsigned* gen;       // [tiles] generation, bumped by each tile's last arriver
  int* err;            // set if a slice waited past the spin bound (results invalid)
  int parallel;
};

constexpr long long SPLIT_SPIN_TICKS = 20000000;  // 200 ms at the 100 MHz constant clock

// Write-through (sc1) 16-byte store / load through a raw buffer resource (aux 16 = sc1):
// hand-off payload that needs no release fence and is read past stale L1/L2 copies
// (cdna_hip_programming.md Guideline 16, R1).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7FFFFFFF,
                                           0x00020000);
}
__device__ __forceinline__ void store_sc1(__amdgpu_buffer_rsrc_t r, int off, const f32x4& v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, v), r, off, 0, 16);
}
__device__ __forceinline__ f32x4 load_sc1(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16));
}

// Tile coordinates of linear tile index t in GROUP_M-row bands: consecutive indices walk
// GROUP_M m-tiles of one n-tile, then the next n-tile.  After xcd_remap an XCD's ~32
// concurrent blocks (one per CU) therefore cover 8 m-tiles x 4 n-tiles -- per k-step 12
// distinct 32 KiB operand slices instead of 33 with m innermost over every m-tile (L2 hit
// rate ~50 % -> ~80 %), and each XCD streams its A rows once instead of once per n-tile.
// Identical to (t % m_tiles, t / m_tiles) for m_tiles <= GROUP_M.
constexpr int GROUP_M = 8;
__device__ __forceinline__ void grouped_tile(int t, int m_tiles, int n_tiles, int& mt, int& nt) {
  const int per_group = GROUP_M * n_tiles;
  const int g = t / per_group, first = g * GROUP_M;
  const int gm = min(m_tiles - first, GROUP_M);
  const int r = t - g * per_group;
  mt = first + r % gm;
  nt = r / gm;
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Waits until at most `pending` x L of this thread's LDS-DMA loads are in flight.
template <int L, int STAGES>
__device__ __forceinline__ void wait_tiles(int pending) {
  if constexpr (STAGES >= 6) {
    if (pending >= 4) { wait_vmcnt<4 * L>(); return; }
  }
  if constexpr (STAGES >= 5) {
    if (pending >= 3) { wait_vmcnt<3 * L>(); return; }
  }
  if constexpr (STAGES >= 4) {
    if (pending >= 2) { wait_vmcnt<2 * L>(); return; }
  }
  if constexpr (STAGES >= 3) {
    if (pending >= 1) { wait_vmcnt<L>(); return; }
  }
  wait_vmcnt<0>();
}

// an address that is the same for all lanes, in scalar registers
__device__ __forceinline__ const char* wave_address(const void* p) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)a), hi = __builtin_amdgcn_readfirstlane((unsigned)(a >> 32));
  return reinterpret_cast<const char*>((uint64_t)hi << 32 | lo);
}

// scalar arguments that are to be in registers from here on
template <typename T>
__device__ __forceinline__ void pin_scalar(const T& v) {
  asm volatile("" ::"s"(v));
}
template <typename... T>
__device__ __forceinline__ void pin_scalars(const T&... v) {
  (pin_scalar(v), ...);
}

// Tiles that read ahead (a workgroup has the CU to itself): 128 rows and more (but see launch_pairs).  In step, eight wavefronts read a half stage,
// waited, multiplied it, and issued the copies between.  These read the next half stage a fragment row at a time under the
// products of the present one, and issue their copies (a scalar address and a lane's constant offset) between the products, into
// the stage whose second half every wave has in registers.  llama3.1-8B, us: down, 1024 rows, in step 173, on four wavefronts
// of 128 x 128 136, now 128 x 256 112 (1080 TFLOP/s); SwiGLU 28672 x 4096, 256 x 256 in four phases with a unit of copies
// each 219, now 195 (1240 TFLOP/s), 398 rows 119, now 102; 4096 x 4096, 128 x 128 on four wavefronts 40, now 35, and with the
// residual 50, now 36; 6144 x 4096, 128 x 192 on four 55, now 47.  256 x 128 measured as 128 x 256.
template <int BM, int BN, int STAGES, bool NORM>
constexpr bool reads_ahead() {
  if (BM * BN == 256 * 256 && NORM) return false;   // (no registers for the sums)
  return BM >= 128 && (STAGES >= 3 || BM * BN >= 192 * 256);
}

template <int BM, int BN, int EPI, bool NORM, bool SPLIT, int STAGES>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2))) void prefill_gemm_kernel(const bf16x8* __restrict__ Wt,
                                                          const bf16* __restrict__ X, int ldx,
                                                          int M, int K, int m_tiles, int n_tiles,
                                                          int up_off, void* __restrict__ out,
                                                          int ldo, float eps, EpiArgs ea,
                                                          SplitArgs sp) {
  constexpr bool PIPE = reads_ahead<BM, BN, STAGES, NORM>();
  constexpr int NWV = NT / 64, WN = NWV / 2;   // 2 x WN wave grid
  constexpr int FM = BM / 32;        // 16-row fragments per wave
  constexpr int FN = BN / (16 * WN);  // 16-col groups per wave
  constexpr int AB = BM / 16 * 2;    // A fragment blocks per stage (x 1 KiB)
  constexpr int BB = BN / 16 * 2;    // B fragment blocks per stage
  constexpr int STAGE = (AB + BB) * 64;  // bf16x8 per stage
  constexpr int AI = AB / NWV, BI = BB / NWV;  // blocks per wave per stage
  constexpr int L = AI + BI;               // LDS-DMA instructions per thread per stage
  constexpr bool RES_AHEAD = BM * BN <= 128 * 256;   // (larger tiles have no registers for them)
  static_assert(AB % NWV == 0 && BB % NWV == 0, "tile");
  static_assert(FM >= 1 && FN >= 2, "tile");
  // PIPE: given at the launch.  A static 160 KiB tells the compiler that one wavefront per SIMD is all there can be, and it
  // moves the accumulators through AGPRs, four copies per product
  extern __shared__ __attribute__((aligned(16))) bf16x8 lds_given[];
  __shared__ __attribute__((aligned(16))) bf16x8 lds_own[PIPE ? 1 : STAGES * STAGE];
  bf16x8* lds = PIPE ? lds_given : lds_own;

  const int splitk = SPLIT ? sp.splitk : 1;
  const int nb = m_tiles * n_tiles * splitk;
  const int b = xcd_remap(blockIdx.x, nb);
  // a tile's K slices are consecutive (same XCD: the reducer reads them from its L2)
  const int tile = b / splitk, split = b % splitk;
  int mt_i, nt_i;
  grouped_tile(tile, m_tiles, n_tiles, mt_i, nt_i);
  const int m0 = mt_i * BM;
  // rows' RMSNorm rstd precomputed by row_rstd_kernel (ea.rstd_in): the host launches the
  // NORM = false instantiation, so no sums of squares ride in the k loop (they cost
  // 12-22 % of the GEMM, profiles/r2_norm_cost.jsonl); applied in the epilogue
  const bool pre = !NORM && ea.rstd_in != nullptr;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w / WN, wn = w % WN;
  const int S = K >> 5;
  const int nk_all = K / BK;
  const int kt0 = split * nk_all / splitk, kt1 = (split + 1) * nk_all / splitk;
  const int n = kt1 - kt0;

  auto group_of = [&](int gi) -> int {  // LDS group slot -> global 16-col group
    if constexpr (EPI == EPI_SILU) {
      constexpr int H = BN / 32;
      return gi < H ? nt_i * H + gi : nt_i * H + (gi - H) + up_off;
    }
    return nt_i * (BN / 16) + gi;
  };

  // ---- per-lane DMA sources (k offsets added per k-tile) ----
  const bf16* asrc[AI];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    // 8 rows x 128 bytes per block, 16-byte chunks of row R permuted by R & 7
    int row = m0 + 8 * (w + NWV * i) + (lane >> 3);
    row = row < M ? row : M - 1;
    asrc[i] = X + (size_t)row * ldx + 8 * ((lane & 7) ^ (lane >> 3));
  }
  const bf16x8* bsrc[BI];
#pragma unroll
  for (int i = 0; i < BI; ++i) {
    const int blk = w + NWV * i;  // = gi * 2 + ks
    bsrc[i] = Wt + ((size_t)group_of(blk >> 1) * S + (blk & 1)) * 64 + lane;
  }

  // asm DMA + asm LDS reads (lds_pipe.h): with the builtins the compiler put vmcnt(0)
  // before every stage read, draining the STAGES-deep pipeline at every k-tile
  auto issue = [&](int kt, int st) {
    bf16x8* base = lds + st * STAGE;
#pragma unroll
    for (int i = 0; i < AI; ++i) ldsp::dma_lds<16>(asrc[i] + kt * BK, base + (w + NWV * i) * 64);
#pragma unroll
    for (int i = 0; i < BI; ++i) ldsp::dma_lds<16>(bsrc[i] + (size_t)kt * 2 * 64, base + (AB + w + NWV * i) * 64);
  };

  int bgi[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    if constexpr (EPI == EPI_SILU) {
      constexpr int H = FN / 2;
      bgi[j] = j < H ? wn * H + j : BN / 32 + wn * H + (j - H);
    } else {
      bgi[j] = wn * FN + j;
    }
  }

  // the residual values of fragment rows i0 .. i1 - 1 of the wave at (wm_, wn_)
  auto residuals = [&](int wm_, int wn_, int i0, int i1, bf16(&res)[FM][4][FN]) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (i < i0 || i >= i1) continue;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int m = min(m0 + wm_ * (BM / 2) + 16 * i + 4 * (lane >> 4) + jj, M - 1);
#pragma unroll
        for (int j = 0; j < FN; ++j)
          res[i][jj][j] = reinterpret_cast<const bf16*>(out)[(size_t)m * ldo + (nt_i * (BN / 16) + wn_ * FN + j) * 16 + (lane & 15)];
      }
    }
  };
  // They are loaded before the copies begin (behind the products they cost 7 us: 4096 x 4096, 1024 rows, 43 us where the plain
  // product takes 36), by the slices of a reduction while they wait for each other
  bf16 res[FM][4][FN];
  if constexpr (EPI == EPI_RESID && !SPLIT && RES_AHEAD) residuals(wm, wn, 0, FM, res);

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) ss[i] = 0.f;

  // ---- STAGES-deep LDS-DMA pipeline: counted vmcnt + raw barriers, so the
  // younger stages stay in flight across the barrier (no vmcnt(0) drain) ----
  if constexpr (!PIPE)
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
      if (t < n) issue(kt0 + t, t);
  if constexpr (PIPE) {
    // copies: a wave-uniform address per stage, a lane's offset that stays
    const char* abase = wave_address(X + (size_t)m0 * ldx + (size_t)kt0 * BK);
    constexpr int HALF = EPI == EPI_SILU ? BI / 2 : BI;   // SwiGLU: a wave's first copies are gate columns, the rest up
    constexpr int TILE_GROUPS = EPI == EPI_SILU ? BN / 32 : BN / 16;
    static_assert(EPI != EPI_SILU || BI % 2 == 0, "halves");
    const char* bbase = wave_address(Wt + ((size_t)nt_i * TILE_GROUPS * S + (size_t)kt0 * 2) * 64);
    const size_t to_up = EPI == EPI_SILU ? (size_t)up_off * S * 1024 : 0;
    unsigned aoff[AI], boff[BI];
#pragma unroll
    for (int i = 0; i < AI; ++i) aoff[i] = (unsigned)((const char*)asrc[i] - reinterpret_cast<const char*>(X + (size_t)m0 * ldx));
#pragma unroll
    for (int i = 0; i < BI; ++i)
      boff[i] = (unsigned)((const char*)(bsrc[i] + (size_t)kt0 * 128) - bbase - (i < HALF ? 0 : to_up));
    const unsigned lds0 = ldsp::lds_off(lds) + __builtin_amdgcn_readfirstlane(w) * 1024;
    auto copy = [&](int i, int t) {   // the i-th of this wave's L copies of stage t
      const unsigned l = lds0 + (t % STAGES) * (STAGE * 16) + (i < AI ? i : AB / NWV + i - AI) * (NWV * 1024);
      if (i < AI) ldsp::dma_lds16(abase + (size_t)t * (BK * 2), aoff[i < AI ? i : 0], l);
      else ldsp::dma_lds16(bbase + (i - AI < HALF ? 0 : to_up) + (size_t)t * 2048, boff[i < AI ? 0 : i - AI], l);
    };
#pragma unroll
    for (int t = 0; t < STAGES; ++t)
      if (t < n)
#pragma unroll
        for (int i = 0; i < L; ++i) copy(i, t);
    // (LDS reads as plain loads: the copies are asm, so the compiler waits for exactly what a product needs)
    const int ar = (wm * FM * 16 + (lane & 15)) * 8, aq = lane >> 4, ax = lane & 7;
    auto read_part = [&](int t, int ks, int i, bf16x8(&af)[FM], bf16x8(&bfr)[FN]) {   // fragment row i and its share of columns
      const bf16x8* sa = lds + (t % STAGES) * STAGE;
      const bf16x8* sb = sa + AB * 64 + lane;
      af[i] = sa[ar + i * 128 + ((4 * ks + aq) ^ ax)];
#pragma unroll
      for (int j = i * FN / FM; j < (i + 1) * FN / FM; ++j) bfr[j] = sb[(bgi[j] * 2 + ks) * 64];
    };
    auto read = [&](int t, int ks, bf16x8(&af)[FM], bf16x8(&bfr)[FN]) {
#pragma unroll
      for (int i = 0; i < FM; ++i) read_part(t, ks, i, af, bfr);
      __builtin_amdgcn_sched_barrier(0);
    };
    // between(i): what is issued behind the products of fragment row i
    auto products = [&](const bf16x8(&af)[FM], const bf16x8(&bfr)[FN], auto&& between) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        between(i);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (NORM) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          if (i % WN == wn) ss[i] = sumsq8(af[i], ss[i]);
      }
    };
    auto nothing = [](int) {};
    auto meet = [] {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");   // (the barrier alone does not order reads of LDS)
    };
    bf16x8 a0[FM], b0[FN], a1[FM], b1[FN];
    // stages 0 .. STAGES - 1 are under way; stage 0 alone has to be there
    wait_tiles<L, STAGES + 1>(min(STAGES - 1, n - 1));
    meet();
    // the epilogue's arguments are loaded now, and lgkmcnt(0) is seen by the compiler: with a scalar load under way where
    // the loop begins it waits for all LDS reads before each product
    pin_scalars(out, ldo, eps, ea.rstd_in);
    if constexpr (EPI == EPI_QKV_ROPE)
      pin_scalars(ea.pos, ea.slots, ea.cs, ea.q_out, ea.ldq, ea.kc, ea.vc, ea.Hq, ea.Hkv);
    if constexpr (EPI == EPI_ARGMAX) pin_scalars(ea.col_offset);
    if constexpr (SPLIT) pin_scalars(sp.splitk, sp.slab, sp.ss_slab, sp.counters, sp.gen, sp.err, sp.parallel);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    read(0, 0, a0, b0);
    // the second half of stage t is in this wave's registers before it meets the others, so from then on the stage's
    // slot takes the next copies: a copy has STAGES - 1 stages' time
    auto used_up = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    int t = 0;
    if constexpr (BM * BN >= 192 * 256) {   // one loop for all stages takes 24 registers fewer, which these tiles do not have
      for (; t + 1 < n; ++t) {
        const bool more = t + STAGES < n;
        products(a0, b0, [&](int i) { read_part(t, 1, i, a1, b1); });
        used_up();
        wait_tiles<L, STAGES>(more ? STAGES - 2 : min(STAGES - 2, n - 2 - t));
        meet();
        products(a1, b1, [&](int i) {
          read_part(t + 1, 0, i, a0, b0);
          if (more)
#pragma unroll
            for (int c = i * L / FM; c < (i + 1) * L / FM; ++c) copy(c, t + STAGES);
        });
      }
    } else {
      for (; t + STAGES < n; ++t) {
        products(a0, b0, [&](int i) { read_part(t, 1, i, a1, b1); });
        used_up();
        wait_vmcnt<(STAGES - 2) * L>();   // stage t + 1 is there, for every wave once they met
        meet();
        products(a1, b1, [&](int i) {
          read_part(t + 1, 0, i, a0, b0);
#pragma unroll
          for (int c = i * L / FM; c < (i + 1) * L / FM; ++c) copy(c, t + STAGES);
        });
      }
      for (; t + 1 < n; ++t) {
        read(t, 1, a1, b1);
        products(a0, b0, nothing);
        wait_tiles<L, STAGES>(min(STAGES - 2, n - 2 - t));
        meet();
        read(t + 1, 0, a0, b0);
        products(a1, b1, nothing);
      }
    }
    read(t, 1, a1, b1);
    products(a0, b0, nothing);
    products(a1, b1, nothing);
  } else {
    for (int t = 0; t < n; ++t) {
      wait_tiles<L, STAGES>(min(STAGES - 2, n - 1 - t));  // tile t landed (this thread's part)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();                       // ... and every other wave's part
      if (t + STAGES - 1 < n) issue(kt0 + t + STAGES - 1, (t + STAGES - 1) % STAGES);
      const bf16x8* sa = lds + (t % STAGES) * STAGE;
      const bf16x8* sb = sa + AB * 64;
  #pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        bf16x8 af[FM], bfr[FN];
  #pragma unroll
        for (int j = 0; j < FN; ++j) bfr[j] = ldsp::lds_rd(sb + (bgi[j] * 2 + ks) * 64 + lane);
  #pragma unroll
        for (int i = 0; i < FM; ++i)
          af[i] = ldsp::lds_rd(sa + ((wm * FM + i) * 16 + (lane & 15)) * 8 + ((4 * ks + (lane >> 4)) ^ (lane & 7)));
        ldsp::lds_wait(af, bfr);
        // keep the MFMA cluster together against the co-resident wave (guide T5)
        __builtin_amdgcn_s_setprio(1);
  #pragma unroll
        for (int i = 0; i < FM; ++i)
  #pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (NORM) {  // RMSNorm sums: fragment i by wave wn == i % 4 (VALU spread)
  #pragma unroll
          for (int i = 0; i < FM; ++i) {
            if ((i & 3) != wn) continue;
            ss[i] = sumsq8(af[i], ss[i]);
          }
        }
      }
    }
  }
  wait_vmcnt<0>();
  __syncthreads();  // every wave done reading the stages before LDS is reused below

  // ---- row rstd (NORM): column-0 waves publish through LDS (stages are free now) ----
  float* ss_row = reinterpret_cast<float*>(lds);
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (i % WN != wn) continue;
      float v = ss[i];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lane < 16) {
        if constexpr (SPLIT)
          __hip_atomic_store(&sp.ss_slab[((size_t)tile * splitk + split) * BM + wm * (BM / 2) + 16 * i + lane],
                             v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // write-through
        else
          ss_row[wm * (BM / 2) + 16 * i + lane] = v;
      }
    }
    if constexpr (!SPLIT) __syncthreads();
  }
  // ---- epilogue of one wave's accumulators (wave grid position wm_, wn_) ----
  const int r = lane & 15, q = lane >> 4;
  // (fragment rows i0 .. i1 - 1)
  auto epilogue = [&](int wm_, int wn_, const f32x4 (&ac)[FM][FN], auto&& scale_of, int i0, int i1) {
    int bg[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (EPI == EPI_SILU) {
        constexpr int H = FN / 2;
        bg[j] = j < H ? wn_ * H + j : BN / 32 + wn_ * H + (j - H);
      } else {
        bg[j] = wn_ * FN + j;
      }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (i < i0 || i >= i1) continue;
      // a fragment row's epilogue operands as one batch (residual values; the rows' positions -> (cos, sin) and KV slots): per
      // element, between the stores they may alias, they were FN x 4 dependent round trips per fragment row
      float resv[4][FN];
      if constexpr (EPI == EPI_RESID) {
        if constexpr (!RES_AHEAD) residuals(wm_, wn_, i, i + 1, res);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
          for (int j = 0; j < FN; ++j) resv[jj][j] = (float)res[i][jj][j];
      }
      float2 csv[4][FN];
      int slotv[4];
      if constexpr (EPI == EPI_QKV_ROPE) {
        int posv[4];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int m = m0 + wm_ * (BM / 2) + 16 * i + 4 * q + jj;
          posv[jj] = 0;
          slotv[jj] = -1;
          if (m < M) {
            posv[jj] = ea.pos[m];
            slotv[jj] = ea.slots[m];
          }
        }
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int g = nt_i * (BN / 16) + bg[j];
            const int kk = g & 7;
            const int dd = ((r < 8) ? 8 * kk + r : 64 + 8 * kk + (r - 8)) & 63;
            const bool ok = m0 + wm_ * (BM / 2) + 16 * i + 4 * q + jj < M;
            csv[jj][j] = ok ? ea.cs[(size_t)posv[jj] * 64 + dd] : float2{1.f, 0.f};
          }
      }
      float scv[4];  // the rows' rstd (loads, with the operands above)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) scv[jj] = scale_of(i, jj);
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int rl = wm_ * (BM / 2) + 16 * i + 4 * q + jj;
        const int m = m0 + rl;
        const bool valid = m < M;
        const float scale = scv[jj];
        if constexpr (EPI == EPI_SILU) {
          constexpr int H = FN / 2;
#pragma unroll
          for (int j = 0; j < H; ++j)
            epi_store<EPI>(m, valid, nt_i * (BN / 32) + wn_ * H + j, r, ac[i][j][jj] * scale,
                           ac[i][j + H][jj] * scale, out, ldo, ea);
        } else if constexpr (EPI == EPI_QKV_ROPE) {
#pragma unroll
          for (int j = 0; j < FN; ++j)
            epi_store<EPI>(m, valid, nt_i * (BN / 16) + bg[j], r, ac[i][j][jj] * scale, 0.f, out,
                           ldo, ea, csv[jj][j], valid ? slotv[jj] : -1);
        } else if constexpr (EPI == EPI_RESID) {
#pragma unroll
          for (int j = 0; j < FN; ++j)
            if (valid)
              reinterpret_cast<bf16*>(out)[(size_t)m * ldo + (nt_i * (BN / 16) + bg[j]) * 16 + r] =
                  f2bf(resv[jj][j] + ac[i][j][jj] * scale);
        } else {
#pragma unroll
          for (int j = 0; j < FN; ++j)
            epi_store<EPI>(m, valid, nt_i * (BN / 16) + bg[j], r, ac[i][j][jj] * scale, 0.f, out,
                           ldo, ea);
        }
      }
    }
  };
  auto rstd_of = [&](float t) { return rsqrtf(t / (float)K + eps); };
  auto rstd_pre = [&](int rl) {
    return pre ? ea.rstd_in[min(m0 + rl, M - 1)] : 1.f;
  };

  if constexpr (SPLIT) {
    f32x4* my = sp.slab + ((size_t)tile * splitk + split) * (FM * FN) * NT;
    // (the 256x256 tile keeps the serial reduction: a second set of 128 accumulator
    // registers for the shared reduction would spill its main loop)
    if (BM * BN <= 128 * 256 && sp.parallel) {
      // ---- parallel split-K: write-through slabs, one generation flip per tile, then
      // every slice reduces and stores its part of the tile (no serial reducer, no release
      // fence) ----
      const __amdgpu_buffer_rsrc_t rsl = raw_rsrc(sp.slab);
      const size_t tile_v = (size_t)tile * splitk * (FM * FN) * NT;  // f32x4 index of slice 0
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          store_sc1(rsl, (int)((tile_v + ((size_t)split * FM * FN + i * FN + j) * NT + tid) * 16),
                    acc[i][j]);
      // the tile's NWV * FM fragment rows go to the slices in equal runs (host guarantees splitk | 8), and a slice's
      // run to its waves in shares that lie within one wave's rows
      const int units = NWV * FM / splitk;
      int share = (units + NWV - 1) / NWV;
      while (FM % share || units % share) ++share;
      const bool has = w * share < units;
      const int unit = split * units + (has ? w * share : 0);
      const int vw = unit / FM, i0 = unit % FM, i1 = has ? i0 + share : i0;  // whose accumulators this wave finishes
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave drains
      if constexpr (EPI == EPI_RESID && RES_AHEAD) residuals(vw / WN, vw % WN, i0, i1, res);
      __syncthreads();
      if (tid == 0) {
        const unsigned g0 = __hip_atomic_load(&sp.gen[tile], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // read the generation BEFORE arriving
        const unsigned t = __hip_atomic_fetch_add(&sp.counters[tile], 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
        if (t == (unsigned)splitk - 1) {
          (void)__hip_atomic_exchange(&sp.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // re-armed before the flip
          __hip_atomic_store(&sp.gen[tile], g0 + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          const long long t0 = wall_clock64();
          while (__hip_atomic_load(&sp.gen[tile], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g0) {
            if (wall_clock64() - t0 > SPLIT_SPIN_TICKS) {
              __hip_atomic_store(sp.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              break;
            }
            __builtin_amdgcn_s_sleep(1);
          }
        }
      }
      __syncthreads();
      if (!has) return;
      // acc is dead after the slab stores: it becomes the total (one fragment row of
      // loads in flight at a time keeps the 256x256 tile inside its register budget)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int s2 = 0; s2 < splitk; ++s2) {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          if (i < i0 || i >= i1) continue;
          f32x4 part[FN];
#pragma unroll
          for (int j = 0; j < FN; ++j)
            part[j] = load_sc1(rsl, (int)((tile_v + ((size_t)s2 * FM * FN + i * FN + j) * NT +
                                           vw * 64 + lane) * 16));
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] += part[j];
        }
      }
      epilogue(
          vw / WN, vw % WN, acc,
          [&](int i, int jj) {
            const int rl = (vw / WN) * (BM / 2) + 16 * i + 4 * q + jj;
            if constexpr (!NORM) return rstd_pre(rl);
            float t = 0.f;
            for (int s2 = 0; s2 < splitk; ++s2)
              t += __hip_atomic_load(&sp.ss_slab[((size_t)tile * splitk + s2) * BM + rl],
                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return rstd_of(t);
          },
          i0, i1);
      return;
    }
    // ---- serial split-K: agent-scope release/acquire through a per-tile ticket; every
    // slice stores its fp32 partial tile, the last arriver reduces all slices in slice
    // order (deterministic) and runs the epilogue ----
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) my[(i * FN + j) * NT + tid] = acc[i][j];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int* flag = reinterpret_cast<int*>(lds) + BM;
    if (tid == 0) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const unsigned t = __hip_atomic_fetch_add(&sp.counters[tile], 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
      *flag = (t == (unsigned)splitk - 1);
    }
    __syncthreads();
    if (!*flag) return;
    if (tid == 0) {
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    const f32x4* base = sp.slab + (size_t)tile * splitk * (FM * FN) * NT;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s2 = 0; s2 < splitk; ++s2) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] += base[((size_t)s2 * FM * FN + i * FN + j) * NT + tid];
        // 256 x 256: all rows' loads in flight beside 128 accumulators would not fit the registers
        if constexpr (BM * BN >= 256 * 256) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (NORM) {
      if (tid < BM) {
        float t = 0.f;
        for (int s2 = 0; s2 < splitk; ++s2) t += sp.ss_slab[((size_t)tile * splitk + s2) * BM + tid];
        ss_row[tid] = t;
      }
      __syncthreads();
    }
    // every slice has arrived: re-arm the ticket for the next launch (the workspace
    // counters are zeroed once at allocation, so no per-launch memset node is needed)
    if (tid == 0) sp.counters[tile] = 0;
    if constexpr (EPI == EPI_RESID && RES_AHEAD) residuals(wm, wn, 0, FM, res);
  }

  epilogue(
      wm, wn, acc,
      [&](int i, int jj) {
        const int rl = wm * (BM / 2) + 16 * i + 4 * q + jj;
        if constexpr (!NORM) return rstd_pre(rl);
        return rstd_of(ss_row[rl]);
      },
      0, FM);
}

// split-K workspace (device, grown on demand outside graph capture)
struct SplitWs {
  void* buf = nullptr;
  size_t bytes = 0;
};
static SplitWs g_split_ws;

// ticket counters: a fixed region at the end of the workspace, zeroed when the
// workspace is (re)allocated and re-armed by each tile's last arriver
constexpr size_t kCounterBytes = 64 * 1024;  // 16384 tiles

// A grown workspace never frees the previous buffer: a hipGraph captured earlier (the
// decode graph of a mid-M batch bucket routed to this kernel) holds its address and its
// ticket counters and replays against it for the life of the process.  Growth is
// geometric, so the retired buffers total less than the live one.
static bool split_ws(size_t bytes, hipStream_t st, char** out) {
  bytes += kCounterBytes;
  if (g_split_ws.bytes < bytes) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(st, &cs);
    if (cs != hipStreamCaptureStatusNone) return false;  // cannot allocate while capturing
    const size_t want = std::max(bytes, 2 * g_split_ws.bytes);
    void* buf = nullptr;
    if (hipMalloc(&buf, want) != hipSuccess) return false;
    if (hipMemsetAsync(buf, 0, want, st) != hipSuccess) return false;
    if (!p2p_split_fault_word_ptr(st)) return false;
    g_split_ws.buf = buf;  // the old buffer stays allocated (see above)
    g_split_ws.bytes = want;
  }
  *out = (char*)g_split_ws.buf;
  return true;
}

static int g_splitk = 0;  // 0 = heuristic, 1 = never split, >1 = forced
static int g_split_parallel = 1;  // parallel split-K reduction where residency allows

// CUs of the current device (cached per device): the parallel reduction needs every slice
// of a tile resident at once, so it is used only for grids of at most one block per CU.
static int cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 0;
    cached[dev] = n > 0 ? n : -1;
  }
  return cached[dev] > 0 ? cached[dev] : 0;
}

// (128 x 192 leaves no registers for a reduction)
template <int BM, int BN>
constexpr bool splits_k() {
  return BN != 192;
}

// LDS stages per tile shape.  Measured on MI355X (bench/prefill_gemm_bench.py): the
// 64-row tiles are latency-bound streams and want 3-4 stages in flight; those that read ahead have the CU's LDS to
// themselves.
template <int BM, int BN>
constexpr int stages_for() {
  constexpr int most = (160 * 1024) / ((BM + BN) * BK * 2);
  if constexpr (reads_ahead<BM, BN, most, false>()) return most;
  return BN <= 128 ? 4 : 3;
}

// K slices fill one round of the CUs where a tile has a CU to itself; not (A/B): some 400 workgroups whatever the tile
static bool g_fill = true;

template <int BM, int BN, int EPI, bool NORM, int STAGES>
int launch_stages(const void* Wt, const void* X, int ldx, int M, int K, int m_tiles, int n_tiles,
                  int up_off, void* out, int ldo, float eps, const EpiArgs& ea, hipStream_t st,
                  int splitk, char* ws, int par) {
  constexpr size_t SHM = reads_ahead<BM, BN, STAGES, NORM>() ? (size_t)STAGES * (BM + BN) * BK * sizeof(bf16) : 0;
  const int tiles = m_tiles * n_tiles;
  auto with_lds = [](const void* k) {
    return SHM ? hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)SHM) : hipSuccess;
  };
  if constexpr (splits_k<BM, BN>()) {
    if (splitk > 1) {
      constexpr auto kernel = prefill_gemm_kernel<BM, BN, EPI, NORM, true, STAGES>;
      if (const hipError_t e = with_lds((const void*)kernel)) return (int)e;
      const size_t slab = (size_t)tiles * splitk * BM * BN * sizeof(float);
      // counters live at the END of the workspace at a fixed offset from the end so a
      // grown workspace keeps them zeroed; see split_ws.  Layout of that region (u32):
      // [0, n/2) arrival tickets, [n/2, n-1) generations, [n-1] the fault word.
      unsigned* ctr = (unsigned*)(ws + g_split_ws.bytes - kCounterBytes);
      constexpr size_t nw = kCounterBytes / sizeof(unsigned);
      int* fw = p2p_split_fault_word_ptr(st);
      SplitArgs sp{splitk, (f32x4*)ws, (float*)(ws + slab), ctr, ctr + nw / 2,
                   fw ? fw : (int*)(ctr + nw - 1), par};
      hipLaunchKernelGGL(kernel, dim3(tiles * splitk), dim3(NT), SHM, st, (const bf16x8*)Wt,
                         (const bf16*)X, ldx, M, K, m_tiles, n_tiles, up_off, out, ldo, eps, ea, sp);
      return (int)hipGetLastError();
    }
  }
  SplitArgs none{1, nullptr, nullptr, nullptr, nullptr, nullptr, 0};
  constexpr auto kernel = prefill_gemm_kernel<BM, BN, EPI, NORM, false, STAGES>;
  if (const hipError_t e = with_lds((const void*)kernel)) return (int)e;
  hipLaunchKernelGGL(kernel, dim3(tiles), dim3(NT), SHM, st, (const bf16x8*)Wt, (const bf16*)X, ldx, M, K, m_tiles,
                     n_tiles, up_off, out, ldo, eps, ea, none);
  return (int)hipGetLastError();
}

template <int BM, int BN, int EPI, bool NORM>
int launch(const void* Wt, const void* X, int ldx, int M, int K, int N, int up_off, void* out,
           int ldo, float eps, const EpiArgs& ea, hipStream_t st) {
  constexpr int STAGES = stages_for<BM, BN>();
  const int m_tiles = (M + BM - 1) / BM;
  const int n_tiles = N / BN;
  const int tiles = m_tiles * n_tiles;
  const int nk = K / BK;
  const int cus = cu_count();
  constexpr bool ALONE = BM >= 128 && BM * BN <= 128 * 256;   // one workgroup per CU whatever the grid
  const bool fill = ALONE && g_fill && cus > 0 && tiles <= cus;
  // too few tiles to fill 256 CUs: split K so every CU gets work (>= 4 k-tiles per slice)
  // (measured on MI355X at 8B shapes: ~400 blocks, >= 16 k-tiles per slice); tiles that have a
  // CU to themselves keep to one block per CU instead (power-of-two slices <= CUs/tiles)
  int splitk;
  if (g_splitk) {
    splitk = g_splitk;
  } else if (fill) {
    const int cap = std::min(8, std::max(1, std::min(cus / tiles, nk / 16)));
    splitk = 1;
    while (splitk * 2 <= cap) splitk *= 2;
  } else {
    // (256 x 256: from 160 tiles on they fill the chip as they are)
    splitk = BM * BN == 256 * 256 && tiles >= 160 ? 1 : std::min(8, std::max(1, std::min(400 / tiles, nk / 16)));
  }
  splitk = splits_k<BM, BN>() ? std::max(1, std::min(splitk, nk / 4)) : 1;
  char* ws = nullptr;
  int par = 0;
  if (splitk > 1 && (size_t)tiles * sizeof(unsigned) < kCounterBytes / 2) {
    const size_t slab = (size_t)tiles * splitk * BM * BN * sizeof(float);
    const size_t ssb = (size_t)tiles * splitk * BM * sizeof(float);
    if (!(split_ws(slab + ssb, st, &ws) && slab + ssb < 0x7FFFFFFF)) splitk = 1;
    par = g_split_parallel && (8 % splitk) == 0 && cus > 0 && tiles * splitk <= cus;
  } else {
    splitk = 1;
  }
  return launch_stages<BM, BN, EPI, NORM, STAGES>(Wt, X, ldx, M, K, m_tiles, n_tiles, up_off, out, ldo, eps, ea, st, splitk, ws, par);
}

// Tiles of eight wavefronts and two stages, of which a CU takes two: one's start and end lie under the other's products.  192 x 128
// of more than one round of the CUs run so (us, a workgroup with the CU to itself / two: normed 16640 x 512, 470 rows 25 / 21,
// 10112 x 768, 2167 rows 62 / 49, SwiGLU 12288 x 2048, 700 rows 55 / 48, 22016 x 4096, 300 rows 96 / 93, 16640 x 7488, 569 rows
// 169 / 157; over 60 shapes with K of 256 to 8192 between 28 % less and, 10240 x 8192, 878 rows, 163 / 168, 3 % more.  So do SwiGLU's
// of a short K in one round, which end before four stages pay (7424 x 320, 557 rows 13.9 / 12.8, 7680 x 832, 692 rows 18.9 / 18.4,
// but 18176 x 1216, 137 rows 23.6 / 26.8; without SwiGLU 8320 x 384, 537 rows 14.6 / 14.8)
template <int BM, int EPI, bool NORM>
int launch_pairs(const void* Wt, const void* X, int ldx, int M, int K, int N, int up_off, void* out, int ldo, float eps,
                 const EpiArgs& ea, hipStream_t st) {
  const int m_tiles = (M + BM - 1) / BM, n_tiles = N / 128;
  SplitArgs none{1, nullptr, nullptr, nullptr, nullptr, nullptr, 0};
  hipLaunchKernelGGL((prefill_gemm_kernel<BM, 128, EPI, NORM, false, 2>), dim3(m_tiles * n_tiles), dim3(NT), 0, st,
                     (const bf16x8*)Wt, (const bf16*)X, ldx, M, K, m_tiles, n_tiles, up_off, out, ldo, eps, ea, none);
  return (int)hipGetLastError();
}

template <int EPI, bool NORM>
int launch_tile(int tile, const void* Wt, const void* X, int ldx, int M, int K, int N, int up_off,
                void* out, int ldo, float eps, const EpiArgs& ea, hipStream_t st) {
  switch (tile) {
    case 1: return launch<256, 256, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 2: return launch<128, 256, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 3: return launch<128, 128, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 4: return launch<64, 128, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 5: return launch<64, 256, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 6: return launch_pairs<128, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 7:
      if constexpr (EPI != EPI_RESID)   // (a residual read ahead leaves registers for one workgroup)
        if (g_splitk <= 1 && ((EPI == EPI_SILU && K <= 832) || (long)((M + 191) / 192) * (N / 128) > cu_count()))
          return launch_pairs<192, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
      return launch<192, 128, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 8: return launch<192, 256, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case 9:
      if constexpr (EPI != EPI_SILU)
        return launch<128, 192, EPI, NORM>(Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
  }
  return (int)hipErrorInvalidValue;
}

// Whether launch_tile has this tile for N columns with this epilogue (128 x 192 is not built for SwiGLU)
static bool tile_fits(int tile, int N, int epi) {
  static const int columns[] = {0, 256, 256, 128, 128, 256, 128, 128, 256, 192};
  return tile >= 1 && tile <= 9 && N % columns[tile] == 0 && (tile != 9 || epi != EPI_SILU);
}

// The tile of a shape, 0 where N does not divide.  M <= 64
// uses the 64-row tiles (no MFMA work or DMA on padding rows beyond one tile).  128-row tiles read ahead of their products
// (prefill_gemm_kernel).  What is left there is a wait for all wavefronts per 64 numbers of K, and a clock of 1.9 GHz.
static int g_tile8 = 1;  // the 192 x 256 gate_up picks below (A/B switch: p2p_prefill_tile8)
static int pick_tile(int M, int N, int K, int epi) {
  if (N % 128) return 0;
  if (M <= 64) return 4;
  const int cus = cu_count() > 0 ? cu_count() : 256;
  auto tiles = [&](int bm, int bn) { return (long)((M + bm - 1) / bm) * (N / bn); };
  // (one-m-tile 384 / 448-row tiles for 321-448 rows measured 1.1-1.3x SLOWER than the
  // 128x128 split-K / 256x256 picks of that time and were removed:
  // profiles/r3_prefill_tiles_384_448.jsonl)
  const long small = tiles(128, 128);
  const bool resid = epi == EPI_RESID;
  if (small <= cus) {
    // One round of 128 x 128 tiles, K cut where they leave CUs idle.  128 x 256 tiles copy a quarter less per product and
    // take twice the slices: they pay where a slice keeps 2048 numbers and four slices fill the chip.  Residual, us,
    // 128 x 128 / 128 x 256: 4096 x 14336, 300, 398, 512, 1024 rows 62 / 57, 66 / 61, 76 / 65, 126 / 111 (1080 TFLOP/s);
    // 4096 x 8192, 398 and 1024 rows 43 / 42, 73 / 71; eight slices: 4096 x 14336, 72 and 128 rows 33 / 39, 34 / 42;
    // 4096 x 4096, 1024 rows 40 / 44.  192 x 128 where its slices fill the chip and those of 128 x 256 leave a quarter of it idle
    // (128 x 256 / 192 x 128, 4096 x 14336, 300, 350, 580, 700, 768 rows 57 / 52, 61 / 55, 96 / 84, 99 / 89, 104 / 93, 4096 x 8192,
    // 700 rows 65 / 57).  The lengths between 6144 and 8191 were measured later and say the same, the line does not yet: 4096 x
    // 6144, 580, 700, 768 rows 49 / 45, 50 / 47, 52 / 48, 4096 x 7168 56 / 50, 57 / 52, 59 / 54
    const long wide = N % 256 == 0 ? tiles(128, 256) : 0;
    if (!(wide * 8 > cus && K >= 6144 && K >= (wide * 4 > cus ? 2 : 4) * 2048 && wide <= cus)) return 3;
    auto blocks = [&](long t) {   // with the slices that launch() cuts K into
      long k = 1;
      while (k * 2 <= std::min<long>(std::min<long>(8, cus / t), K / BK / 16)) k *= 2;
      return t * k;
    };
    const long tall = tiles(192, 128);
    return K >= 8192 && tall <= cus && blocks(wide) * 4 <= cus * 3l && blocks(tall) * 8 > cus * 7l ? 7 : 2;
  }
  if (N >= 16384 && M > 128 && M <= 192) return 7;   // one row of tiles, 192 x 128: SwiGLU 28672 x 4096 60 us, 128 x 128 80
  // A residual product with a short K that gives 160 tiles of 256 x 256 and more waits for its residual and its first and last
  // stages: pairs of workgroups per CU hide that, but where the larger tiles' last round fills the CUs and K gives them time.
  // The line was drawn when tiles loaded the residual behind their products (us, pairs / 128 x 256 / 256 x 256: 8192 x 1024, 2048
  // rows 59 / 68 / 62, 8192 x 3072, 2048 rows 115 / 117 / 110, 1500 rows 93 / 106 / 104, 6144 x 2048, 4096 rows 124 / 131 / 160).
  // They load it before them now, and the larger ones have gained more: 44 / 46 / 40, 110 / 99 / 87, 94 / 89 / 76, 113 / 104 / 112
  if (resid && K <= 3072 && N % 256 == 0 && tiles(256, 256) >= 160) {
    const long last = tiles(256, 256) % cus;
    return K >= 2560 && (last == 0 || last * 6 > cus * 5) ? 1 : 6;
  }
  if (N % 256 == 0 && !(resid && K <= 3072)) {
    // More than a round of 128 x 128: the tile whose rounds of the CUs take the shortest time.  The relative times of a round are
    // from SwiGLU of 16384 to 36864 columns and K = 2048 and 4096 on kernels of which 256 x 256 and 192 x 256 have become 10 %
    // faster; what they pick is the best, or 1 % from it, on these too.  us with norm, 256 x 256 / 192 x 256 / 128 x 256 / 192 x
    // 128 at K = 4096: 28672 columns, 250 rows 125 / 93 / 69 / 97, 300 rows 101 / 93 / 111 / 96, 398 rows 104 / 159 / 114 / 147,
    // 512 rows 104 / 164 / 122 / 148, 600 rows 183 / 168 / 168 / 178, 1024 rows 201 / 242 / 229 / 264; 22016 columns, 300 rows
    // 94 / 129 / 101 / 90, 600 rows 169 / 159 / 116 / 144; 36864 columns, 300 rows 180 / 166 / 117 / 146; 12288 x 2048, 400 rows
    // 56 / 71 / 33 / 45, 700 rows 92 / 91 / 59 / 50.  128 x 192, without SwiGLU: 6144 x 4096, 700 rows 48, 128 x 256 54, 192 x
    // 128 48.  192 x 256 from 200 tiles: launch() cuts K below; 256 x 256 from 160 tiles.
    auto time = [&](int bm, int bn, int round) { return (tiles(bm, bn) + cus - 1) / cus * round; };
    int best = 2;
    long t = time(128, 256, 57);
    auto take = [&](int tile, long other) {
      if (other < t) t = other, best = tile;
    };
    take(7, time(192, 128, 44));
    if (tile_fits(9, N, epi) && !(resid && K <= 1024)) take(9, time(128, 192, 43));
    if (g_tile8 && tiles(192, 256) > 200) take(8, time(192, 256, 87));
    if (tiles(256, 256) >= 160) take(1, time(256, 256, 103));
    return best;
  }
  // 128 x 128 takes more than one round, a workgroup per CU: a larger tile that takes one.  us, 128 x 128 / 192 x 128 /
  // 128 x 192: normed 9216 x 4096, 448 rows 71 / 49 / 49; residual 6144 x 2048, 700 rows 37 / 26 / 25
  const bool tall = tiles(192, 128) <= cus;
  if (!(resid && K <= 1024) && tile_fits(9, N, epi) && tiles(128, 192) <= cus) return 9;
  if (tall) return 7;
  // no tile takes one.  Two workgroups on a CU hide what one waits for: the first and the last stages of a short K, and, when
  // the lines were drawn, the reads of the residual, which are ahead of the products now (us then; now: pairs / 128 x 192 / 128 x
  // 256: residual 3072 x 1024, 2048 rows 35 / 37 / 38; 22 / 20 / 21, 11264 x 2368, 456 rows 57 / - / 64; 43 / - / 37, SwiGLU 22016
  // x 4096, 256 rows 95 / - / 91; 78 / - / 64; pairs / 128 x 128: 8320 x 1024, 600 rows 28 / 31; 20 / 23, 8320 x 4096, 600 rows
  // 77 / 72; 61 / 70, residual 86 / 91; 63 / 71); over more rounds 192 x 128 has fewer (192 x 128 / pairs / 128 x 128 now: 10112
  // x 768, 2167 rows 46 / 48 / 61, residual 66 / 53 / 68, 8320 x 4096, 1042 rows 90 / 115 / 101)
  const bool two = small <= 2 * cus;
  if (N % 256 == 0) return resid && two && K <= 3072 ? 6 : 2;
  if (two) return K <= (resid ? 4096 : 1024) ? 6 : 3;
  return resid || K <= 2048 ? 7 : 3;
}

// Per-row RMSNorm statistics for the prefill GEMMs (one wave per row, every 16-byte load
// of the row issued before the first use): rstd[m] = rsqrt(mean_k X[m,k]^2 + eps).  Run
// once per normed projection instead of inside every n-tile's k loop.
static __global__ __launch_bounds__(256) void row_rstd_kernel(const bf16* __restrict__ X, int ldx, int M,
                                                       int K, float eps, float* __restrict__ out) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const bf16x8* p = reinterpret_cast<const bf16x8*>(X + (size_t)row * ldx);
  const int nv = K / 8;
  float s = 0.f;
  for (int c0 = 0; c0 < nv; c0 += 64 * 16) {
    bf16x8 v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int c = c0 + 64 * j + lane;
      v[j] = c < nv ? p[c] : zero_bf16x8();
    }
#pragma unroll
    for (int j = 0; j < 16; ++j)
      s = sumsq8(v[j], s);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) out[row] = rsqrtf(s / (float)K + eps);
}

// rstd workspace: grow-only like the split-K workspace (a captured graph keeps its address);
// never grown while capturing (the GEMM then keeps the in-loop sums)
static SplitWs g_rstd_ws;
static int g_pre_rstd = 1;  // 0: always in-loop sums (A/B)
static const float* pre_rstd(const void* X, int ldx, int M, int K, float eps, hipStream_t st) {
  if (!g_pre_rstd || M < 128 || (ldx % 8) || (K % 8) || ((uintptr_t)X % 16)) return nullptr;
  const size_t bytes = (size_t)M * sizeof(float);
  if (g_rstd_ws.bytes < bytes) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(st, &cs);
    if (cs != hipStreamCaptureStatusNone) return nullptr;
    void* buf = nullptr;
    const size_t want = std::max(bytes, 2 * g_rstd_ws.bytes);
    if (hipMalloc(&buf, want) != hipSuccess) return nullptr;
    g_rstd_ws.buf = buf;  // the old buffer stays allocated (see split_ws)
    g_rstd_ws.bytes = want;
  }
  float* out = (float*)g_rstd_ws.buf;
  hipLaunchKernelGGL(row_rstd_kernel, dim3((M + 3) / 4), dim3(256), 0, st, (const bf16*)X, ldx, M,
                     K, eps, out);
  return hipGetLastError() == hipSuccess ? out : nullptr;
}

}  // namespace pgemm

#ifndef PGEMM_NO_DISPATCH  // (wide_gemm.hip uses the split-K helpers only)
static int g_prefill_tile = 0;  // 0 = heuristic (benchmarks can force 1..3)

// Used by the p2p_tiled_gemm* entry points (tiled_gemm.hip).  Returns
// hipErrorInvalidValue if the shape does not tile (caller falls back).
static int prefill_dispatch(const void* Wt, const void* X, int ldx, int M, int K, int N, int epi,
                         int norm, void* out, int ldo, float eps, const EpiArgs& ea,
                         hipStream_t st) {
  using namespace pgemm;
  if (M <= 0 || K % BK) return (int)hipErrorInvalidValue;
  const int tile = g_prefill_tile ? g_prefill_tile : pick_tile(M, N, K, epi);
  if (!tile_fits(tile, N, epi)) return (int)hipErrorInvalidValue;
  const int up_off = (epi == EPI_SILU) ? N / 32 : 0;
  // normed projections from 128 rows: rstd by row_rstd_kernel, GEMM without in-loop sums
  if (norm) {
    if (const float* r = pre_rstd(X, ldx, M, K, eps, st)) {
      EpiArgs e2 = ea;
      e2.rstd_in = r;
      switch (epi) {
        case EPI_STORE: return launch_tile<EPI_STORE, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, e2, st);
        case EPI_SILU: return launch_tile<EPI_SILU, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, e2, st);
        case EPI_F32: return launch_tile<EPI_F32, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, e2, st);
        case EPI_QKV_ROPE: return launch_tile<EPI_QKV_ROPE, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, e2, st);
        case EPI_ARGMAX: return launch_tile<EPI_ARGMAX, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, e2, st);
      }
    }
  }
  switch (epi) {
    case EPI_STORE:
      return norm ? launch_tile<EPI_STORE, true>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st)
                  : launch_tile<EPI_STORE, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case EPI_RESID:
      return launch_tile<EPI_RESID, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case EPI_SILU:
      return launch_tile<EPI_SILU, true>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case EPI_F32:
      return norm ? launch_tile<EPI_F32, true>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st)
                  : launch_tile<EPI_F32, false>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case EPI_QKV_ROPE:
      return launch_tile<EPI_QKV_ROPE, true>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
    case EPI_ARGMAX:
      return launch_tile<EPI_ARGMAX, true>(tile, Wt, X, ldx, M, K, N, up_off, out, ldo, eps, ea, st);
  }
  return (int)hipErrorInvalidValue;
}
#endif  // PGEMM_NO_DISPATCH
