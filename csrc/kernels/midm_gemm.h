// Mid-M GEMM (1 < M <= 64 rows: chat-length prompts, batched decode), the WHOLE K of NG x 16 columns (SwiGLU: of the
// gate and up columns) per workgroup, one workgroup per CU.
//
//   out[m, 16 g + r] = epilogue( rstd[m] * sum_k X[m, k] * W[16 g + r, k] )
//
// Beside wide_gemm.hip, which shares the activations among 128 columns and therefore cuts K over workgroups where a
// projection has few columns (its slices meet through memory, 5 to 6 us a launch): here nothing meets across workgroups,
// and every workgroup reads all of X.  That is cheap where X comes in whole lines: what bounds a CU's intake is the
// number of 128-byte lines its load instructions touch, and 1 KiB as 8 rows x 128 bytes comes in at 95 to 100 KB/us,
// as the 16 rows x 64 bytes of an MFMA fragment at 58 KB/us (LDS copies, 256 workgroups, rows of 14336 numbers; weights
// contiguous).
//
// Eight wavefronts; wavefront w takes chunks w, w + 8, .. of 64 numbers of K and works alone until the end: its own ring
// of D chunks of X in LDS (copies of 8 rows x 128 bytes; 16-byte piece p of row R lies at p ^ (R & 7), so the fragments
// are read without bank conflicts) and its weight fragments (fragment-major in HBM, read once, non-temporal) straight
// in registers, D chunks ahead.  D fills LDS: 144 KiB of activations and 48 KiB of weights in flight per CU at 48 rows.
// The eight partial tiles meet in LDS; RMSNorm's sums of squares ride on the fragments.
//
// Cold weights, us, 32, 48 and 64 rows, wide kernel / this: qkv of llama3.1-8B with norm and rotation (6144 x 4096,
// NG 2) 16.9 / 15.0, 19.0 / 16.5, 20.0 / 18.3; its output product (4096 x 4096, NG 1) 12.6 / 11.5, 14.2 / 13.8, 15.9 /
// 14.9; 8192 x 1024, 48 rows 12.0 / 8.3, 8192 x 3584 19.8 / 15.8.  Long K stays with the wide kernel (4096 x 14336
// 27.4 / 31.6, 28.4 / 36.6, 30.2 / 41.8): X is then three times the workgroup's weights.  Four wavefronts that met at a
// barrier per chunk of 128 numbers, with copies of 16 rows x 64 bytes, had 17.6, 21 and 24 for that qkv.
#pragma once
#include "gemm_epilogue.h"
#include "lds_pipe.h"

namespace midm {

constexpr int NW = 8;        // wavefronts
constexpr int NT = NW * 64;
constexpr int KC = 64;       // numbers of K per chunk: a line of a row
// chunks in flight per wavefront: 2 KiB of X per 16 rows and chunk, 160 KiB of LDS for 8 wavefronts; at most 6 (registers)
template <int MT>
constexpr int depth() { return 10 / MT > 6 ? 6 : 10 / MT; }

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
template <int PER, int MAX>
__device__ __forceinline__ void wait_chunks(int pending) {   // at most `pending` (<= MAX) chunks of PER loads in flight
  if constexpr (MAX > 0) {
    if (pending < MAX) return wait_chunks<PER, MAX - 1>(pending);
  }
  wait_vmcnt<MAX * PER>();
}

// The weight fragments of a chunk, as asm for the reason that lds_pipe.h gives; none goes out for c >= n (the branch
// is inside the asm: around it the compiler would copy registers whose loads are in flight)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_pair(bf16x8& a, bf16x8& b, const bf16x8* p, int c, int n) {
  asm volatile(
      "s_cmp_lt_i32 %3, %4\n\ts_cbranch_scc0 1f\n\t"
      "global_load_dwordx4 %0, %2, off nt\n\tglobal_load_dwordx4 %1, %2, off offset:1024 nt\n1:"
      : "=&v"(a), "=&v"(b)
      : "v"(p), "s"(c), "s"(n)
      : "scc");
}
#pragma clang diagnostic pop

template <int MT, int EPI, bool NORM, int NG>
__global__ __launch_bounds__(NT, 2) void midm_kernel(const bf16x8* __restrict__ Wt,
                                                     const bf16* __restrict__ X, int ldx, int M,
                                                     int K, int groups, int up_off, void* __restrict__ out,
                                                     int ldo, float eps, EpiArgs ea) {
  constexpr int NB = EPI == EPI_SILU ? 2 : 1;
  constexpr int NF = NB * NG;                 // column fragments
  constexpr int D = depth<MT>();
  constexpr int PER = 2 * MT + 2 * NF;        // loads of a wavefront per chunk
  constexpr int SLOT = MT * 2 * 64;           // bf16x8 per ring slot
  constexpr int RING = NW * D * SLOT, RED = (NW * NF * MT * 4 * 64 + NW * MT * 16) / 4;
  __shared__ __attribute__((aligned(16))) bf16x8 lds[RING > RED ? RING : RED];

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g0 = blockIdx.x * NG;
  const int S = K >> 5;                       // k-steps
  const int chunks = K / KC, n = (chunks - w + NW - 1) / NW;   // this wavefront's

  const bf16* asrc[2 * MT];                   // 8 rows each
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) {
    const int row = min(8 * i + (lane >> 3), M - 1);
    asrc[i] = X + (size_t)row * ldx + w * KC + 8 * ((lane & 7) ^ (lane >> 3));
  }
  const bf16x8* wsrc[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int g = min(g0 + f / NB, groups - 1) + (f % NB) * up_off;
    wsrc[f] = Wt + ((size_t)g * S + 2 * w) * 64 + lane;
  }
  bf16x8* ring = lds + w * D * SLOT;
  auto issue_x = [&](int c, int slot) {
    if (c < n) {
#pragma unroll
      for (int i = 0; i < 2 * MT; ++i) ldsp::dma_lds<16>(asrc[i] + (size_t)c * (NW * KC), ring + slot * SLOT + i * 64);
    }
  };
  auto issue_w = [&](int c, bf16x8(&wr)[2 * NF]) {
#pragma unroll
    for (int f = 0; f < NF; ++f) load_pair(wr[2 * f], wr[2 * f + 1], wsrc[f] + (size_t)min(c, n - 1) * (NW * 2 * 64), c, n);
  };

  f32x4 acc[NF][MT];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[f][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) ss[mt] = 0.f;

  const int r = lane & 15, q = lane >> 4;
  const int at0 = r * 8 + (q ^ (r & 7)), at1 = r * 8 + ((4 + q) ^ (r & 7));
  bf16x8 wr[D][2 * NF];
  if (n > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      issue_x(d, d);
      issue_w(d, wr[d]);
    }
  }
  for (int tb = 0; tb < n; tb += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int t = tb + d;
      if (t >= n) break;
      wait_chunks<PER, D - 1>(min(D - 1, n - 1 - t));
#pragma unroll
      for (int k = 0; k < 2 * NF; ++k) asm volatile("" : "+v"(wr[d][k]));   // landed
      const bf16x8* st = ring + d * SLOT;
      bf16x8 a[2 * MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        a[2 * mt] = ldsp::lds_rd(st + mt * 128 + at0);
        a[2 * mt + 1] = ldsp::lds_rd(st + mt * 128 + at1);
      }
      ldsp::lds_wait(a);
      issue_x(t + D, d);      // the slot's fragments are in registers
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
          for (int f = 0; f < NF; ++f)
            acc[f][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2 * mt + ks], wr[d][2 * f + ks], acc[f][mt], 0, 0, 0);
          if constexpr (NORM) ss[mt] = sumsq8(a[2 * mt + ks], ss[mt]);
        }
      issue_w(t + D, wr[d]);
    }
  }
  wait_vmcnt<0>();
  __syncthreads();  // every wavefront is done with its ring: LDS becomes the reduction buffer

  // ---- the eight partial tiles; wavefront w finishes fragments w, w + 8, .. of (unit, m-tile) ----
  float* red = reinterpret_cast<float*>(lds);  // [NW][NF][MT][4][64]
  float* red_ss = red + NW * NF * MT * 4 * 64; // [NW][MT][16]
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[(((w * NF + f) * MT + mt) * 4 + j) * 64 + lane] = acc[f][mt][j];
  if constexpr (NORM) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float v = ss[mt];
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lane < 16) red_ss[(w * MT + mt) * 16 + lane] = v;
    }
  }
  __syncthreads();
  for (int unit = w; unit < NG * MT; unit += NW) {
    const int u = unit / MT, mt = unit % MT, g = g0 + u;
    if (g >= groups) continue;
    float tot[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) v += red[(((ww * NF + u * NB + b) * MT + mt) * 4 + j) * 64 + lane];
        tot[b][j] = v;
      }
    // epilogue operands of the 4 rows as one batch (residual values / rows' KV slot and
    // (cos, sin)): loaded per element between the stores they were 4 dependent round trips
    float resv[4];
    float2 csv[4];
    int slotv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = 16 * mt + 4 * q + j;
      resv[j] = 0.f;
      csv[j] = float2{1.f, 0.f};
      slotv[j] = -1;
      if constexpr (EPI == EPI_RESID)
        if (m < M) resv[j] = (float)reinterpret_cast<const bf16*>(out)[(size_t)m * ldo + g * 16 + r];
      if constexpr (EPI == EPI_QKV_ROPE) {
        if (m < M) {
          const int kk = g & 7;
          const int dd = ((r < 8) ? 8 * kk + r : 64 + 8 * kk + (r - 8)) & 63;
          csv[j] = ea.cs[(size_t)ea.pos[m] * 64 + dd];
          slotv[j] = ea.slots[m];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = 16 * mt + 4 * q + j;
      const bool valid = m < M;
      float scale = 1.f;
      if constexpr (NORM) {
        float t2 = 0.f;
#pragma unroll
        for (int ww = 0; ww < NW; ++ww) t2 += red_ss[(ww * MT + mt) * 16 + 4 * q + j];
        scale = rsqrtf(t2 / (float)K + eps);
      }
      if constexpr (EPI == EPI_QKV_ROPE) {
        epi_store<EPI>(m, valid, g, r, tot[0][j] * scale, 0.f, out, ldo, ea, csv[j], slotv[j]);
      } else if constexpr (EPI == EPI_RESID) {
        if (valid)
          reinterpret_cast<bf16*>(out)[(size_t)m * ldo + g * 16 + r] = f2bf(resv[j] + tot[0][j] * scale);
      } else {
        epi_store<EPI>(m, valid, g, r, tot[0][j] * scale, tot[NB - 1][j] * scale, out, ldo, ea);
      }
    }
  }
}

template <int MT, int EPI, bool NORM>
int launch_mt(const void* Wt, const void* X, int ldx, int M, int K, int groups, int up_off,
              void* out, int ldo, float eps, const EpiArgs& ea, hipStream_t st, int cus) {
  constexpr int NB = EPI == EPI_SILU ? 2 : 1;
  // one or two units per workgroup: rounds of the CUs times the lines of a round (X, then the columns)
  auto cost = [&](int ng) { return (((groups + ng - 1) / ng + cus - 1) / cus) * (MT + NB * ng); };
  if (cost(2) < cost(1))
    hipLaunchKernelGGL((midm_kernel<MT, EPI, NORM, 2>), dim3((groups + 1) / 2), dim3(NT), 0, st,
                       (const bf16x8*)Wt, (const bf16*)X, ldx, M, K, groups, up_off, out, ldo, eps, ea);
  else
    hipLaunchKernelGGL((midm_kernel<MT, EPI, NORM, 1>), dim3(groups), dim3(NT), 0, st,
                       (const bf16x8*)Wt, (const bf16*)X, ldx, M, K, groups, up_off, out, ldo, eps, ea);
  return (int)hipGetLastError();
}

static int cu_count() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (!cached[dev]) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

// M <= 64 rows, K % 128 == 0; groups = column groups (SwiGLU: gate/up pairs).
template <int EPI, bool NORM>
int launch(const void* Wt, const void* X, int ldx, int M, int K, int groups, int up_off,
           void* out, int ldo, float eps, const EpiArgs& ea, hipStream_t st) {
  if (M <= 0 || M > 64 || K % 128 != 0) return (int)hipErrorInvalidValue;
  const int cus = cu_count();
  switch ((M + 15) / 16) {
    case 1: return launch_mt<1, EPI, NORM>(Wt, X, ldx, M, K, groups, up_off, out, ldo, eps, ea, st, cus);
    case 2: return launch_mt<2, EPI, NORM>(Wt, X, ldx, M, K, groups, up_off, out, ldo, eps, ea, st, cus);
    case 3: return launch_mt<3, EPI, NORM>(Wt, X, ldx, M, K, groups, up_off, out, ldo, eps, ea, st, cus);
    case 4: return launch_mt<4, EPI, NORM>(Wt, X, ldx, M, K, groups, up_off, out, ldo, eps, ea, st, cus);
  }
  return (int)hipErrorInvalidValue;
}

}  // namespace midm
