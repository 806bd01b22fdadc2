// Products of prompts in fp32 (prompt_gemm.h).  The matrix cores take 16 times as long for a stage as in bf16 and are what bounds
// them from some 250 workgroups on (128 x 128, 4096 x 1024, 2048 rows 134 us, 128 TFLOP/s), so tiles stay small enough to give
// every CU the same.  us, the library's -> this: 1024 x 1024, 17 and 1024 rows 8.3 -> 6.0, 20.2 -> 20.3; 1544 x 1024, 40, 389
// and 2048 rows 8.6 -> 6.3, 16.9 -> 20.1, 78.8 -> 66.2; 1024 x 1536, 778 rows 29.3 -> 27.5; a call of the library's costs 15 us
// more of host time, which steps of few hundred rows wait for.
#include "prompt_gemm.h"

// Fitted to products of 968 to 32000 columns, K 512 to 2048 and 8 to 2048 rows (2 % off; what the rule takes is 0.1 % above the
// best tile on average, 2 % at worst)
static const Tile TILES[] = {
    {32, 16, false, 2.9f, 1.6f, 0.100f, 0.103f}, {32, 32, true, 3.4f, 2.4f, 0.173f, 0.166f},
    {64, 32, true, 4.5f, 2.6f, 0.261f, 0.255f},  {64, 64, true, 4.7f, 3.0f, 0.484f, 0.482f},
    {64, 64, true, 4.2f, 0.4f, 0.533f, 0.492f},  {96, 64, true, 4.4f, 1.1f, 0.742f, 0.691f},
    {64, 96, false, 5.1f, 1.0f, 0.755f, 0.710f}, {128, 64, true, 4.7f, 3.2f, 0.956f, 0.950f},
    {128, 128, true, 6.5f, 4.8f, 1.894f, 1.904f}};

int prompt_gemm_f32(const GemmArgs& a, int tile, hipStream_t st) {
  switch (tile ? tile : pick_tile(TILES, a.M, a.act >= 0 ? 2 * a.N : a.N, (a.K + 31) / 32, a.act >= 0)) {
    case 1: return launch_gemm<float, 32, 16, 1, 1, 4, 4>(a, st);
    case 2: return launch_gemm<float, 32, 32, 1, 1, 4, 4>(a, st);
    case 3: return launch_gemm<float, 64, 32, 2, 1, 4, 3>(a, st);
    case 4: return launch_gemm<float, 64, 64, 2, 2, 2, 3>(a, st);
    case 5: return launch_gemm<float, 64, 64, 4, 2, 1, 4>(a, st);
    case 6: return launch_gemm<float, 96, 64, 2, 2, 2, 2>(a, st);
    case 7: return launch_gemm<float, 64, 96, 2, 2, 1, 3>(a, st);
    case 8: return launch_gemm<float, 128, 64, 4, 2, 1, 4>(a, st);
    case 9: return launch_gemm<float, 128, 128, 2, 4, 1, 4>(a, st);
  }
  return (int)hipErrorInvalidValue;
}
