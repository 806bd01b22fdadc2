// Products of prompts in bf16 (prompt_gemm.h), and the entry for both types.
#include "prompt_gemm.h"

// Fitted to products of 192 to 16384 columns, K 128 to 8192 and 20 to 2644 rows (4 % off at the tiles that win; what the rule takes
// is 0.3 % above the best tile on average, 15 % at worst), weights not in the caches.
static const Tile TILES[] = {
    {32, 16, false, 2.8f, 1.2f, 0.067f, 0.082f},   {32, 32, true, 3.3f, 1.4f, 0.090f, 0.115f},
    {32, 64, true, 3.0f, 1.5f, 0.155f, 0.164f},    {64, 32, true, 3.2f, 1.7f, 0.136f, 0.147f},
    {64, 64, true, 3.2f, 1.6f, 0.192f, 0.222f},    {64, 64, true, 2.7f, 0.7f, 0.243f, 0.189f},
    {128, 64, true, 3.0f, 2.1f, 0.289f, 0.286f},   {128, 128, true, 3.6f, 3.1f, 0.449f, 0.452f},
    {192, 128, true, 5.2f, 2.9f, 0.580f, 0.636f},  {256, 128, true, 7.4f, 3.3f, 0.681f, 0.803f},
    {192, 256, true, 6.9f, 0.0f, 1.055f, 1.264f},  {256, 256, true, 7.9f, 0.0f, 1.278f, 1.498f},
    {192, 192, false, 9.9f, 6.3f, 0.686f, 0.833f}, {256, 192, false, 9.7f, 5.7f, 0.974f, 1.198f}};

extern "C" {

// x: M rows, or with `rows` those of `span` numbers that it names; act < 0: no gated unit; tile: 0 by the rule
int p2p_sm_prompt_gemm(const void* x, const int* rows, long span, int ldx, const void* w, const void* bias, void* out, int ldo, int M,
                       int N, int K, int tanh_from, int act, float limit, float alpha, int tile, int f32, hipStream_t st) {
  if (M <= 0 || N <= 0) return 0;
  const int size = f32 ? 4 : 2, ks = 128 / size;
  if (K < 1 || (K % ks && K != ks / 2) || ldx < 0 || ldx % (16 / size) || (size_t)x % 16 || (size_t)w % 16 || act > 2 || (f32 && tanh_from < N) ||
      (rows ? span * size : (long)ldx * 256 * size) >= 1l << 31 || (long)K * size * (act >= 0 ? N + 256l : 256l) >= 1l << 31)
    return (int)hipErrorInvalidValue;
  // neighbours that a store takes at once
  const int wide = !f32 && ldo % 8 == 0 && N % 8 == 0 && (size_t)out % 16 == 0 ? 8
                   : ldo % 4 == 0 && N % 4 == 0 && (size_t)out % (4 * size) == 0 ? 4 : 0;
  const GemmArgs a = {x, rows, ldx, w, bias, out, ldo, M, N, K, tanh_from, act, limit, alpha, 0, 0, wide};
  if (f32) return prompt_gemm_f32(a, tile, st);
  switch (tile ? tile : pick_tile(TILES, M, act >= 0 ? 2 * N : N, (K + ks - 1) / ks, act >= 0)) {
    case 1: return launch_gemm<bf16, 32, 16, 1, 1, 4, 4>(a, st);
    case 2: return launch_gemm<bf16, 32, 32, 1, 1, 4, 4>(a, st);
    case 3: return launch_gemm<bf16, 32, 64, 1, 2, 2, 4>(a, st);
    case 4: return launch_gemm<bf16, 64, 32, 2, 1, 4, 3>(a, st);
    case 5: return launch_gemm<bf16, 64, 64, 2, 2, 2, 3>(a, st);
    case 6: return launch_gemm<bf16, 64, 64, 2, 2, 1, 4>(a, st);
    case 7: return launch_gemm<bf16, 128, 64, 4, 2, 1, 4>(a, st);
    case 8: return launch_gemm<bf16, 128, 128, 2, 4, 1, 4>(a, st);
    case 9: return launch_gemm<bf16, 192, 128, 2, 4, 1, 3>(a, st);
    case 10: return launch_gemm<bf16, 256, 128, 4, 2, 1, 3>(a, st);
    case 11: return launch_gemm<bf16, 192, 256, 2, 4, 1, 2>(a, st);
    case 12: return launch_gemm<bf16, 256, 256, 2, 4, 1, 2>(a, st);
    case 13: return launch_gemm<bf16, 192, 192, 2, 4, 1, 3>(a, st);
    case 14: return launch_gemm<bf16, 256, 192, 2, 4, 1, 2>(a, st);
  }
  return (int)hipErrorInvalidValue;
}

}  // extern "C"
