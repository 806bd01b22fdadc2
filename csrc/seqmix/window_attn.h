// What the two matrix-core window attention kernels (window_attn_mfma.hip, window_attn_tile.hip) share.
#pragma once
#include "common.h"

enum { KEYS_WINDOW = 0, KEYS_BLOCKS = 1, KEYS_KEPT = 2 };

struct WindowArgs {
  const sm::bf16* q;
  int ldq;
  const sm::bf16* pool;
  const int* bt;
  int max_pages;
  const int *row_ent, *pos, *units;
  int U;
  const float* sink;
  float scale;
  int win;
  sm::bf16* out;
  int ldo, H, G, D, V, page, HS, splits;
  float* part;
  float out_scale, cap;
  const float *r1, *r2;
  const sm::bf16* gate;
  int ldg, gate_pc;
  const sm::bf16* blk;
  int P, keep;
  float lam, eps;
};

inline int window_pad32(int n) {   // 32-channel steps the kernels are instantiated for
  const int s = (n + 31) / 32;
  return s <= 1 ? 1 : s <= 2 ? 2 : s <= 4 ? 4 : 8;
}

// What prompt_attn_k takes beside it (prompt_attn.hip)
struct PromptArgs {
  WindowArgs w;
  int qhs;                        // between the queries of two heads
  const sm::bf16* qrot;           // [rows, H * Rd] rotated query parts
  int ldqr;
  const sm::bf16* kv;             // keys and values formed for the step
  int ldkv;
  const int* kbase;
  int kstride;
  int ldr, rot0, Rd;              // rows of the pool, where the rotated key part stands in them, its channels
  int gate_wide, out_wide;        // four numbers at once
};
// (row, head) pairs of its workgroups
#define PROMPT_PAIRS 64
int prompt_attn_paged(const WindowArgs& w, hipStream_t st);

// (row, head) pairs of a workgroup of window_attn_tile_k
#define WINDOW_TILE_PAIRS 64
int window_attn_tile(const WindowArgs& a, int maps, hipStream_t st);
