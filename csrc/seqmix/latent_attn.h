// What the two matrix-core latent attention kernels (latent_attn_mfma.hip, latent_attn_tile.hip) share.
#pragma once
#include "common.h"

struct LatentArgs {
  const sm::bf16* qa;
  long sqh, sqr;
  const sm::bf16* cache;
  const int* bt;
  int max_pages;
  const int *row_ent, *pos, *units;
  int U;
  const float* sink;
  float scale;
  int win;
  sm::bf16* out;
  long soh, sor;
  int H, rank, page, HS, splits;
  float* part;
};

// (row, head) pairs of a workgroup of latent_attn_tile_k
#define LATENT_TILE_PAIRS 64
// the kernel takes latents (padded to 64, 128, 256 or 512) of more than 32 numbers
int latent_attn_tile(const LatentArgs& a, hipStream_t st);
