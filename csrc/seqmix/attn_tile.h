// Pieces of the attention kernels that stage key tiles in LDS for several wavefronts.
//
// A tile's rows go from the paged pool straight into LDS (16 bytes per lane, no registers) while
// the tile before it is being used.  The copy is written as inline asm: with the builtin the
// compiler cannot tell which LDS bytes a pending copy writes and waits for all of them before
// every LDS read.  Nothing in a register depends on it; the kernel's own wait (tile_wait) and a
// barrier stand between a copy and the first read of what it brought.
//
// Rows are stored without padding (a copy's 64 lanes write 1 KiB in a row), their 16-byte pieces
// permuted by swz() so that both kinds of reads spread over the banks: 16 rows x one piece (the
// first product's operand) and 16 keys x 32 bytes (the second product's, read transposed).
#pragma once
#include "common.h"

namespace sm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// Lane i's 16 bytes land at LDS byte address l + 16 * i (l the same for the whole wavefront); they come
// from g, or from the common address g at a byte offset per lane (below 2 GiB).
__device__ __forceinline__ void copy_lds16(const void* g, unsigned l) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(l)
               : "memory", "m0");
}
__device__ __forceinline__ void copy_lds16_at(const void* g, int at, unsigned l) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0" ::"s"(g), "v"(at), "s"(l)
               : "memory", "m0");
}
// The same to LDS byte address l + ON + 16 * i
template <int ON>
__device__ __forceinline__ void copy_lds16_on(const void* g, int at, unsigned l) {
  asm volatile("s_add_u32 m0, %2, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %0" ::"s"(g), "v"(at), "s"(l), "n"(ON)
               : "memory", "m0", "scc");
}
#pragma clang diagnostic pop

__device__ __forceinline__ unsigned lds_address(const void* p) {
  return __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p);
}
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// What is computed from x after this is computed after this: keeps a loop's addresses out of registers
// that its accumulators need.
__device__ __forceinline__ void again(int& x) { asm volatile("" : "+v"(x)); }

typedef float f32x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ bf16x8 to_bf16(f32x8 v) { return __builtin_convertvector(v, bf16x8); }

// every copy this wavefront has issued has landed
__device__ __forceinline__ void tile_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// which piece of row r a place holds (and the other way round), `mask` + 1 pieces per row or 16
__device__ __forceinline__ int swz(int r, int mask) { return (((r & 7) << 1) | ((r >> 3) & 1)) & mask; }

// A place for block blockIdx.x in a list that goes from the longest work to the shortest: every other
// 256 blocks (one per CU) in reverse, so that a CU's second block is short where its first was long.
__device__ __forceinline__ int folded_block() {
  const int b = blockIdx.x, c = b >> 8;
  return (c & 1) && (c + 1) << 8 <= (int)gridDim.x ? (c << 8) + 255 - (b & 255) : b;
}

// B operand of a 16x16x32 product from a [key][channel] tile, keys in the order of the P operand
// (slot quad * 8 + i is key quad * 4 + i for i < 4, 16 + quad * 4 + i - 4 after that), columns c0 ..
// c0 + 15.  ds_read_b64_tr_b16: within 16 lanes, lane L names row L / 4, channels (L % 4) * 4 ..; lane
// i receives channel i of the four rows.
template <int PIECES>
__device__ __forceinline__ bf16x8 read_keys_by_channel(const unsigned short* tile, int key0, int c0, int lane) {
  const int L = lane & 15, quad = lane >> 4;
  constexpr int MASK = PIECES < 16 ? PIECES - 1 : 15;
  const int k = key0 + quad * 4 + (L >> 2), c = c0 + (L & 3) * 4;
  typedef __attribute__((address_space(3))) s16x4* lds_t;
  const unsigned short* lo = tile + ((k * PIECES + ((c >> 3) ^ swz(k, MASK))) << 3) + (c & 7);
  // sixteen keys on: the same permutation
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)lo);
  const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(lo + 16 * PIECES * 8));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// A place out of a row's sight has weight zero, but 0 * inf is nan: through the tiles' products a value that is not finite
// reaches rows of the group that do not see it.  Groups whose sums are not finite are therefore done again pair by pair,
// by a wavefront each, over the places that the pair's row sees.  Slow and rare; it stands behind the tile loop, whose
// registers it must not take (a second walk through the tiles cost 13 % by its spills).
// z: 0 while all numbers are finite, then nan
__device__ __forceinline__ void not_finite(f32x4 v, float& z) {
#pragma unroll
  for (int e = 0; e < 4; e++) z = fmaf(v[e], 0.0f, z);
}

template <typename T>
__device__ __forceinline__ float wave_dot(const T* x, const T* y, int n) {
  float s = 0.0f;
  for (int c = threadIdx.x & 63; c < n; c += 64) s = fmaf(ldf(x, c), ldf(y, c), s);
  return wave_sum(s);
}

// softmax sums of one pair; a lane has every 64th channel
template <int NC>
struct PairSums {
  float m, l, o[NC];
  __device__ __forceinline__ void begin(float sink, bool sunk) {   // natural units
    m = sunk ? sink : -1e30f;
    l = sunk ? 1.0f : 0.0f;
#pragma unroll
    for (int t = 0; t < NC; t++) o[t] = 0.0f;
  }
  template <typename T>
  __device__ __forceinline__ void add(float s, const T* v, int V) {
    const float up = fmaxf(m, s), f = m == up ? 1.0f : expf(m - up), w = expf(s - up);
    m = up;
    l = l * f + w;
#pragma unroll
    for (int t = 0; t < NC; t++) {
      const int c = t * 64 + (threadIdx.x & 63);
      o[t] = c < V ? o[t] * f + w * ldf(v, c) : 0.0f;
    }
  }
};

}  // namespace sm
