// wir_split.h -- what the split attention kernels (attn_splitkv.hip,
// attn_bwd_split.hip) share.
#pragma once
#include "wir_cdna4.h"

namespace wir {

typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

// A split kernel's workgroup takes SPLIT_ROWS rows of one side and divides
// the other side's tiles over its waves.
constexpr int SPLIT_WAVES = 4, SPLIT_ROWS = 32;

// Program -> (block of SPLIT_ROWS rows, head, batch).  Causal launches end on
// the short blocks: the LDS holds one workgroup per CU, so the order sets the
// tail (dK/dV, heads in turn -> this order, B1 H4 S4096 D64 52.8 -> 40.2 us, H20
// S768 D64 19.1 -> 16.0, H12 S1024 D128 27.2 -> 24.3, H8 S2048 D64 25.1 -> 25.0).
template <bool CAUSAL, bool REVERSE>
__device__ __forceinline__ void split_program(int& x, int& h, int& b) {
  const int nx = gridDim.x, ny = gridDim.y, heads = ny * gridDim.z;
  const int hw = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
  int head;
  if (CAUSAL) {
    longest_first<REVERSE, 2048>(hw, nx, heads, x, head);
  } else {
    const int id = remap_xcd(hw, nx * heads);
    x = id % nx;
    head = id / nx;
  }
  h = head % ny;
  b = head / ny;
}

// Floats per row of a wave's partial result in LDS: 16 rows land in 16
// different 16-byte bank slots.
template <int D>
constexpr int split_pitch = D + 4;

// The wave's partial result -> part[wave][row][column].
template <int D>
__device__ __forceinline__ void put_partial(lds_float* part, const RTile<32, 32, D>& t, int wave) {
  const int lane = lane_id(), lr = lane % 32, lh = lane / 32;
#pragma unroll
  for (int cb = 0; cb < D / 32; ++cb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = t.f[cb][0][4 * g + j];
      *(lds_f32x4*)(part + (wave * SPLIT_ROWS + lr) * split_pitch<D> + cb * 32 + ccol<32>(4 * g, lh)) = v;
    }
}

// Rows row0.. (SPLIT_ROWS of them) of (b, d) of a bf16 global, D columns,
// written in 16-byte chunks with the bounds of store_tile_staged: elements
// outside the tensor are dropped in every dimension (the grid and its batch
// and head ids come from Q's shape, which the destination's need not match),
// and rows that are not 16-byte aligned (the host checks the row stride, not
// the batch and head strides) take single stores.  `whole`, the same for all
// lanes, skips the checks.  Forward, us, stores without bounds / a test per
// chunk / this: B1 H8 S512 D64 5.79 / 5.99 / 5.87, D128 9.3 / - / 9.45.
struct RowStore {
  bf16* base;
  int row0;
  bool in, whole;

  __device__ __forceinline__ RowStore() {}
  __device__ __forceinline__ RowStore(const gl<bf16>& g, int b, int d, int row0_, int cols) : row0(row0_) {
    base = g.data + (long long)b * g.sb + (long long)d * g.sd;
    in = (unsigned)b < (unsigned)g.b && (unsigned)d < (unsigned)g.d;
    whole = in && row0 + SPLIT_ROWS <= g.r && cols <= g.c && (g.sr & 7) == 0 && ((size_t)base & 15) == 0;
  }

  // v -> columns col.. (a multiple of 8) of row row0 + row
  __device__ __forceinline__ void put8(const gl<bf16>& g, int row, int col, const bf16x8& v) const {
    bf16* p = base + (long long)(row0 + row) * g.sr + col;
    if (whole) {
      *(bf16x8*)p = v;
    } else if (in && row0 + row < g.r) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (col + j < g.c) p[j] = v[j];
    }
  }
};

}  // namespace wir

#define WIR_SPLIT_KERNEL(NAME, ARGS, CALL)                                                                     \
  extern "C" __global__ void __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(1, 1))) \
  NAME(const ARGS args) {                                                                                      \
    CALL(args);                                                                                                \
  }
