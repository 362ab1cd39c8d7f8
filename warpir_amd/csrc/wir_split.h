// wir_split.h -- what the split attention kernels (attn_splitkv.hip,
// attn_bwd_split.hip) share.
#pragma once
#include "wir_cdna4.h"

namespace wir {

// Rows of (b, d) of a bf16 global, written in 16-byte chunks with the bounds
// of store_tile_staged: elements outside the tensor are dropped in every
// dimension (the grid and its batch and head ids come from Q's shape, which
// the destination's need not match), and rows that are not 16-byte aligned
// (the host checks the row stride, not the batch and head strides) take
// single stores.
struct RowStore {
  bf16* base;
  int rows, vec_cols;   // 0 rows: (b, d) is outside

  __device__ __forceinline__ RowStore(const gl<bf16>& g, int b, int d) {
    base = g.data + (long long)b * g.sb + (long long)d * g.sd;
    rows = (unsigned)b < (unsigned)g.b && (unsigned)d < (unsigned)g.d ? g.r : 0;
    vec_cols = (g.sr & 7) == 0 && ((size_t)base & 15) == 0 ? g.c : 0;
  }

  // v -> columns col.. (a multiple of 8) of `row`
  __device__ __forceinline__ void put8(const gl<bf16>& g, int row, int col, const bf16x8& v) const {
    if (row >= rows) return;
    bf16* p = base + (long long)row * g.sr + col;
    if (col + 8 <= vec_cols) {
      *(bf16x8*)p = v;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (col + j < g.c) p[j] = v[j];
    }
  }
};

}  // namespace wir
