// Entries of the token-tile list that the matrix-core grouped GEMM walks (layout: mfma.hip, k_build_tiles).
#pragma once

#include <hip/hip_runtime.h>

namespace xabe {

// Whether the routed launches of a pass take narrow tiles: while an expert's share of it averages at most 48 rows, so that
// most experts are one tile either way (1500 tokens of the routed model, 47 a share: 365 us against 388 wide; 2200, 69: 544
// against 454).
__host__ __device__ inline bool narrow_tiles(size_t tokens, size_t top_k, size_t num_experts) { return tokens * top_k <= 48 * num_experts; }

// The tiles of expert e (`count` selections from slot `base`), the first of them entry `first` of the list: as few as tiles
// of `h` token rows (a multiple of 32) allow, their 32-row blocks shared out evenly, since a tile's time is that of
// its blocks: 264 rows are tiles of 160 and 104, not of 256 and 8.
__device__ __forceinline__ void write_tile_entries(int e, int count, int base, int first, int h, int capacity, int* list) {
  const int nt = (count + h - 1) / h, blocks = (count + 31) / 32;
  for (int i = 0; i < nt; ++i) {
    const int idx = first + i;
    if (idx >= capacity) break;
    const int lo = blocks * i / nt * 32, hi = min(blocks * (i + 1) / nt * 32, count);
    *reinterpret_cast<int4*>(list + 4 + 4 * idx) = make_int4(e, base + lo, hi - lo, 0);
  }
}

}  // namespace xabe
