// Rows of a bf16 matrix into LDS, swizzled by row: 16-byte chunk c of row rr at
// chunk c ^ (rr % 16), so the 16 rows that a 16-lane group of an MFMA A operand
// reads fall on 16 distinct bank groups.
#pragma once
#include "common.hpp"

namespace spk {

// Wave w of WAVES takes rows w, w + WAVES, ... of the LDS tile's `rows`; row rr comes
// from row_of(rr) of x if take(rr), both wave-uniform (rows past the batch are left
// as they are: nobody reads their products).  chunks: 16-byte chunks per row, a
// multiple of 16, so the swizzle stays within a row's whole and partial 64-chunk
// runs and a row costs one address: its loads step by 1 KB.  (One run over all
// chunks of the tile took a division per load.  Long-K linear, 16 rows x 608
// chunks a workgroup: 4 rows 7.1 -> 5.3 us, 64 rows 7.15 -> 6.4, 256 rows 12.2 ->
// 10.9; o projection, 112 chunks a row: 4 rows 3.9 -> 3.5, 64 rows unchanged; 64
// chunks a row, a load each: 64 rows 3.5 -> 3.6.)
template <int WAVES, class Take, class RowOf>
__device__ __forceinline__ void stage_rows(char *smem, const uint16_t *x, int rows, int chunks, int wave, int lane,
                                           Take take, RowOf row_of) {
  const int full = chunks >> 6, rem = chunks & 63;
#pragma unroll 1
  for (int rr = __builtin_amdgcn_readfirstlane(wave); rr < rows; rr += WAVES) {
    if (!take(rr)) continue;
    const uint16_t *src = x + row_of(rr) * (8 * chunks) + 8 * (lane ^ (rr & 15));
    char *dst = smem + rr * chunks * 16;
    for (int i = 0; i < full; ++i)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const void *>(src + 512 * i),
                                       (__attribute__((address_space(3))) void *)(dst + 1024 * i), 16, 0, 0);
    if (lane < rem)
      __builtin_amdgcn_global_load_lds(reinterpret_cast<const void *>(src + 512 * full),
                                       (__attribute__((address_space(3))) void *)(dst + 1024 * full), 16, 0, 0);
  }
}

}  // namespace spk
