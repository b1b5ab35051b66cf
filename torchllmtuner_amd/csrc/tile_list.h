// The rows that a plan's tile list names, for kernels that find their rows from the experts' counts.
#pragma once
#include "common.h"

namespace mi355 {
namespace {

constexpr int kListTile = 256;  // rows of a listed tile, mi355_grouped_tile_m

struct TileList {
  const int32_t *expert, *row0, *num;
  int capacity;
  __device__ __forceinline__ int size() const { return min(*(const int32_t __attribute__((address_space(4)))*)num, capacity); }
};

__device__ __forceinline__ int listed_tiles(int count) { return (count + kListTile - 1) / kListTile; }

// Of the `rows` rows from `row0` on, at most 128 of expert e's (`count` from `first` on), those of listed tiles; false: none are.  They are consecutive: only the last
// of an expert's tiles has fewer than 128 rows where it has two or more, so no such run touches three.  For lists that leave tiles out; whole ones need no search.
__device__ __forceinline__ bool listed_rows(const TileList& list, int e, int first, int count, int& row0, int& rows) {
  const int lane = threadIdx.x & 63, n = list.size(), height = even_tile_rows(count, kListTile);
  int from = row0 + rows, to = row0;
  for (int b = 0; b < n; b += 64) {
    const int i = b + lane;
    if (i < n && list.expert[i] == e) {
      const int top = list.row0[i], lo = max(top, row0), hi = min(min(top + height, first + count), row0 + rows);
      if (lo < hi) {
        from = min(from, lo);
        to = max(to, hi);
      }
    }
  }
#pragma unroll
  for (int o = 1; o < 64; o *= 2) {
    from = min(from, __shfl_xor(from, o));
    to = max(to, __shfl_xor(to, o));
  }
  row0 = __builtin_amdgcn_readfirstlane(from);
  rows = __builtin_amdgcn_readfirstlane(to) - row0;
  return rows > 0;
}

}  // namespace
}  // namespace mi355
