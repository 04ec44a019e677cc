// The scheduling map without its kernel: what a work-group of a gmm or tgmm launch needs to know about its tile - the
// group, its rows, its band of the walk - worked out by each wave for itself from group_sizes.
//
// The map kernel (rd_sched.hip) takes 4-8 us in front of every product, more than a small product itself, and the
// look-ups in the map are a chain of four dependent loads at the start of every tile.  Here a wave loads the sizes of up
// to 256 groups at once (four per lane), scans them with twelve data-parallel moves per 64 groups and finds its tile's
// group by a ballot: one round trip to L2 and about 0.3 us of arithmetic, whatever the tile.  512 x 256 x 512 in 4 groups,
// forward + gradients: 69 -> 58 us a pass; 4099 x 1001 x 1515 in 12: 137 -> 122 us.  The map kernel stays where a launch
// needs what only it makes: the interleaved block order, cleared K-split counters, the deferred short tiles, the order by
// size class, or more groups than are scanned here.
#pragma once
#include "rd_common.h"
#include "rd_sched.h"

namespace rd {

constexpr int kLookupGroups = 256;
constexpr int kLookupChunks = kLookupGroups / 64;

// Inclusive sum over the lanes of a wave.
__device__ __forceinline__ int wave_inclusive_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1 within rows of 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// All groups of a gmm launch, as one wave holds them: lane l of chunk c has group 64 c + l.
template <int BM>
struct GroupScan {
  int size[kLookupChunks], tiles[kLookupChunks], rows[kLookupChunks];  // rows and row tiles up to and including the group
  int total_tiles, total_rows;

  __device__ __forceinline__ void init(const int32_t* __restrict__ gs, int g) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < kLookupChunks; ++c) size[c] = 64 * c + lane < g ? imax(gs[64 * c + lane], 0) : 0;
    int tiles_before = 0, rows_before = 0;
#pragma unroll
    for (int c = 0; c < kLookupChunks; ++c) {
      tiles[c] = tiles_before; rows[c] = rows_before;
      if (64 * c < g) {
        tiles[c] += wave_inclusive_sum((size[c] + BM - 1) / BM);
        rows[c] += wave_inclusive_sum(size[c]);
        tiles_before = __builtin_amdgcn_readlane(tiles[c], 63);
        rows_before = __builtin_amdgcn_readlane(rows[c], 63);
      }
    }
    total_tiles = tiles_before; total_rows = rows_before;
  }

  // The group that row tile `t` (below total_tiles) belongs to: its index, rows, first row and first row tile.
  __device__ __forceinline__ void find(int t, int* group, int* group_rows, int* first_row, int* first_tile) const {
    bool found = false;
#pragma unroll
    for (int c = 0; c < kLookupChunks; ++c) {
      const unsigned long long past = __ballot(tiles[c] > t);
      if (!found && past) {
        found = true;
        const int l = __ffsll(past) - 1;
        const int sz = __builtin_amdgcn_readlane(size[c], l);
        *group = 64 * c + l;
        *group_rows = sz;
        *first_row = __builtin_amdgcn_readlane(rows[c], l) - sz;
        *first_tile = __builtin_amdgcn_readlane(tiles[c], l) - (sz + BM - 1) / BM;
      }
    }
  }
};

// A group's `tiles` row tiles are cut into ceil(tiles / most) bands of nearly equal height, the first tiles % bands of them
// one taller: the band of the group's row tile `it`, as its first row tile within the group and its height.
__host__ __device__ __forceinline__ void band_of(int tiles, int most, int it, int* first, int* height) {
  const int bands = (tiles + most - 1) / most, h = tiles / bands, taller = tiles - h * bands;
  if (it < taller * (h + 1)) { *height = h + 1; *first = it / (h + 1) * (h + 1); }
  else { *height = h; *first = taller * (h + 1) + (it - taller * (h + 1)) / h * h; }
}

// First row of group `want`: the sum of the sizes before it.
__device__ __forceinline__ int rows_before_group(const int32_t* __restrict__ gs, int want) {
  const int lane = threadIdx.x & 63;
  int sum = 0;
  for (int j = lane; j < want; j += 64) sum += imax(gs[j], 0);
  return __builtin_amdgcn_readlane(wave_inclusive_sum(sum), 63);
}

}  // namespace rd
