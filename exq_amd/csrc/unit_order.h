// unit_order.h -- which work-group takes which unit (token group x weight tile).
// Plain integer arithmetic, used by the kernels and by the host code that sizes
// their grids; needs no HIP header.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define EXQ_HD __host__ __device__ inline
#else
#define EXQ_HD inline
#endif

namespace exq {

// Work-groups of the unit range over n token groups (a multiple of eight groups
// times the weight tiles per group).
template <typename I>
EXQ_HD I unit_count(I n, int n_tiles) {
  return ((n + 7) >> 3) * 8 * n_tiles;
}

// Weight tiles per token group in each range of the combined tile launch
// (tile_mix_kernel), in the order of its grid.  A range whose cap is 0 has no
// tiles: its token groups, if the list holds any, belong to another kernel, and
// the device counts no units for them.
struct MixTiles {
  int ps;   // 128 x 256 INT4 tiles
  int i8;   // 128 x 256 INT8 tiles
  int t64;  // 64 x 256 INT4 tiles
  int bf;   // 128 x 128 BF16 tiles
};

inline MixTiles mix_tiles(int tiles256, int tiles128, int64_t cap_ps, int64_t cap_i8,
                          int64_t cap_64, int64_t cap_bf) {
  return MixTiles{cap_ps > 0 ? tiles256 : 0, cap_i8 > 0 ? tiles256 : 0,
                  cap_64 > 0 ? tiles256 : 0, cap_bf > 0 ? tiles128 : 0};
}

// Its grid: enough work-groups for every range at its cap of token groups.
inline int64_t mix_grid(const MixTiles& t, int64_t cap_ps, int64_t cap_i8, int64_t cap_64,
                        int64_t cap_bf) {
  return unit_count(cap_ps, t.ps) + unit_count(cap_i8, t.i8) + unit_count(cap_64, t.t64) +
         unit_count(cap_bf, t.bf);
}

// Unit (token group tgi of n, weight tile nt of n_tiles) of work-group bid of the
// rows kernels; false: none.  XCD-aware (work-group i runs on XCD i % 8): each XCD
// takes an eighth of the units in a row, blocks of 8 token groups x all weight
// tiles with the groups fastest, so that the groups of one expert share its
// weights in that XCD's L2.  The last 9 .. 15 groups are two blocks of half as
// many: as 8 and a few padded to 8 they left the XCDs of the padded block idle
// (unquantised 4096 x 28672 weights, 8 experts, 128 tokens: 521 us, 384 so).
EXQ_HD bool rows_unit_of(int bid, int n, int n_tiles, int& tgi, int& nt) {
  const int U = n * n_tiles;
  const int per = (U + 7) >> 3;
  const int local = bid >> 3;
  int v = (bid & 7) * per + local;
  if (local >= per || v >= U) return false;
  const int full = n <= 8 ? 0 : (n & 7) == 0 ? n : (n & ~7) - 8;  // groups in blocks of 8
  if (v < full * n_tiles) {
    const int tb = v / (8 * n_tiles);
    const int rem = v - tb * 8 * n_tiles;
    nt = rem >> 3;
    tgi = tb * 8 + (rem & 7);
    return true;
  }
  v -= full * n_tiles;
  int first = full, size = n - full;
  if (size > 8) {
    const int half = (size + 1) >> 1;
    if (v < half * n_tiles) {
      size = half;
    } else {
      v -= half * n_tiles;
      first += half;
      size -= half;
    }
  }
  nt = v / size;
  tgi = first + v - nt * size;
  return true;
}

}  // namespace exq
