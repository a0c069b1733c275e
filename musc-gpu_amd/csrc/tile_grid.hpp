// Launch grid of the pair kernels: a workgroup per tile.  Host code only.
#pragma once

namespace musc {
namespace msm {

// HIP launches fewer than 2^32 threads in a grid dimension, which is 16.7 million workgroups of
// 256: more tiles go on in gridDim.z, in slices of equal size (gridDim.y counts pools).  x is a
// multiple of `multiple`; the ids past the last tile, fewer than z * multiple, end at once.
struct TileGrid {
  unsigned x, z;
};

// false: more tiles than a grid of 2^31 - 1 workgroups holds.
inline bool tile_grid(long long tiles, int threads, int multiple, TileGrid* grid) {
  if ((tiles + multiple - 1) / multiple * multiple > 0x7fffffffLL) return false;
  const long long most = 0xffffffffLL / threads / multiple * multiple;
  const long long slices = (tiles + most - 1) / most;
  grid->x = (unsigned)(((tiles + slices - 1) / slices + multiple - 1) / multiple * multiple);
  grid->z = (unsigned)slices;
  return true;
}

}  // namespace msm
}  // namespace musc
