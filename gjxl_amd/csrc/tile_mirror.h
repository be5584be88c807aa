// Which sample of a line a tile's halo reads, for the kernels that load whole
// tiles: every lane of the tile reads, also the ones that lie further outside
// the line than any output needs.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define GJXL_AMD_HD __host__ __device__
#else
#define GJXL_AMD_HD
#endif

namespace gjxl_amd {

// The mirrored coordinate of c in a line of `size` samples, c >= -size, by
// selects: one reflection, which is all that -size <= c < 2 * size needs.  A
// tile of 64 columns reaches past 2 * size in a short line; what it reads
// there is never used, and the reflected coordinate, which would lie in front
// of the line, is held at its first sample.  The result is in 0 .. size - 1.
GJXL_AMD_HD inline int TileMirror(int c, int size) {
  c = c < 0 ? -c - 1 : c;
  c = c >= size ? 2 * size - 1 - c : c;
  return c < 0 ? 0 : c;
}

}  // namespace gjxl_amd
