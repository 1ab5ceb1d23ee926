// launch_grid.h -- grid of a launch whose blocks are one wavefront each.
#pragma once

namespace oqph {

struct Grid2 {
  unsigned x, y;
};

// `blocks` blocks of 64 lanes in up to 65535 rows of about 65536 (wider when that many
// rows do not suffice); the kernel numbers them blockIdx.y gridDim.x + blockIdx.x and the
// last few have no work.  One dimension of a launch holds fewer than 2^32 threads, which
// a single row reaches at 4.3e9 quartets of a class (about (H2O)128/cc-pVTZ).
inline Grid2 wave_grid(long long blocks) {
  long long y = (blocks + 65535) / 65536;
  y = y < 1 ? 1 : y > 65535 ? 65535 : y;
  return {(unsigned)((blocks + y - 1) / y), (unsigned)y};
}

}  // namespace oqph
