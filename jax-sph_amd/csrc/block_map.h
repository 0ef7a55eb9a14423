// Which particles a workgroup of a launch serves.  Plain C++ outside hipcc, so
// that the CPU tests compile it on its own.
#pragma once

#ifdef __HIP__
#include <hip/hip_runtime.h>
#define SPH_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define SPH_HOST_DEVICE inline
#endif

namespace sph {

// ------------------------------------------------------------ XCD mapping
// MI355X dispatches the workgroups of a launch to its 8 XCDs round-robin by
// workgroup id, and each XCD has its own L2.  With remap on (and a grid that
// is a multiple of 8), XCD x runs the contiguous logical blocks
// [x * per, (x + 1) * per): cell-sorted particles that share neighbours then
// share one L2 instead of being spread over all eight, and a sweep finds there
// what the launch before left of the same particles.
constexpr int kXcds = 8;
SPH_HOST_DEVICE int logical_block_of(int b, int blocks, int remap) {
  if (!remap) return b;
  const int per = blocks / kXcds;
  return (b % kXcds) * per + b / kXcds;
}
SPH_HOST_DEVICE unsigned xcd_grid(long long blocks, int remap) {
  return (unsigned)(remap ? (blocks + kXcds - 1) / kXcds * kXcds : blocks);
}

// A sweep that also reduces the partials of an earlier launch has eight
// workgroups more in front, the first of which does that while the others end
// at once: one more would move every block to the next XCD, away from what the
// launches around it hold in their L2 (force sweep of 90,000 2D particles with
// one 17.7 us, with eight 15.6, Riemann 20.4 and 17.6; 128^3 1,578 and 1,566).
// Returns the logical block of workgroup b, or for those eight the first past
// the last.
constexpr int kTailBlocks = kXcds;
SPH_HOST_DEVICE int sweep_block_of(int b, int grid, bool tail, int remap) {
  const int extra = tail ? kTailBlocks : 0, blocks = grid - extra;
  const int l = logical_block_of(b - extra, blocks, remap);
  return b < extra ? blocks : l;
}

}  // namespace sph
