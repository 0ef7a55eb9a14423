// The bounds within which the matrix-core pair build may decide a pair by the
// expanded square |a|^2 + |b|^2 - 2 a.b in float32.  Plain C++ (no HIP), so
// that the CPU tests compile it on its own.
#pragma once

#include <cmath>

namespace sph {

// Squares below lo are inside the cutoff, at or above hi outside; in between,
// and for every candidate of a piece with a particle further than inside[d]
// from its cell's centre along an axis, the filter of nl_build_body decides.
struct TileBand {
  float lo, hi;
  float inside[3];
};

// Outside the band both filters decide the same.  Per component the exact
// metric is within 2 ulp(box) of the true one, the fast square within 1 and the
// expanded one (its centre less an image) within 1: for a pair at `reach`,
// 2 reach sqrt(3) 3 ulp(box) < 16 reach ulp(box).  The expanded square itself
// loses at most 15 2^-24 (|a| + |b|)^2, with |b| <= |a| + reach, and gets twice
// that.  |a| is half a cell an axis, and what rounding the cell's number and
// its centre adds (under 2 ulp(box)); a particle off the grid, which is clamped
// into its outer cells, may lie further out and is left to the other filter.
inline TileBand tile_band(const float* box, const float* cell, int dim, float reach,
                          float cutoff_sq) {
  double maxbox = 0.0, a_sq = 0.0;
  for (int d = 0; d < dim; ++d) maxbox = std::fmax(maxbox, (double)box[d]);
  const double ulp_box = std::nextafter((float)maxbox, INFINITY) - (float)maxbox;
  TileBand t{0.0f, 0.0f, {INFINITY, INFINITY, INFINITY}};
  for (int d = 0; d < dim; ++d) {
    t.inside[d] = (float)(0.5 * cell[d] + 4.0 * ulp_box);
    a_sq += (double)t.inside[d] * t.inside[d];
  }
  const double m = 2.0 * std::sqrt(a_sq) + reach;
  const double band = 16.0 * reach * ulp_box + 16.0 * std::ldexp(m * m, -23);
  t.lo = (float)(cutoff_sq - band);
  t.hi = (float)(cutoff_sq + band);
  return t;
}

}  // namespace sph
