// Index of a volume's daughters for the navigator: which daughters a stretch
// of a ray can meet, or a point can be in.
//
// Each of four coordinates of the mother's frame -- x, y, z and the distance
// rho from the z axis -- is cut into slices.  A slice holds two bit masks of
// the daughters: those whose extent along the coordinate ends in the slice
// or beyond it, and those whose extent begins in the slice or before it.  A
// stretch whose coordinate runs from slice i to slice j can only meet the
// daughters in the first mask of i and the second of j, and the AND over the
// coordinates is a superset of the daughters it meets: four or six 8-byte
// words stand for the box tests of up to 64 daughters.
//
// The end slices reach to infinity, so every finite point has valid masks.
// All extents are widened by a pad that covers the rounding of the slice
// numbers.
#pragma once

#include <cstdint>
#include <vector>

#include "vg_math.hpp"

namespace vga {

constexpr int kIndexCoords = 4;  // x, y, z, rho
constexpr int kIndexAxes = 3;    // coordinates looked up at most

// One looked-up coordinate: slice of u is (u - lo) * inv clamped to
// [0, slices - 1]; its masks are words off + (2 * slice + which) * words +
// word, words = ceil(daughters / 64), which = 0: extent ends here or beyond,
// 1: extent begins here or before.
struct DaughterAxis {
  float lo, inv;
  int32_t off, slices;
};

struct DaughterIndex {
  float first;         // first stretch of a ray to search (mm)
  float near;          // first distance around a point to search for its safety (mm)
  float lo[3], hi[3];  // box of all daughters' extents
  DaughterAxis axis[kIndexAxes];
};
static_assert(sizeof(DaughterIndex) == 80, "five 16-byte loads");

// Which coordinates an index looks up: the first `count` entries of coord; and
// whether every daughter is safe (DaughterExtent::safe).
struct IndexAxes {
  int count = 0;
  int coord[kIndexAxes] = {};
  bool safe = false;
};

// One daughter's extent in its mother's frame: x, y, z and rho.
struct DaughterExtent {
  double lo[kIndexCoords], hi[kIndexCoords];
  // SafetyToIn is at least 0.7 times a point's distance from the extent in
  // any one coordinate: the Orb (the distance itself), a Box turned about z
  // only (the largest of its three axes' distances), a Tube without phi
  // section about the mother's z axis (its z and rho distances).
  bool safe;
};

// Extent of the shape's surface and inside (every point where its Contains
// holds or its DistanceToIn ends) under placement X, joined with the float
// box `box` (lo xyz, hi xyz).
DaughterExtent ExtentInMother(int type, const double *blk, const Xf &X, const double lo[3], const double hi[3],
                              const double box[6]);

// Words of masks that an index over nd daughters takes at most.
size_t DaughterIndexWords(int nd);

// Builds the index of one volume over its daughters' extents; the masks are
// appended to `masks`.
DaughterIndex BuildDaughterIndex(const std::vector<DaughterExtent> &d, std::vector<uint64_t> &masks, IndexAxes *axes);

}  // namespace vga
