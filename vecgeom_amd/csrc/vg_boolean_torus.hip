// Basket queries on Boolean volumes with a Torus operand.
#include "vg_boolean_kernels.hpp"

namespace vga {

int LaunchBooleanTorus(int q, const double *blk, const PlacedRec &pr, const QArgs &a, hipStream_t s) {
  return LaunchBooleanSet<kBoolAll>(q, blk, pr, a, s);
}

}  // namespace vga
