// Basket queries on Boolean volumes (shapes_boolean.hpp), one query per
// lane.  The Boolean's placement is applied as the reference's
// SpecializedBooleanVolume does (Transform<transCode, rotCode> for the point,
// TransformDirection for the direction); the operands' parameter blocks are
// read from global memory through the Boolean's block (they are small and
// stay in the caches).  Query semantics, including the Minimize forms and the
// DistanceToOut next-node output, are those of the other shapes' basket
// kernels (volumes/ShapeImplementationHelper.h:588-748).
#include "vg_boolean_kernels.hpp"

namespace vga {

int LaunchBooleanQuery(const vg_geometry *g, int32_t placed, int q, const QArgs &a, hipStream_t s) {
  if (a.n == 0) return VG_OK;
  const PlacedRec &pr = g->placed[placed];
  const double *blk = g->d_params + pr.param_off;
  const double *host = g->params.data() + pr.param_off;
  const bool torus = (int)host[1] == VG_TORUS || (int)host[4] == VG_TORUS;  // the operands' types
  return torus ? LaunchBooleanTorus(q, blk, pr, a, s) : LaunchBooleanSet<kBoolNoTorus>(q, blk, pr, a, s);
}

}  // namespace vga
