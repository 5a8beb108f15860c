// Host-side flattening of a vg_flat_geometry into the records the device
// kernels read (the work CudaManager::Synchronize does for the reference,
// source/CudaManager.cpp:40-160), plus the error state shared by the C-ABI.
// Nothing here touches a device, so the same code also builds geometries for
// host-only checks of the navigation code.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "shapes.hpp"
#include "vg_internal.hpp"

namespace vga {

namespace {
thread_local std::string g_last_error;
}  // namespace

int SetError(int code, const std::string &msg) {
  g_last_error = msg;
  return code;
}

const char *LastError() { return g_last_error.c_str(); }

int CheckHip(hipError_t e, const char *what) {
  if (e == hipSuccess) return VG_OK;
  return SetError(VG_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

bool ShapeHasKernels(int type) {
  switch (type) {
    case VG_BOX: case VG_TUBE: case VG_ORB: case VG_TRD: case VG_PARALLELEPIPED: case VG_PARABOLOID:
    case VG_TRAPEZOID: case VG_SPHERE: case VG_CONE: case VG_POLYCONE: case VG_TORUS: case VG_POLYHEDRON:
    case VG_BOOLEAN:
      return true;
  }
  return false;
}

namespace {

// Placement kind as Transformation3D::SetProperties decides it
// (source/Transformation3D.cpp:81-90, 139-150).
int KindOfPlacement(const double *xf12) {
  const bool hasT = std::fabs(xf12[0]) > kTolerance || std::fabs(xf12[1]) > kTolerance || std::fabs(xf12[2]) > kTolerance;
  int code = 0;
  for (int i = 0; i < 9; ++i) code |= (1 << i) * (std::fabs(xf12[3 + i]) > kTolerance);
  if (code == 0x111 && xf12[3] == 1. && xf12[7] == 1. && xf12[11] == 1.) code = 0x200;
  const bool hasR = code != 0x200;
  if (!hasT && !hasR) return kXfIdentity;
  if (hasT && !hasR) return kXfTranslation;
  if (!hasT && hasR) return kXfRotation;
  return kXfGeneral;
}

// ABBoxManager::ComputeABBox, source/ABBoxManager.cpp:128-161: the 8 corners
// of the local extent mapped by InverseTransform
// (base/Transformation3D.h:601-632), padded by 1e-3.
void ComputeAABB(const double lo[3], const double hi[3], const Xf &X, double *out6) {
  const double delta[3] = {hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]};
  double mn[3] = {kInfinity, kInfinity, kInfinity}, mx[3] = {-kInfinity, -kInfinity, -kInfinity};
  for (int ix = 0; ix <= 1; ++ix)
    for (int iy = 0; iy <= 1; ++iy)
      for (int iz = 0; iz <= 1; ++iz) {
        const double c[3] = {lo[0] + ix * delta[0], lo[1] + iy * delta[1], lo[2] + iz * delta[2]};
        double m[3];
        for (int r = 0; r < 3; ++r) {
          m[r] = X.t[r];
          m[r] += c[0] * X.r[3 * r + 0];
          m[r] += c[1] * X.r[3 * r + 1];
          m[r] += c[2] * X.r[3 * r + 2];
        }
        for (int r = 0; r < 3; ++r) {
          mn[r] = std::min(mn[r], m[r]);
          mx[r] = std::max(mx[r], m[r]);
        }
      }
  for (int r = 0; r < 3; ++r) {
    out6[r] = mn[r] - 1E-3;
    out6[3 + r] = mx[r] + 1E-3;
  }
}

// A rotation whose rows are unit vectors at right angles.
bool Orthonormal(const Xf &X) {
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j <= i; ++j) {
      double s = 0;
      for (int k = 0; k < 3; ++k) s += X.r[3 * i + k] * X.r[3 * j + k];
      if (!(std::fabs(s - (i == j ? 1. : 0.)) < 1e-9)) return false;
    }
  return true;
}

bool Bits(double a, double b) { return std::memcmp(&a, &b, sizeof a) == 0; }

// The navigator's record of a placed volume.  A placement that is no exact
// translation or rotation about z keeps its full matrix; a matrix that is
// one is restored bit for bit from the numbers kept.
NavRec MakeNavRec(const PlacedRec &r, const double *blk) {
  NavRec n{};
  n.index = -1;
  n.dbegin = r.dbegin;
  n.nd = r.dend - r.dbegin;
  n.type = r.type;
  n.param_off = r.param_off;
  n.code = kFormGeneral;
  switch (r.type) {
    case VG_BOX: {
      const BoxP &b = *reinterpret_cast<const BoxP *>(blk);
      n.code = kFormBox;
      for (int i = 0; i < 3; ++i) n.s[i] = b.d[i];
      break;
    }
    case VG_TUBE: {
      const TubeP &t = *reinterpret_cast<const TubeP *>(blk);
      if (t.hasPhi != 0) break;
      n.code = kFormTube;
      n.s[0] = t.rmin;
      n.s[1] = t.rmax;
      n.s[2] = t.z;
      break;
    }
    case VG_TRD: {
      const TrdP &t = *reinterpret_cast<const TrdP *>(blk);
      n.code = kFormTrd;
      n.s[0] = t.dx1;
      n.s[1] = t.dx2;
      n.s[2] = t.dy1;
      n.s[3] = t.dy2;
      n.s[4] = t.dz;
      n.s[5] = t.fx;
      break;
    }
    case VG_ORB: {
      const OrbP &o = *reinterpret_cast<const OrbP *>(blk);
      n.code = kFormOrb;
      n.s[0] = o.r;
      n.s[1] = o.rTolI;
      n.s[2] = o.rTolO;
      break;
    }
  }
  n.code |= r.xfkind << kNavKindShift;
  const double *m = r.xf.r;
  bool about_z = Bits(m[8], 1.);
  for (int i : {2, 5, 6, 7}) about_z &= Bits(m[i], 0.);
  const bool unit = about_z && Bits(m[0], 1.) && Bits(m[1], 0.) && Bits(m[3], 0.) && Bits(m[4], 1.);
  const bool still = Bits(r.xf.t[0], 0.) && Bits(r.xf.t[1], 0.) && Bits(r.xf.t[2], 0.);
  if (!about_z) {
    n.code |= kNavMatrix;
    return n;
  }
  if (!still) n.code |= kNavMoves;
  if (!unit) n.code |= kNavTurns;
  for (int i = 0; i < 3; ++i) n.t[i] = r.xf.t[i];
  n.r[0] = m[0];
  n.r[1] = m[1];
  n.r[2] = m[3];
  n.r[3] = m[4];
  return n;
}

// Daughter indexes of the logical volumes with at least kIndexMinDaughters
// daughters.  A volume with a daughter whose matrix is no rotation gets none
// (its extent along the mother's axes would mean nothing), and none is built
// beyond kIndexMaxWords of masks in all.
//
// The search for the next boundary takes the index where it has enough
// daughters.  Below that a loop in which the lanes of a wave test the same
// daughter beats searches that take different ones: the more so the longer
// the shapes' code, and less for the Simple navigators, which have no box
// tests to sort out most daughters.  Traces of 262,144 tracks in a world of n
// daughters, loop and index: ABBox 16 boxes 197 and 234 us, 24 264 and 281,
// 32 314 and 280; of all shapes 24 1097 and 1335, 32 1022 and 1174, 48 1648
// and 1722 (65,536 tracks: 24 518 and 555, 32 516 and 512, 48 699 and 650);
// Simple 6 boxes 135 and 157, 9 170 and 146; of all shapes 12 668 and 866, 24
// 1264 and 1409, 32 1381 and 1246.  In volumes below the world the lanes are in
// different ones and the loop gains less: the nested geometry's 8 Trds in a
// box as a loop 4.85 ms, with the index 4.5.
//
// In single-step kernels the lanes of a wave stay in step and the loop holds
// out longer, most of all where waves are full (kBigStep).  262,144 tracks,
// loop and index: ABBox 40 boxes 48 and 96 us, 96 147 and 216, 96 daughters with
// phi tubes 319 and 327, of all shapes 989 and 1084; Simple 40 with phi tubes 158
// and 182, 96 353 and 427, of all shapes 773 and 1294.  1,000 tracks: ABBox 64
// boxes 37 and 28, 32 26 and 21, 24 21 and 23; Simple 24 boxes 54 and 30, 96 of
// all shapes 260 and 250.
constexpr int kIndexMinDaughters = 3;
struct WalkMin {
  int abbox[3], simple[3];  // by WalkKernel
};
constexpr WalkMin kWalkWorld = {{20, 64, 100}, {9, 32, 100}}, kWalkWorldGeneral = {{32, 100, 100}, {20, 128, 128}};
constexpr WalkMin kWalkBelow = {{8, 8, 8}, {8, 8, 8}}, kWalkBelowGeneral = {{12, 12, 12}, {12, 12, 12}};
// Where boxes lie in one another (the nested geometry's 64 coaxial shells) box
// tests sort out little and the loop evaluates most daughters: the minima of
// kWalkBelow hold in the world, too.  One step of 65,536 vertex tracks there as
// a loop 140 us, with the index 15.
constexpr double kCrowded = 2;

// The mean number of daughters whose box holds the centre of a daughter's box.
double Crowd(const vg_geometry *g, int db, int de) {
  long in = 0;
  for (int k = db; k < de; ++k) {
    const double *b = g->aabb.data() + 6 * (size_t)g->daughters[k];
    for (int j = db; j < de; ++j) {
      const double *o = g->aabb.data() + 6 * (size_t)g->daughters[j];
      bool inside = true;
      for (int a = 0; a < 3; ++a) {
        const double c = 0.5 * (b[a] + b[3 + a]);
        inside &= c >= o[a] && c <= o[3 + a];
      }
      in += inside;
    }
  }
  return (double)in / (de - db);
}

// The safety takes the index from kSafeMin daughters on (figures at GetSafety).
constexpr int kSafeMin = 32;
constexpr size_t kIndexMaxWords = size_t(1) << 25;  // 256 MiB

void BuildIndexes(vg_geometry *g) {
  const int nl = (int)g->logical_shape.size();
  std::vector<int32_t> of(nl, -1), axes_code(nl, 0);
  std::vector<DaughterExtent> ext;
  for (int l = 0; l < nl; ++l) {
    const int db = g->logical_dbegin[l], de = g->logical_dbegin[l + 1];
    if (de - db < kIndexMinDaughters) continue;
    ext.clear();
    bool ok = true, basic = true;
    for (int k = db; k < de && ok; ++k) {
      const PlacedRec &r = g->placed[g->daughters[k]];
      basic &= r.type == VG_BOX || r.type == VG_TUBE || r.type == VG_ORB || r.type == VG_TRD;
      const double *blk = g->params.data() + r.param_off;
      double lo[3], hi[3];
      ok = Orthonormal(r.xf) && ShapeExtent(r.type, blk, lo, hi);
      if (ok) ext.push_back(ExtentInMother(r.type, blk, r.xf, lo, hi, g->aabb.data() + 6 * (size_t)g->daughters[k]));
    }
    if (!ok) continue;
    if (g->dmasks.size() + DaughterIndexWords(de - db) > kIndexMaxWords) continue;
    of[l] = (int32_t)g->dindex.size();
    IndexAxes axes;
    g->dindex.push_back(BuildDaughterIndex(ext, g->dmasks, &axes));
    axes_code[l] = axes.count << kNavAxesShift;
    for (int a = 0; a < axes.count; ++a) axes_code[l] |= axes.coord[a] << (kNavCoordShift + 2 * a);
    // (From 128 daughters on every kernel takes the index.)
    const bool spread = l == g->placed[g->world].logical && de - db < 128 && Crowd(g, db, de) < kCrowded;
    const WalkMin min = spread ? (basic ? kWalkWorld : kWalkWorldGeneral) : (basic ? kWalkBelow : kWalkBelowGeneral);
    for (const WalkKernel k : {kWalkTrace, kWalkStep, kWalkBigStep}) {
      if (de - db >= min.abbox[k]) axes_code[l] |= WalkBit(true, k);
      if (de - db >= min.simple[k]) axes_code[l] |= WalkBit(false, k);
    }
    if (axes.safe && de - db >= kSafeMin) axes_code[l] |= kNavSafe;
  }
  for (int l = 0; l < nl; ++l)
    g->safety_scans |= g->logical_dbegin[l + 1] - g->logical_dbegin[l] >= kIndexMinDaughters && !(axes_code[l] & kNavSafe);
  g->nav.resize(g->placed.size());
  for (size_t p = 0; p < g->placed.size(); ++p) {
    const PlacedRec &r = g->placed[p];
    g->nav[p] = MakeNavRec(r, g->params.data() + r.param_off);
    g->nav[p].code |= axes_code[r.logical];
    g->nav[p].index = of[r.logical];
  }
}

int Depth(const vg_geometry *g, int32_t placed, int level, int limit) {
  if (level > limit) return -1;
  const PlacedRec &p = g->placed[placed];
  int best = level;
  for (int k = p.dbegin; k < p.dend; ++k) {
    int d = Depth(g, g->daughters[k], level + 1, limit);
    if (d < 0) return -1;
    best = std::max(best, d);
  }
  return best;
}

}  // namespace

int BuildGeometry(const vg_flat_geometry *f, vg_geometry *g) {
  if (f->n_shapes < 0 || f->n_logical < 0 || f->n_placed <= 0)
    return SetError(VG_ERR_INVALID, "geometry needs at least one placed volume");
  if (!f->shape_type || !f->shape_param_begin || !f->logical_shape || !f->logical_daughter_begin ||
      !f->placed_logical || !f->placed_transform)
    return SetError(VG_ERR_INVALID, "null geometry array");
  if (f->world < 0 || f->world >= f->n_placed) return SetError(VG_ERR_INVALID, "world id out of range");

  g->world = f->world;
  // Shapes: parameter blocks.
  g->shapes.resize(f->n_shapes);
  for (int s = 0; s < f->n_shapes; ++s) {
    const int b = f->shape_param_begin[s], e = f->shape_param_begin[s + 1];
    if (b < 0 || e < b || (e > b && !f->params)) {
      return SetError(VG_ERR_INVALID, "bad parameter range for shape " + std::to_string(s));
    }
    std::string err;
    std::vector<double> block = BuildParams(f->shape_type[s], f->params + b, e - b, &err);
    if (block.empty()) {
      return SetError(ShapeHasKernels(f->shape_type[s]) ? VG_ERR_INVALID : VG_ERR_UNSUPPORTED,
                      "shape " + std::to_string(s) + ": " + err);
    }
    if (block.size() > (size_t)kMaxParamDoubles) {
      return SetError(VG_ERR_CAPACITY, "shape " + std::to_string(s) + ": parameter block too large");
    }
    // Keep every block 16-byte aligned within the device array.
    if (g->params.size() % 2) g->params.push_back(0.);
    g->shapes[s] = ShapeRec{f->shape_type[s], (int32_t)g->params.size(), (int32_t)block.size(), 0};
    g->params.insert(g->params.end(), block.begin(), block.end());
  }
  // Logical volumes.
  g->logical_shape.assign(f->logical_shape, f->logical_shape + f->n_logical);
  g->logical_dbegin.assign(f->logical_daughter_begin, f->logical_daughter_begin + f->n_logical + 1);
  const int nd = f->n_logical > 0 ? g->logical_dbegin[f->n_logical] : 0;
  if (nd > 0 && !f->daughters) {
    return SetError(VG_ERR_INVALID, "null daughters array");
  }
  g->daughters.assign(f->daughters, f->daughters + nd);
  for (int l = 0; l < f->n_logical; ++l) {
    if (g->logical_shape[l] < 0 || g->logical_shape[l] >= f->n_shapes || g->logical_dbegin[l] < 0 ||
        g->logical_dbegin[l + 1] < g->logical_dbegin[l] || g->logical_dbegin[l + 1] > nd) {
      return SetError(VG_ERR_INVALID, "bad logical volume " + std::to_string(l));
    }
  }
  for (int k = 0; k < nd; ++k) {
    if (g->daughters[k] < 0 || g->daughters[k] >= f->n_placed) {
      return SetError(VG_ERR_INVALID, "daughter id out of range");
    }
  }
  // Placed volumes.
  g->placed.resize(f->n_placed);
  g->aabb.resize(6 * (size_t)f->n_placed);
  g->b32.resize(f->n_placed);
  g->extent32.resize(6 * (size_t)f->n_placed);
  g->b32side.clear();
  for (int p = 0; p < f->n_placed; ++p) {
    const int l = f->placed_logical[p];
    if (l < 0 || l >= f->n_logical) {
      return SetError(VG_ERR_INVALID, "placed volume " + std::to_string(p) + " has a bad logical id");
    }
    PlacedRec &r = g->placed[p];
    const double *x = f->placed_transform + 12 * (size_t)p;
    r.logical = l;
    r.shape = g->logical_shape[l];
    r.type = g->shapes[r.shape].type;
    r.xfkind = KindOfPlacement(x);
    r.param_off = g->shapes[r.shape].param_off;
    r.dbegin = g->logical_dbegin[l];
    r.dend = g->logical_dbegin[l + 1];
    r.pad = 0;
    for (int i = 0; i < 3; ++i) r.xf.t[i] = x[i];
    for (int i = 0; i < 9; ++i) r.xf.r[i] = x[3 + i];
    double lo[3], hi[3];
    if (!ShapeExtent(r.type, g->params.data() + r.param_off, lo, hi)) {
      return SetError(VG_ERR_UNSUPPORTED, "no extent for shape type " + std::to_string(r.type));
    }
    ComputeAABB(lo, hi, r.xf, g->aabb.data() + 6 * (size_t)p);
    BuildBound32(r.type, g->params.data() + r.param_off, r.xf, lo, hi, g->b32[p], g->b32side);
    for (int i = 0; i < 3; ++i) {
      g->extent32[6 * (size_t)p + i] = (float)lo[i];
      g->extent32[6 * (size_t)p + 3 + i] = (float)hi[i];
    }
    // Navigation and serving dispatch primitive shapes only.
    if (!g->nav_bad_type && (!ShapeHasKernels(r.type) || r.type == VG_BOOLEAN)) g->nav_bad_type = r.type;
    if (r.type >= 0 && r.type < 32) g->type_mask |= 1u << r.type;
    if (r.type == VG_TUBE && reinterpret_cast<const TubeP *>(g->params.data() + r.param_off)->hasPhi != 0)
      g->type_mask |= 1u;
  }
  // The daughters' float boxes in daughter-slot order, each with the
  // daughter's placed id: one record answers slot k's box test and says where
  // its volume is.
  g->slot_aabb.assign(8 * g->daughters.size(), 0.f);
  for (size_t k = 0; k < g->daughters.size(); ++k) {
    for (int i = 0; i < 6; ++i) g->slot_aabb[8 * k + i] = (float)g->aabb[6 * (size_t)g->daughters[k] + i];
    std::memcpy(&g->slot_aabb[8 * k + 6], &g->daughters[k], sizeof(int32_t));
  }
  BuildIndexes(g);
  g->max_depth = Depth(g, g->world, 1, 64);
  if (g->max_depth < 0) {
    return SetError(VG_ERR_INVALID, "volume tree deeper than 64 levels or cyclic");
  }
  return VG_OK;
}

int PlacementKind(const double *xf12) { return KindOfPlacement(xf12); }

}  // namespace vga
