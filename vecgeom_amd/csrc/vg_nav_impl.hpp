// Navigation functions shared by the device kernels (vg_nav.hip) and a
// host-only build used to check their logic on the CPU.  Behaviour and
// reference citations are described in vg_nav.hip.
//
// With VGA_NAV_HOST_CHECKS defined (host builds only) every table access is
// bounds-checked and a violation aborts with a message.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <type_traits>
#include <cstdint>
#if defined(VGA_NAV_HOST_CHECKS)
#include <cstdio>
#include <cstdlib>
#define VGA_NAV_CHECK(cond, msg)                                  \
  do {                                                            \
    if (!(cond)) {                                                \
      std::fprintf(stderr, "navigation check failed: %s\n", msg); \
      std::abort();                                               \
    }                                                             \
  } while (0)
#else
#define VGA_NAV_CHECK(cond, msg) ((void)0)
#endif
#define VGA_NAV __host__ __device__ __forceinline__

#include "shapes.hpp"
#include "vg_internal.hpp"

namespace vga {
namespace nav {

constexpr float kInfF = __builtin_huge_valf();

struct NavDev {
  const NavRec *nav;            // per placed volume
  const PlacedRec *placed;      // full placements (kNavMatrix; safeties among all shapes)
  const double *params;         // parameter blocks (kFormGeneral)
  const float *slot_box;        // daughter boxes in slot order, 8 floats each
  const DaughterIndex *dindex;  // daughter indexes (NavRec::index)
  const uint64_t *dmasks;       // their masks
  int32_t world;
  int32_t n_placed;
  int32_t n_daughters;
  int32_t n_index;
  int32_t n_masks;
  int32_t walks;  // WalkBit of the kernel
  VGA_NAV const NavRec &Nav(int id) const {
    VGA_NAV_CHECK(id >= 0 && id < n_placed, "placed id out of range");
    return nav[id];
  }
  VGA_NAV const PlacedRec &Placed(int id) const {
    VGA_NAV_CHECK(id >= 0 && id < n_placed, "placed id out of range");
    return placed[id];
  }
  VGA_NAV const float *SlotBox(int k) const {
    VGA_NAV_CHECK(k >= 0 && k < n_daughters, "box slot out of range");
    return slot_box + 8 * (size_t)k;
  }
  VGA_NAV int Daughter(int k) const {
    int id;
    __builtin_memcpy(&id, SlotBox(k) + 6, sizeof id);
    return id;
  }
  VGA_NAV const DaughterIndex &Index(int i) const {
    VGA_NAV_CHECK(i >= 0 && i < n_index, "daughter index out of range");
    return dindex[i];
  }
  VGA_NAV uint64_t Mask(int i) const {
    VGA_NAV_CHECK(i >= 0 && i < n_masks, "daughter mask out of range");
    return dmasks[i];
  }
};

// Shape sets of specialised navigators (bit t: shape type t; bit 0: a Tube
// with a phi section).
constexpr uint32_t kPhiTube = 1u;
constexpr uint32_t kAllShapes = kPhiTube | (1u << VG_BOX) | (1u << VG_TUBE) | (1u << VG_ORB) | (1u << VG_SPHERE) |
                                (1u << VG_CONE) | (1u << VG_TRD) | (1u << VG_TRAPEZOID) |
                                (1u << VG_PARALLELEPIPED) | (1u << VG_PARABOLOID) | (1u << VG_TORUS) |
                                (1u << VG_POLYCONE) | (1u << VG_POLYHEDRON);
// Box, Tube, Orb and Trd: evaluated from the volume's NavRec alone (but for
// the phi tubes).
constexpr uint32_t kBasicShapes = (1u << VG_BOX) | (1u << VG_TUBE) | (1u << VG_ORB) | (1u << VG_TRD);
// Shapes of daughters that an index serves for the safety (DaughterExtent::safe).
constexpr uint32_t kSafeShapes = (1u << VG_BOX) | (1u << VG_TUBE) | (1u << VG_ORB);
// The shapes of set M that are evaluated from their parameter blocks.
constexpr uint32_t BlockShapes(uint32_t m) {
  return (m & ~kBasicShapes & ~kPhiTube) | ((m & kPhiTube) ? (1u << VG_TUBE) : 0u);
}

// ------------------------------------------------------------ shape switch
// Shape switch over the compile-time shape set M (bit t set: shape type t
// may occur).  A navigator specialised for the shapes of one geometry
// carries only their code, which keeps its register count down.
#define VGA_SHAPE_CASES(TYPE, BODY)                   \
  switch (TYPE) {                                     \
    case VG_BOX:                                      \
      if constexpr ((M >> VG_BOX) & 1u) {             \
        using S = BoxS;                               \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_TUBE:                                     \
      if constexpr ((M >> VG_TUBE) & 1u) {            \
        using S = TubeS;                              \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_ORB:                                      \
      if constexpr ((M >> VG_ORB) & 1u) {             \
        using S = OrbS;                               \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_TRD:                                      \
      if constexpr ((M >> VG_TRD) & 1u) {             \
        using S = TrdS;                               \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_PARALLELEPIPED:                           \
      if constexpr ((M >> VG_PARALLELEPIPED) & 1u) {  \
        using S = ParaS;                              \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_PARABOLOID:                               \
      if constexpr ((M >> VG_PARABOLOID) & 1u) {      \
        using S = ParabS;                             \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_TRAPEZOID:                                \
      if constexpr ((M >> VG_TRAPEZOID) & 1u) {       \
        using S = TrapS;                              \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_SPHERE:                                   \
      if constexpr ((M >> VG_SPHERE) & 1u) {          \
        using S = SphereS;                            \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_CONE:                                     \
      if constexpr ((M >> VG_CONE) & 1u) {            \
        using S = ConeS;                              \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_POLYCONE:                                 \
      if constexpr ((M >> VG_POLYCONE) & 1u) {        \
        using S = PolyconeS;                          \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_TORUS:                                    \
      if constexpr ((M >> VG_TORUS) & 1u) {           \
        using S = TorusS;                             \
        BODY;                                         \
      }                                               \
      break;                                          \
    case VG_POLYHEDRON:                               \
      if constexpr ((M >> VG_POLYHEDRON) & 1u) {      \
        using S = PolyhedronS;                        \
        BODY;                                         \
      }                                               \
      break;                                          \
  }

#define VGA_P(blk) (ParamView<S>::Get(blk))

template <uint32_t M = kAllShapes>
VGA_NAV bool DContains(int type, const double *blk, V3 p) {
  VGA_SHAPE_CASES(type, return S::Contains(VGA_P(blk), p));
  return false;
}
template <uint32_t M = kAllShapes>
VGA_NAV int DInside(int type, const double *blk, V3 p) {
  VGA_SHAPE_CASES(type, return S::Inside(VGA_P(blk), p));
  return kOutside;
}
template <uint32_t M = kAllShapes>
VGA_NAV double DDistIn(int type, const double *blk, V3 p, V3 d, double sm) {
  VGA_SHAPE_CASES(type, return S::DistanceToIn(VGA_P(blk), p, d, sm));
  return kInfinity;
}
template <uint32_t M = kAllShapes>
VGA_NAV double DDistOut(int type, const double *blk, V3 p, V3 d, double sm) {
  VGA_SHAPE_CASES(type, return S::DistanceToOut(VGA_P(blk), p, d, sm));
  return kInfinity;
}
template <uint32_t M = kAllShapes>
VGA_NAV double DSafeIn(int type, const double *blk, V3 p) {
  VGA_SHAPE_CASES(type, return S::SafetyToIn(VGA_P(blk), p));
  return kInfinity;
}
template <uint32_t M = kAllShapes>
VGA_NAV double DSafeOut(int type, const double *blk, V3 p) {
  VGA_SHAPE_CASES(type, return S::SafetyToOut(VGA_P(blk), p));
  return kInfinity;
}

#undef VGA_P
#undef VGA_SHAPE_CASES

// The safeties among all shapes as calls: inlined, the Sphere's and the
// Polyhedron's code put the safety kernel at 203 VGPRs and two waves per SIMD
// instead of three (262,144 points among 48 of all shapes 421 us, as calls 377).
template <uint32_t M>
__host__ __device__ __attribute__((noinline)) double CallSafeIn(int type, const double *blk, V3 p) {
  return DSafeIn<M>(type, blk, p);
}
template <uint32_t M>
__host__ __device__ __attribute__((noinline)) double CallSafeOut(int type, const double *blk, V3 p) {
  return DSafeOut<M>(type, blk, p);
}
template <uint32_t M>
VGA_NAV double BlockSafeIn(int type, const double *blk, V3 p) {
  if constexpr ((M & ~(kBasicShapes | kPhiTube)) != 0) return CallSafeIn<M>(type, blk, p);
  return DSafeIn<M>(type, blk, p);
}
template <uint32_t M>
VGA_NAV double BlockSafeOut(int type, const double *blk, V3 p) {
  if constexpr ((M & ~(kBasicShapes | kPhiTube)) != 0) return CallSafeOut<M>(type, blk, p);
  return DSafeOut<M>(type, blk, p);
}

// The first half of a NavRec, in registers.
struct Head {
  int code, index, dbegin, nd;
  double s[6];
};
VGA_NAV Head LoadHead(const NavDev &g, int id) {
  const NavRec &r = g.Nav(id);
  Head h{r.code, r.index, r.dbegin, r.nd, {}};
#pragma unroll
  for (int i = 0; i < 6; ++i) h.s[i] = r.s[i];
  return h;
}

// Calls f(shape, parameters) for the simple shapes, their parameter blocks
// rebuilt from the record (the same operations as the host's constructors,
// so the same bits; the unused members stay undefined), or general(type,
// block) for the others.
template <uint32_t M, bool Safety, class F, class G>
VGA_NAV auto WithShape(const NavDev &g, int id, const Head &h, F f, G general) {
  switch (h.code & kNavFormMask) {
    case kFormBox:
      if constexpr ((M >> VG_BOX) & 1u) return f(BoxS{}, BoxP{{h.s[0], h.s[1], h.s[2]}});
      break;
    case kFormTube:
      if constexpr ((M >> VG_TUBE) & 1u) {
        TubeP t;
        t.rmin = h.s[0];
        t.rmax = h.s[1];
        t.z = h.s[2];
        t.rmin2 = t.rmin * t.rmin;
        t.rmax2 = t.rmax * t.rmax;
        const double lo = t.rmin + kTolerance, hi = t.rmax - kTolerance;
        t.tolIrmin2 = lo * lo;
        t.tolIrmax2 = hi * hi;
        t.hasRmin = t.rmin > 0 ? 1. : 0.;
        t.hasPhi = 0.;
        return f(TubeS{}, t);
      }
      break;
    case kFormTrd:
      if constexpr ((M >> VG_TRD) & 1u) {
        TrdP t;
        t.dx1 = h.s[0];
        t.dx2 = h.s[1];
        t.dy1 = h.s[2];
        t.dy2 = h.s[3];
        t.dz = h.s[4];
        t.x2minusx1 = t.dx2 - t.dx1;
        t.y2minusy1 = t.dy2 - t.dy1;
        t.halfx1plusx2 = 0.5 * (t.dx1 + t.dx2);
        t.halfy1plusy2 = 0.5 * (t.dy1 + t.dy2);
        t.dztimes2 = t.dz * 2;
        t.fx = h.s[5];
        t.fy = 0.5 * (t.dy1 - t.dy2) / t.dz;
        if constexpr (Safety) {
          t.calfx = 1. / Sqrt(1.0 + t.fx * t.fx);
          t.calfy = 1. / Sqrt(1.0 + t.fy * t.fy);
        }
        t.varyingY = t.dy1 != t.dy2 ? 1. : 0.;
        return f(TrdS{}, t);
      }
      break;
    case kFormOrb:
      if constexpr ((M >> VG_ORB) & 1u) return f(OrbS{}, OrbP{h.s[0], h.s[1], h.s[2], 0.});
      break;
  }
  if constexpr (BlockShapes(M) != 0) {
    const NavRec &r = g.Nav(id);
    return general(r.type, g.params + r.param_off);
  } else {
    return decltype(f(BoxS{}, BoxP{}))(0);  // no such volume
  }
}
template <uint32_t M>
VGA_NAV bool NContains(const NavDev &g, int id, const Head &h, V3 p) {
  return WithShape<M, false>(
      g, id, h, [&](auto s, const auto &q) { return decltype(s)::Contains(q, p); },
      [&](int type, const double *blk) { return DContains<BlockShapes(M)>(type, blk, p); });
}
template <uint32_t M>
VGA_NAV double NDistIn(const NavDev &g, int id, const Head &h, V3 p, V3 d, double sm) {
  return WithShape<M, false>(
      g, id, h, [&](auto s, const auto &q) { return decltype(s)::DistanceToIn(q, p, d, sm); },
      [&](int type, const double *blk) { return DDistIn<BlockShapes(M)>(type, blk, p, d, sm); });
}
template <uint32_t M>
VGA_NAV double NDistOut(const NavDev &g, int id, const Head &h, V3 p, V3 d, double sm) {
  return WithShape<M, false>(
      g, id, h, [&](auto s, const auto &q) { return decltype(s)::DistanceToOut(q, p, d, sm); },
      [&](int type, const double *blk) { return DDistOut<BlockShapes(M)>(type, blk, p, d, sm); });
}
template <uint32_t M>
VGA_NAV double NSafeIn(const NavDev &g, int id, const Head &h, V3 p) {
  return WithShape<M, true>(
      g, id, h, [&](auto s, const auto &q) { return decltype(s)::SafetyToIn(q, p); },
      [&](int type, const double *blk) { return DSafeIn<BlockShapes(M)>(type, blk, p); });
}
template <uint32_t M>
VGA_NAV double NSafeOut(const NavDev &g, int id, const Head &h, V3 p) {
  return WithShape<M, true>(
      g, id, h, [&](auto s, const auto &q) { return decltype(s)::SafetyToOut(q, p); },
      [&](int type, const double *blk) { return DSafeOut<BlockShapes(M)>(type, blk, p); });
}

// ------------------------------------------------------------------ path
template <int D>
struct DPath {
  int v[D];
  int level;
  int boundary;
  VGA_NAV void Clear() {
#pragma unroll
    for (int k = 0; k < D; ++k) v[k] = -1;
    level = 0;
    boundary = 0;
  }
  VGA_NAV int Get(int l) const {
    int r = -1;
#pragma unroll
    for (int k = 0; k < D; ++k) r = (k == l) ? v[k] : r;
    return r;
  }
  VGA_NAV void Set(int l, int x) {
#pragma unroll
    for (int k = 0; k < D; ++k) v[k] = (k == l) ? x : v[k];
  }
  VGA_NAV int Top() const { return level > 0 ? Get(level - 1) : -1; }
  // The host checks that the geometry depth is at most D, so a push never
  // runs past the array (a path holds at most one volume per depth).
  VGA_NAV void Push(int x) {
    VGA_NAV_CHECK(level < D, "navigation path deeper than its register array");
    Set(level, x);
    ++level;
  }
  VGA_NAV void Pop() {
    if (level > 0) {
      --level;
      Set(level, -1);
    }
  }
};

// --------------------------------------------------------------- matrices
// Transformation3D::MultiplyFromRight (base/Transformation3D.h:662-708)
// with the right-hand placement's translation / rotation flags.
VGA_NAV void MultiplyFromRight(Xf &m, const Xf &rhs, int kind) {
  if (kind == kXfIdentity) return;
  if (kind == kXfTranslation || kind == kXfGeneral) {
    double t0 = m.t[0], t1 = m.t[1], t2 = m.t[2];
    t0 += m.r[0] * rhs.t[0];
    t0 += m.r[1] * rhs.t[1];
    t0 += m.r[2] * rhs.t[2];
    t1 += m.r[3] * rhs.t[0];
    t1 += m.r[4] * rhs.t[1];
    t1 += m.r[5] * rhs.t[2];
    t2 += m.r[6] * rhs.t[0];
    t2 += m.r[7] * rhs.t[1];
    t2 += m.r[8] * rhs.t[2];
    m.t[0] = t0;
    m.t[1] = t1;
    m.t[2] = t2;
  }
  if (kind == kXfRotation || kind == kXfGeneral) {
#pragma unroll
    for (int row = 0; row < 3; ++row) {
      const double tx = m.r[3 * row], ty = m.r[3 * row + 1], tz = m.r[3 * row + 2];
      double a = tx * rhs.r[0], b = tx * rhs.r[1], c = tx * rhs.r[2];
      a += ty * rhs.r[3];
      b += ty * rhs.r[4];
      c += ty * rhs.r[5];
      a += tz * rhs.r[6];
      b += tz * rhs.r[7];
      c += tz * rhs.r[8];
      m.r[3 * row] = a;
      m.r[3 * row + 1] = b;
      m.r[3 * row + 2] = c;
    }
  }
}

// The placement of volume id with code `code`: only the parts that are not
// the identity's are read.
VGA_NAV Xf LoadXf(const NavDev &g, int id, int code) {
  Xf x{{0., 0., 0.}, {1., 0., 0., 0., 1., 0., 0., 0., 1.}};
  if (code & (kNavMoves | kNavTurns)) {
    const NavRec &r = g.Nav(id);
#pragma unroll
    for (int i = 0; i < 3; ++i) x.t[i] = r.t[i];
    if (code & kNavTurns) {
      x.r[0] = r.r[0];
      x.r[1] = r.r[1];
      x.r[3] = r.r[2];
      x.r[4] = r.r[3];
    }
  } else if (code & kNavMatrix) {
    const Xf &m = g.Placed(id).xf;
#pragma unroll
    for (int i = 0; i < 3; ++i) x.t[i] = m.t[i];
#pragma unroll
    for (int i = 0; i < 9; ++i) x.r[i] = m.r[i];
  }
  return x;
}
VGA_NAV int KindOf(int code) { return (code >> kNavKindShift) & 3; }

// The unspecialised Transform (all terms), used on TopMatrix and on the
// pushed point after a boundary.
VGA_NAV V3 ApplyGeneric(const Xf &m, V3 p) { return Rotate(m, V3{p.x - m.t[0], p.y - m.t[1], p.z - m.t[2]}); }

// InverseTransformKernel<false> (base/Transformation3D.h:601-632).
VGA_NAV V3 InversePoint(const Xf &X, V3 l) {
  double x = X.t[0], y = X.t[1], z = X.t[2];
  x += l.x * X.r[0];
  x += l.y * X.r[1];
  x += l.z * X.r[2];
  y += l.x * X.r[3];
  y += l.y * X.r[4];
  y += l.z * X.r[5];
  z += l.x * X.r[6];
  z += l.y * X.r[7];
  z += l.z * X.r[8];
  return {x, y, z};
}

template <int D>
VGA_NAV Xf TopMatrix(const NavDev &g, const DPath<D> &s) {
  Xf m;
#pragma unroll
  for (int i = 0; i < 3; ++i) m.t[i] = 0.;
#pragma unroll
  for (int i = 0; i < 9; ++i) m.r[i] = (i % 4 == 0) ? 1. : 0.;
  for (int l = 1; l < s.level; ++l) {
    const int id = s.Get(l), code = g.Nav(id).code;
    if (KindOf(code) != kXfIdentity) MultiplyFromRight(m, LoadXf(g, id, code), KindOf(code));
  }
  return m;
}

// ---------------------------------------------------- daughters on the way
// The daughters of a volume that can meet a stretch of a ray (or hold a
// point), as bit masks over its daughter slots (vg_daughter_index.hpp): word
// w of a mask is slots dbegin + 64 w + bit.
struct Meet {
  int nd, words, axes;         // axes: NavRec::code
  const DaughterIndex *index;  // null: every daughter
  int l0, l1, l2, h0, h1, h2;  // rows of the stretch's ends in the tables

  VGA_NAV Meet(const NavDev &g, int code, int ix, int n, bool use) {
    nd = n;
    words = (nd + 63) >> 6;
    axes = code >> kNavAxesShift;
    index = use && ix >= 0 ? &g.Index(ix) : nullptr;
    l0 = l1 = l2 = h0 = h1 = h2 = 0;
  }
  VGA_NAV int Count() const { return axes & 3; }
  VGA_NAV int Row(const DaughterAxis &ax, float u) const {
    const float s = (u - ax.lo) * ax.inv;
    const int i = s < (float)(ax.slices - 1) ? (s > 0.f ? (int)s : 0) : ax.slices - 1;
    return ax.off + i * (2 * words);
  }
  template <int A, class F>
  VGA_NAV void Axis(F f, int &l, int &h) {
    if (A >= Count()) return;
    float u0, u1;
    f((axes >> (kNavCoordShift - kNavAxesShift + 2 * A)) & 3, u0, u1);
    const DaughterAxis ax = index->axis[A];
    l = Row(ax, u0);
    h = Row(ax, u1);
  }
  template <class F>
  VGA_NAV void Axes(F f) {
    if (!index) return;
    Axis<0>(f, l0, h0);
    Axis<1>(f, l1, h1);
    Axis<2>(f, l2, h2);
  }
  // The points within `reach` of p in every coordinate.
  VGA_NAV void Around(F3 p, float reach) {
    const float e = reach + 2e-6f * (Abs1(p) + reach);
    Axes([&](int c, float &u0, float &u1) {
      const float u = c == 0 ? p.x : c == 1 ? p.y : c == 2 ? p.z : __builtin_sqrtf(p.x * p.x + p.y * p.y);
      u0 = u - e;
      u1 = u + e;
    });
  }
  // The stretch p + t d, t0 <= t <= t1; its coordinates are widened by the
  // rounding of their float evaluation and by slack * t (Slack).
  VGA_NAV void Stretch(F3 p, F3 d, float t0, float t1, float slack) {
    const float e = 2e-6f * (Abs1(p) + t1) + slack * t1;
    const F3 a{p.x + t0 * d.x, p.y + t0 * d.y, p.z + t0 * d.z}, b{p.x + t1 * d.x, p.y + t1 * d.y, p.z + t1 * d.z};
    Axes([&](int c, float &u0, float &u1) {
      if (c < 3) {
        const float q = c == 0 ? a.x : c == 1 ? a.y : a.z, r = c == 0 ? b.x : c == 1 ? b.y : b.z;
        u0 = q < r ? q : r;
        u1 = q < r ? r : q;
      } else {
        // rho^2 is convex along the ray: largest at an end, smallest at the
        // closest approach to the axis.
        const float aa = d.x * d.x + d.y * d.y;
        float tm = aa > 0.f ? -(p.x * d.x + p.y * d.y) / aa : t0;
        tm = tm > t0 ? (tm < t1 ? tm : t1) : t0;
        const float xm = p.x + tm * d.x, ym = p.y + tm * d.y;
        const float ra = a.x * a.x + a.y * a.y, rb = b.x * b.x + b.y * b.y;
        u0 = __builtin_sqrtf(xm * xm + ym * ym);
        u1 = __builtin_sqrtf(ra < rb ? rb : ra);
      }
      u0 -= e;
      u1 += e;
    });
  }
  static VGA_NAV float Abs1(F3 p) { return __builtin_fabsf(p.x) + __builtin_fabsf(p.y) + __builtin_fabsf(p.z); }
  VGA_NAV uint64_t Full(int w) const { return nd - 64 * w >= 64 ? ~0ull : (1ull << (nd - 64 * w)) - 1; }
  VGA_NAV uint64_t Mask(const NavDev &g, int w) const {
    uint64_t m = Full(w);
    if (!index) return m;
    const int c = Count();
    if (c > 0) m &= g.Mask(l0 + w) & g.Mask(h0 + words + w);
    if (c > 1) m &= g.Mask(l1 + w) & g.Mask(h1 + words + w);
    if (c > 2) m &= g.Mask(l2 + w) & g.Mask(h2 + words + w);
    return m;
  }
};
// How far from a shape's extent a distance t to it can end, over t, where
// |d|^2 differs from 1 by `off`: the shapes' quadrics take d for a unit
// vector (1 - dz^2 for dx^2 + dy^2, t^2 for t^2 |d|^2), so the point p + t d
// that they find misses the surface's equation by off t^2 in the square of a
// length, and the surface by sqrt(off) t at most.  Planes take d as it is.
// Up to 1e-12 the margins of Stretch and Clip hold that; beyond kNearUnit
// every daughter is taken.
constexpr double kNearUnit = 1e-6;  // directions stored as float: 1.2e-7
VGA_NAV float Slack(double off) { return off < 1e-12 ? 0.f : __builtin_sqrtf(2.f * (float)off); }

// The part of a ray's way t >= 0 that lies in the box of all the index's
// daughters, widened by the rounding of t and the slack; false when there is
// none.
VGA_NAV bool Clip(const DaughterIndex &ix, F3 p, F3 d, float slack, float &t0, float &t1) {
  t0 = 0.f;
  t1 = kInfF;
  const float pv[3] = {p.x, p.y, p.z}, dv[3] = {d.x, d.y, d.z};
  float e = 4e-6f * Meet::Abs1(p);
  if (slack > 0.f) {  // t is at most about the way to the box's farthest corner
    float way = Meet::Abs1(p);
#pragma unroll
    for (int c = 0; c < 3; ++c) way += __builtin_fabsf(ix.lo[c]) + __builtin_fabsf(ix.hi[c]);
    e += 1.01f * slack * way;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const float a = ix.lo[c] - e - pv[c], b = ix.hi[c] + e - pv[c];
    if (__builtin_fabsf(dv[c]) > 1e-12f) {
      const float inv = 1.f / dv[c], u = a * inv, v = b * inv;
      t0 = t0 > (u < v ? u : v) ? t0 : (u < v ? u : v);
      t1 = t1 < (u < v ? v : u) ? t1 : (u < v ? v : u);
    } else if (a > 1e-3f || b < -1e-3f) {
      // Moves less than 1e-3 in this coordinate over 1e9.
      return false;
    }
  }
  t0 = t0 * (1.f - 4e-6f);
  t1 = t1 * (1.f + 4e-6f);
  return t0 <= t1;
}
// A point whose coordinates the index's floats hold.
VGA_NAV bool Finite(V3 p) { return p.Mag2() < 1e30; }

// ----------------------------------------------------------- locate family
// The daughter scan below tests only the daughters near the point, in the
// order of the full scan: a daughter that is not near cannot contain it.

// Where a track goes on: from volume vol, already on its path, at `point` of
// vol's frame.  vol < 0: nowhere.
struct Target {
  int vol, excluded;
  V3 point;
  bool down;
};

// Descends from the target: the first daughter in the scan's order that
// contains the point, and so on down; returns the deepest volume.  Rising
// daughter index (SimpleNavigator::LocatePoint) or, with `down`, falling and
// never into `excluded` (LocatePointExclVolume).
template <int D, uint32_t M>
VGA_NAV int Descend(const NavDev &g, Target t, DPath<D> &path) {
  bool deeper = t.vol >= 0;
  while (deeper) {
    const NavRec &C = g.Nav(t.vol);
    const int db = C.dbegin, nd = C.nd;
    if (nd <= 0) break;
    deeper = false;
    Meet near(g, C.code, C.index, nd, Finite(t.point));
    near.Around(F3{(float)t.point.x, (float)t.point.y, (float)t.point.z}, 0.f);
    for (int j = 0; j < near.words && !deeper; ++j) {
      const int w = t.down ? near.words - 1 - j : j;
      uint64_t m = near.Mask(g, w);
      while (m && !deeper) {
        const int bit = t.down ? 63 - __builtin_clzll(m) : __builtin_ctzll(m);
        m ^= 1ull << bit;
        const int nx = g.Daughter(db + 64 * w + bit);
        if (t.down && nx == t.excluded) continue;
        const Head h = LoadHead(g, nx);
        const V3 local = XfPointRt(LoadXf(g, nx, h.code), KindOf(h.code), t.point);
        if (NContains<M>(g, nx, h, local)) {
          path.Push(nx);
          t.point = local;
          t.vol = nx;
          deeper = true;
        }
      }
    }
  }
  return t.vol;
}

// SimpleNavigator::LocatePoint from the world.
template <int D, uint32_t M>
VGA_NAV Target FromWorld(const NavDev &g, V3 point, DPath<D> &path) {
  if (!NContains<M>(g, g.world, LoadHead(g, g.world), point)) return Target{-1, -1, point, false};
  path.Push(g.world);
  return Target{g.world, -1, point, false};
}

// LocatePoint in daughter nv, entered at `point` of its mother's frame.
template <int D>
VGA_NAV Target Into(const NavDev &g, int nv, V3 point, DPath<D> &path) {
  path.Push(nv);
  return Target{nv, -1, ApplyGeneric(LoadXf(g, nv, g.Nav(nv).code), point), false};
}

// RelocatePointFromPath: up to the first volume of the path that contains
// the point.
template <int D, uint32_t M>
VGA_NAV Target Relocate(const NavDev &g, V3 point, DPath<D> &path) {
  int mother = path.Top();
  while (mother >= 0) {
    const Head h = LoadHead(g, mother);
    if (NContains<M>(g, mother, h, point)) break;
    path.Pop();
    point = InversePoint(LoadXf(g, mother, h.code), point);
    mother = path.Top();
  }
  return Target{mother, mother, point, true};
}

// The navigators, as template arguments: each kernel carries the code of one
// (the mixed ABBox navigator is the ABBox one: its daughters are preselected
// in FP32 by the daughter index, and its results are the same).
enum NavWay : int { kWayAbbox, kWaySimple, kWayBasket, kWayAbboxSorted };
VGA_NAV constexpr bool Abbox(int way) { return way == kWayAbbox || way == kWayAbboxSorted; }

// ------------------------------------------------------------ ABBox search
constexpr float kReach = 4.f;  // growth of the searched stretch
constexpr float kNear = 8.f;   // a step within this many first stretches is searched at once
constexpr float kLeast = 1e-6f;  // shortest first stretch, as a share of the way to its begin

struct Ray {
  float p[3];
  float inv[3];
  int sign[3];
};

// IntersectCachedKernel2 on a float box, t0 = 0, t1 = +inf.  Max/Min are
// written as the reference's std::max / std::min (second operand when the
// first compares false), not fmaxf / fminf.
VGA_NAV float IntersectBox(const float *b, const Ray &r) {
  const float c0x = r.sign[0] ? b[3] : b[0], c1x = r.sign[0] ? b[0] : b[3];
  const float c0y = r.sign[1] ? b[4] : b[1], c1y = r.sign[1] ? b[1] : b[4];
  const float c0z = r.sign[2] ? b[5] : b[2], c1z = r.sign[2] ? b[2] : b[5];
  float tmin = (c0x - r.p[0]) * r.inv[0];
  const float tymax = (c1y - r.p[1]) * r.inv[1];
  if (tmin > tymax) return kInfF;
  float tmax = (c1x - r.p[0]) * r.inv[0];
  const float tymin = (c0y - r.p[1]) * r.inv[1];
  if (tymin > tmax) return kInfF;
  tmin = (tmin < tymin) ? tymin : tmin;
  tmax = (tymax < tmax) ? tymax : tmax;
  const float tzmin = (c0z - r.p[2]) * r.inv[2];
  const float tzmax = (c1z - r.p[2]) * r.inv[2];
  if ((tmin > tzmax) || (tzmin > tmax)) return kInfF;
  tmin = (tmin < tzmin) ? tzmin : tmin;
  tmax = (tzmax < tmax) ? tzmax : tmax;
  if (!((tmin < kInfF) && (tmax > 0.f))) tmin = kInfF;
  return tmin;
}

// Which of n boxes (64 at most) the ray hits (IntersectBox below infinity), as
// a bit mask: the full walk's box tests, without branches so that the loads of
// several boxes are in flight at once (traces of 262,144 tracks in a world of 6
// boxes 191 -> 119 us, of nine shapes 421 -> 292).
VGA_NAV uint64_t Hits(const NavDev &g, int slot, int n, const Ray &r) {
  uint64_t hit = 0;
#pragma unroll 4
  for (int k = 0; k < n; ++k) {
    const float *b = g.SlotBox(slot + k);
    float tmin = -kInfF, tmax = kInfF;
    bool miss = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float lo = ((r.sign[a] ? b[3 + a] : b[a]) - r.p[a]) * r.inv[a];
      const float hi = ((r.sign[a] ? b[a] : b[3 + a]) - r.p[a]) * r.inv[a];
      if (a > 0) miss |= (tmin > hi) | (lo > tmax);
      tmin = a > 0 && !(tmin < lo) ? tmin : lo;
      tmax = a > 0 && !(hi < tmax) ? tmax : hi;
    }
    miss |= !((tmin < kInfF) & (tmax > 0.f));
    hit |= (uint64_t)!miss << k;
  }
  return hit;
}

VGA_NAV Ray MakeRay(V3 lp, V3 ld) {
  Ray r;
  r.inv[0] = 1.f / (float)ld.x;
  r.inv[1] = 1.f / (float)ld.y;
  r.inv[2] = 1.f / (float)ld.z;
  r.p[0] = (float)lp.x;
  r.p[1] = (float)lp.y;
  r.p[2] = (float)lp.z;
#pragma unroll
  for (int i = 0; i < 3; ++i) r.sign[i] = r.inv[i] < 0;
  return r;
}

// Where the next stretch to search ends, given its begin T0, the end T of
// the one searched before (0: none) and the step known: at the step where
// that is near, else kReach times as far as before, and never beyond T1.
//
// The search ends: floats at T0 lie less than 1.2e-7 T0 apart, so a first
// stretch of kLeast T0 or more ends beyond T0, every later one is longer than
// the one before it, and T reaches T1 or the step (or infinity, which is T1).
VGA_NAV float Reach(const Meet &way, float T0, float T1, float T, double step) {
  if (!way.index) return 0.f;
  const float first = way.index->first, least = kLeast * T0;
  const float far = T0 + (T > 0.f ? kReach * (T - T0) : first > least ? first : least);
  const double to = step * (1. + 1e-6) + 1e-6;  // not below step as a float
  const float end = to <= (double)(T0 + kNear * first) || to <= (double)far ? (float)to : far;
  return end < T1 ? end : T1;
}

// Whether the best daughter's distance can depend on the step limit.  Only
// the Box and the Parallelepiped look at the limit in a way that can change
// an answer below it (the Polyhedron returns the limit in the place of a
// larger distance).  A Box's excesses exceed its distance only for a point
// inside it, or by rounding at nearly equal distances: the ABBox walk orders
// the first case and gives every daughter the first step as limit in the
// second; the Simple ones ask.
enum Limited : int { kLimitFree, kLimited, kSheared };  // kSheared: a Parallelepiped, looked at in the end
template <uint32_t M, int Way>
VGA_NAV int LimitedBy(const NavDev &g, int id, const Head &h, V3 p, double dist) {
  if constexpr (!Abbox(Way))
    if ((h.code & kNavFormMask) == kFormBox)
      return BoxS::LimitFree(BoxP{{h.s[0], h.s[1], h.s[2]}}, p, dist) ? kLimitFree : kLimited;
  if constexpr ((M >> VG_PARALLELEPIPED) & 1u)
    if ((h.code & kNavFormMask) == kFormGeneral && g.Nav(id).type == VG_PARALLELEPIPED) return kSheared;
  return kLimitFree;
}
// The Parallelepiped `id` at distance dist from lp of its mother's frame.
VGA_NAV bool ShearedLimitFree(const NavDev &g, int id, V3 lp, double dist) {
  const NavRec &r = g.Nav(id);
  const V3 p = XfPointRt(LoadXf(g, id, r.code), KindOf(r.code), lp);
  return ParaS::LimitFree(ParamView<ParaS>::Get(g.params + r.param_off), p, dist);
}

// The candidate walk of ABBoxNavigator::FindNextBoundaryAndStep
// (ABBoxNavigator.h:296-333) over daughters [db, de).  On entry `step`
// holds the mother's DistanceToOut (kInfinity if negative).  Returns 1 if
// the exact sorted-order walk was needed.  kWayAbboxSorted skips the
// order-free walk (used by the host-side checks of the exact walk).
//
// The walk searches the ray in growing stretches from its start: the
// daughters whose extents the stretch can meet, less those seen already, in
// index order; it ends with the first stretch that reaches the best step
// found.  Every daughter left lies beyond that step: it cannot contain the
// start, and its DistanceToIn exceeds the step, so it can neither win nor
// tie.  That argument needs the shapes' distances to be distances, which
// takes a unit direction, or nearly one and a wider stretch (Slack); any other
// direction takes every daughter at once.  (262,144 nested tracks with
// directions that were stored as float: 29.6 ms over every daughter, 4.6 with
// the stretch.)
//
// Every daughter is given the first step as limit, not the running one: a
// limit only takes away answers, and the winner under the first limit is the
// winner in any order, if its distance does not depend on the limit
// (Limited).
//
// Where the outcome does depend on the order the walk starts again and takes
// the hits in ascending (entry distance, daughter index) order, the order of
// a stable sort of the hit list, by repeated selection of the next one.  Both
// orders share the code that evaluates a daughter.
//
// SimpleNavigator's loop over the daughters (kWaySimple, kWayBasket) is the
// same search without the box tests: it takes the smallest DistanceToIn, of
// equal ones the daughter with the lowest index (an index-order loop with a
// strict comparison); where the winner depends on the limit, it walks again
// over every daughter in index order with the running step as limit.
template <uint32_t M, int Way>
VGA_NAV int Candidates(const NavDev &g, const Head &C, V3 lp, V3 ld, double &step, int &next) {
  const int db = C.dbegin;
  const Ray ray = MakeRay(lp, ld);
  const double step0 = step;
  const double off = Abs(ld.Mag2() - 1.);
  const float slack = Slack(off);
  Meet way(g, C.code, C.index, C.nd, (C.code & g.walks) && Finite(lp) && off < kNearUnit);
  // Word w of the daughters to look at.
  auto word = [&](int w) {
    if constexpr (Abbox(Way))
      if (!way.index) return Hits(g, db + 64 * w, C.nd - 64 * w < 64 ? C.nd - 64 * w : 64, ray);
    return way.Mask(g, w);
  };
  const F3 fp{ray.p[0], ray.p[1], ray.p[2]}, fd{(float)ld.x, (float)ld.y, (float)ld.z};
  // The stretch [T0, T] of the ray is searched next; beyond T1 it meets no
  // daughter.
  float T0 = 0.f, T1 = kInfF, T = 0.f;
  int w = 0;
  uint64_t m, seen = 0;
  if (way.index && (!Clip(*way.index, fp, fd, slack, T0, T1) || (double)T0 > step)) {
    m = 0;
    T = T1 = 0.f;
    w = way.words;
  } else {
    T = Reach(way, T0, T1, 0.f, step);
    way.Stretch(fp, fd, T0, T, slack);
    seen = m = word(0);
  }
  float behind = 0.f;
  bool sorted = Way == kWayAbboxSorted;
  int ties = 0;
  int limited = kLimitFree;  // of the best step
  float lastb = -kInfF;
  int lastk = -1;
  next = -1;
  while (true) {
    int k;
    float b;
    if (!sorted) {
      if (!m) {
        if (++w < way.words) {
          m = word(w);
          if (behind > 0.f) {
            Meet before = way;
            before.Stretch(fp, fd, T0, behind, slack);
            m &= ~before.Mask(g, w);
          }
        } else {
          if (!way.index || T >= T1 || step <= (double)T) {
            if constexpr ((M >> VG_PARALLELEPIPED) & 1u)
              if (limited == kSheared && ShearedLimitFree(g, g.Daughter(db + next), lp, step)) limited = kLimitFree;
            if ((!Abbox(Way) || ties <= 1) && limited == kLimitFree) return 0;
            step = step0;
            next = -1;
            if constexpr (Abbox(Way)) {
              sorted = true;
            } else {
              limited = kLimitFree;
              way.index = nullptr;
              behind = 0.f;
              w = 0;
              m = way.Mask(g, 0);
            }
            continue;
          }
          behind = T;
          T = Reach(way, T0, T1, T, step);
          way.Stretch(fp, fd, T0, T, slack);
          w = 0;
          const uint64_t all = way.Mask(g, 0);
          m = all & ~seen;
          seen = all;
        }
        continue;
      }
      k = 64 * w + __builtin_ctzll(m);
      m &= m - 1;
      if constexpr (Abbox(Way)) {
        b = IntersectBox(g.SlotBox(db + k), ray);
        if (!(b < kInfF)) continue;
      } else {
        b = 0.f;
      }
    } else {
      k = -1;
      b = kInfF;
      for (int j = 0; j < C.nd; ++j) {
        const float bj = IntersectBox(g.SlotBox(db + j), ray);
        const bool after = bj < kInfF && (bj > lastb || (bj == lastb && j > lastk));
        if (after && (k < 0 || bj < b)) {
          b = bj;
          k = j;
        }
      }
      if (k < 0 || step < (double)b) return 1;
      lastb = b;
      lastk = k;
    }
    const int cand = g.Daughter(db + k);
    const Head h = LoadHead(g, cand);
    const Xf x = LoadXf(g, cand, h.code);
    const V3 tp = XfPointRt(x, KindOf(h.code), lp);
    const bool within = b < 0.f && NContains<M>(g, cand, h, tp);
    if (within && sorted) {
      step = 0;
      next = k;
      return 1;
    }
    // The limit: the running step where the daughters come in the navigator's
    // own order, else the first one.
    const double sm = (Abbox(Way) ? sorted : !way.index) ? step : step0;
    const double dd = NDistIn<M>(g, cand, h, tp, XfDirRt(x, KindOf(h.code), ld), sm);
    if (!Abbox(Way)) {
      if ((dd < step || (dd == step && k < next)) && !(Way == kWaySimple && __builtin_isinf(dd))) {
        step = dd;
        next = k;
        if (way.index) limited = LimitedBy<M, Way>(g, cand, h, tp, dd);
      }
    } else if (sorted) {
      if (dd < step) {
        next = k;
        step = dd;
      }
    } else if (within || dd < 0. || dd < (double)b) {
      sorted = true;
      step = step0;
      next = -1;
    } else if (dd < step) {
      step = dd;
      next = k;
      ties = 1;
      limited = LimitedBy<M, Way>(g, cand, h, tp, dd);
    } else if (dd == step) {
      ++ties;
    }
  }
}

// One step of a track up to its relocation: the step length, the state's
// boundary flag, and where the track goes on (the state is complete when the
// target is nowhere).  `exact` is raised if the ABBox walk took the sorted
// order.  `vol` is the current volume; basket form: of the basket's first
// track.
//
// kWayAbbox, kWaySimple: FindNextBoundaryAndStep of the two navigators.
// kWayBasket: SimpleNavigator::FindNextBoundaryAndStep for baskets
// (navigation/SimpleNavigator.h:638-743), for one track of a basket whose
// current volume is `vol` (the top of the basket's first state, :672): the
// track's own TopMatrix (:660-667); the volume's DistanceToOut with pstep as
// step limit and no repair of values <= 0 (:678-679); DistanceToInMinimize
// over the daughters in order, each with the current distance as step
// limit, taken if strictly smaller (ShapeImplementationHelper.h:637-658);
// distance > pstep -> physics step off boundary (:708-713); otherwise push
// by 1e-9 and LocatePoint into the daughter or RelocatePointFromPath
// (:715-740).
template <int D, uint32_t M, int Way>
VGA_NAV Target StepTo(const NavDev &g, V3 gp, V3 gd, DPath<D> &nst, double pstep, double &step, int vol, int &exact) {
  const Target nowhere{-1, -1, V3{0., 0., 0.}, false};
  V3 lp, ld;
  {
    const Xf m = TopMatrix(g, nst);
    lp = ApplyGeneric(m, gp);
    ld = Rotate(m, gd);
  }
  const Head C = LoadHead(g, vol);
  int next = -1;
  step = NDistOut<M>(g, vol, C, lp, ld, pstep);
  if constexpr (Abbox(Way)) {
    if (step < 0.) step = kInfinity;
    if (C.nd > 0) exact += Candidates<M, Way>(g, C, lp, ld, step, next);
    if (step > pstep) {
      step = pstep;
      nst.boundary = 0;
      return nowhere;
    }
    nst.boundary = 1;
    if (step > 1E30) {
      step = 0;
      nst.Pop();
      return nowhere;
    }
  } else {
    if (Way == kWaySimple && step <= 0.) step = kInfinity;
    if (C.nd > 0) Candidates<M, Way>(g, C, lp, ld, step, next);
    if (Way == kWaySimple && step == kInfinity && pstep > 0.) {
      step = 0;
      nst.Pop();
      nst.boundary = 1;
      return nowhere;
    }
    if (step > pstep) {
      step = pstep;
      nst.boundary = 0;
      return nowhere;
    }
    nst.boundary = 1;
  }
  if (Way != kWayBasket && step < 0.) step = 0.;
  const double push = step + (Way == kWayBasket ? 1E-9 : 1E-6);
  const V3 np{ld.x * push + lp.x, ld.y * push + lp.y, ld.z * push + lp.z};
  if (next != -1) return Into(g, g.Daughter(C.dbegin + next), np, nst);
  return Relocate<D, M>(g, np, nst);
}

// The rest of the step: descend into the target; the ABBox navigator leaves a
// volume that a relocation found again (`vol`, the volume before the step).
template <int D, uint32_t M, int Way>
VGA_NAV void Arrive(const NavDev &g, const Target &t, int vol, DPath<D> &nst) {
  Descend<D, M>(g, t, nst);
  if (Abbox(Way) && t.down)
    while (nst.Top() == vol) nst.Pop();
}

// FindNextBoundaryAndStep on the state `nst` in place.
template <int D, uint32_t M, int Way>
VGA_NAV void FindNextBoundaryAndStep(const NavDev &g, V3 gp, V3 gd, DPath<D> &nst, double pstep, double &step,
                                     int vol) {
  int exact = 0;
  const Target t = StepTo<D, M, Way>(g, gp, gd, nst, pstep, step, vol, exact);
  Arrive<D, M, Way>(g, t, vol, nst);
}

// ABBoxNavigator::GetSafety: the smallest of the volume's SafetyToOut and
// its daughters' SafetyToIn.  Where the index says that every daughter's
// SafetyToIn is at least kSafetyShare of the point's distance from its extent
// in each coordinate, daughters farther than the least safety found so far
// allows are left out; else every daughter is looked at, all lanes the same
// one at a time.  Safety of 65,536 points in a world of 48 boxes 30 us looking
// at all of them, 18 with the index, 32 boxes 21 and 19.7, 20 boxes 13.4 and 21
// (see kSafeMin); scattered in the nested geometry 63 and 31.
constexpr float kSafetyShare = 0.7f;  // a box turned about z: 1 / sqrt(2)
template <int D, uint32_t M>
VGA_NAV double GetSafety(const NavDev &g, V3 gp, const DPath<D> &cur) {
  const Xf m = TopMatrix(g, cur);
  const V3 lp = ApplyGeneric(m, gp);
  const int cv = cur.Top();
  const Head C = LoadHead(g, cv);
  // Sets with shapes that need their parameter blocks read them for all (48
  // daughters with phi tubes, 65,536 points: 43.8 us through the records, 38.2).
  constexpr bool kBlocks = BlockShapes(M) != 0;
  double safety;
  if constexpr (kBlocks) {
    const PlacedRec &r = g.Placed(cv);
    safety = BlockSafeOut<M>(r.type, g.params + r.param_off, lp);
  } else {
    safety = NSafeOut<M>(g, cv, C, lp);
  }
  if (C.nd <= 0) return safety;
  if (!(C.code & kNavSafe) || !Finite(lp)) {
    int ahead = g.Daughter(C.dbegin);  // one daughter ahead: its record is loaded by it
    for (int k = 0; k < C.nd; ++k) {
      const int id = ahead;
      ahead = g.Daughter(C.dbegin + (k + 1 < C.nd ? k + 1 : k));
      double t;
      if constexpr (kBlocks) {
        const PlacedRec &r = g.Placed(id);
        t = BlockSafeIn<M>(r.type, g.params + r.param_off, XfPointRt(r.xf, r.xfkind, lp));
      } else {
        const Head h = LoadHead(g, id);
        t = NSafeIn<M>(g, id, h, XfPointRt(LoadXf(g, id, h.code), KindOf(h.code), lp));
      }
      safety = Min(safety, t);
    }
    return safety;
  }
  Meet near(g, C.code, C.index, C.nd, true);
  const F3 p{(float)lp.x, (float)lp.y, (float)lp.z};
  // SafetyToOut bounds the answer: a distance beyond it is not searched.
  float reach = near.index->near;
  if (safety * 1.5 + 1e-3 < (double)reach) reach = safety > 0. ? (float)(safety * 1.5) + 1e-3f : 1e-3f;
  near.Around(p, reach);
  int w = 0;
  uint64_t todo = near.Mask(g, 0), seen = todo;
  while (true) {
    if (!todo) {
      if (++w < near.words) {
        todo = near.Mask(g, w);  // (a daughter seen before changes nothing)
        continue;
      }
      // All nearer ones seen, all seen, or no number to compare with.
      if (safety <= (double)(kSafetyShare * reach) || !(reach < 1e30f) || (near.words == 1 && seen == near.Full(0)))
        return safety;
      reach = safety < (double)(2.f * reach) ? (float)(safety * 1.5) + 1e-3f : 4.f * reach;
      near.Around(p, reach);
      w = 0;
      const uint64_t all = near.Mask(g, 0);
      todo = all & ~seen;
      seen = all;
      continue;
    }
    const int id = g.Daughter(C.dbegin + 64 * w + __builtin_ctzll(todo));
    todo &= todo - 1;
    const Head h = LoadHead(g, id);
    safety = Min(safety, NSafeIn<M & kSafeShapes>(g, id, h, XfPointRt(LoadXf(g, id, h.code), KindOf(h.code), lp)));
  }
}

// The TraceTrack loop for one track (TraceTrack.cpp:170-220): locate from
// the world, then FindNextBoundaryAndStep and p += d * (step + 1e-6) until the
// state leaves the world or max_steps steps were taken.  Returns the number
// of steps; p ends at the final point.  The hash folds
// (new top id + 1) * 2 + boundary after every step.
template <int D, uint32_t M, int Way>
VGA_NAV int TraceOne(const NavDev &g, V3 &p, V3 d, double pstep, int max_steps, double &dist, uint64_t &h,
                     int &nexact) {
  DPath<D> cur;
  cur.Clear();
  Target t = FromWorld<D, M>(g, p, cur);
  int k = -1, vol = -1;
  nexact = 0;
  dist = 0;
  h = 1469598103934665603ULL;
  double step = 0;
  while (true) {
    Arrive<D, M, Way>(g, t, vol, cur);
    if (++k > 0) {
      dist += step;
      const double s = step + 1E-6;
      p = V3{p.x + d.x * s, p.y + d.y * s, p.z + d.z * s};
      const uint64_t v = (uint64_t)(uint32_t)(cur.Top() + 1) * 2ULL + (cur.boundary ? 1ULL : 0ULL);
      h = (h ^ v) * 1099511628211ULL;
    }
    if (!(cur.level > 0 && k < max_steps)) return k;
    vol = cur.Top();
    t = StepTo<D, M, Way>(g, p, d, cur, pstep, step, vol, nexact);
  }
}

// Tracks per wave of a navigation launch over n tracks, as a power of two: 64
// where that gives the chip two waves per SIMD, fewer for small baskets.  A
// wave runs as long as its slowest lane and through the code of every volume
// type that its lanes meet, so spreading few tracks over idle SIMDs shortens
// every step: 1,000 nested tracks 4.3 -> 1.9 ms, 4,000 2.3 ms with 1,024
// waves, 1.50 with 2,048 and 2.71 with 4,096; one step of 65,537 tracks with
// its locate and safety 85, 86 and 105 us.
constexpr uint64_t kNavWaves = 2048;
inline int LanesShift(uint64_t n) {
  int s = 0;
  while (s < 6 && (n >> s) > kNavWaves) ++s;
  return s;
}
// The lane's track under that shift (waves of 64 threads); n or more: none.
VGA_NAV uint64_t TrackOf(uint64_t thread, int shift, uint64_t n) {
  const uint64_t lane = thread & 63;
  return (lane >> shift) ? n : ((thread >> 6) << shift) + lane;
}

// The navigator's view of an uploaded geometry, for kernels of one WalkBit.
inline NavDev DeviceNav(const vg_geometry *g, int walks = 0) {
  return NavDev{g->d_nav,
                g->d_placed,
                g->d_params,
                g->d_slot_aabb,
                g->d_dindex,
                g->d_dmasks,
                g->world,
                (int32_t)g->placed.size(),
                (int32_t)g->daughters.size(),
                (int32_t)g->dindex.size(),
                (int32_t)g->dmasks.size(),
                walks};
}

// Calls f(D, M) with the path depth D (4, 8 or 16) that holds the geometry
// and the smallest shape set M of three that holds its shapes (both
// std::integral_constant).
template <class F>
void WithVariant(const vg_geometry *g, F f) {
  const uint32_t beyond = g->type_mask & ~kBasicShapes;
  auto shapes = [&](auto depth) {
    if (beyond == 0)
      f(depth, std::integral_constant<uint32_t, kBasicShapes>{});
    else if (beyond == kPhiTube)
      f(depth, std::integral_constant<uint32_t, kBasicShapes | kPhiTube>{});
    else
      f(depth, std::integral_constant<uint32_t, kAllShapes>{});
  };
  if (g->max_depth <= 4)
    shapes(std::integral_constant<int, 4>{});
  else if (g->max_depth <= 8)
    shapes(std::integral_constant<int, 8>{});
  else
    shapes(std::integral_constant<int, 16>{});
}

}  // namespace nav
}  // namespace vga
