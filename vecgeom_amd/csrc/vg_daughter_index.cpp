// Host-side construction of the daughter indexes (vg_daughter_index.hpp).
#include "vg_daughter_index.hpp"

#include <algorithm>
#include <cmath>

#include "shapes.hpp"
#include "vg_internal.hpp"

namespace vga {

namespace {

constexpr int kMinSlices = 32, kMaxSlices = 512;
constexpr int kSamples = 256;  // points at which coordinates are compared
// First stretch of a ray to search, as a share of the diagonal of the
// daughters' extent.
constexpr double kFirst = 1. / 512;
// First distance to search for a safety, as a share of the diagonal over the
// cube root of the number of daughters (the pitch of a cubic grid is 0.58):
// 262,144 points scattered in the nested geometry 43 us from 1/512 of the
// diagonal, 38 with 0.12, 49 with 0.2, 70 with 0.35.
constexpr double kNearShare = 0.12;

// Local extent along z and from the z axis of a shape that turns about z
// (rlo is 0 where the hollow's depth is not bounded simply).
bool RadialExtent(int type, const double *b, double *rlo, double *rhi, double *zlo, double *zhi) {
  switch (type) {
    case VG_TUBE: {
      const TubeP &t = *reinterpret_cast<const TubeP *>(b);
      *rlo = t.rmin; *rhi = t.rmax; *zlo = -t.z; *zhi = t.z;
      return true;
    }
    case VG_CONE: {
      const ConeP &c = *reinterpret_cast<const ConeP *>(b);
      *rlo = std::min(c.rmin1, c.rmin2); *rhi = std::max(c.rmax1, c.rmax2); *zlo = -c.dz; *zhi = c.dz;
      return true;
    }
    case VG_TORUS: {
      const TorusP &t = *reinterpret_cast<const TorusP *>(b);
      *rlo = std::max(0., t.rtor - t.rmax); *rhi = t.rtor + t.rmax; *zlo = -t.rmax; *zhi = t.rmax;
      return true;
    }
    case VG_POLYHEDRON: {
      // Its Contains does not test the phi section, so the whole bounding
      // tube counts (the tube's outer radius is the corners').
      const PolyhedronP q{b};
      const TubeP &t = PolyhedronS::Tube(q);
      *rlo = 0.; *rhi = t.rmax; *zlo = b[4] - t.z; *zhi = b[4] + t.z;
      return true;
    }
  }
  return false;
}

}  // namespace

DaughterExtent ExtentInMother(int type, const double *blk, const Xf &X, const double elo[3], const double ehi[3],
                              const double box[6]) {
  double lo[3] = {elo[0], elo[1], elo[2]}, hi[3] = {ehi[0], ehi[1], ehi[2]};
  double rlo = 0., rhi = kInfinity, zlo, zhi;
  const bool radial = RadialExtent(type, blk, &rlo, &rhi, &zlo, &zhi);
  if (radial) {  // the full turn, whatever the phi section
    lo[0] = lo[1] = -rhi;
    hi[0] = hi[1] = rhi;
    lo[2] = std::min(lo[2], zlo);
    hi[2] = std::max(hi[2], zhi);
  }
  if (type == VG_TRD) {  // its extent takes dy1 for the upper x bound
    const TrdP &t = *reinterpret_cast<const TrdP *>(blk);
    hi[0] = std::max(hi[0], Max(t.dx1, t.dx2));
  }
  DaughterExtent e;
  for (int a = 0; a < 3; ++a) {
    double c = X.t[a], w = 0;
    for (int i = 0; i < 3; ++i) {
      c += X.r[3 * a + i] * 0.5 * (lo[i] + hi[i]);
      w += std::fabs(X.r[3 * a + i]) * 0.5 * (hi[i] - lo[i]);
    }
    e.lo[a] = std::min(c - w, box[a]);
    e.hi[a] = std::max(c + w, box[3 + a]);
  }
  // rho: about the projected centre of the box's corners, tightened where the
  // daughter's z axis is parallel to the mother's.
  double cx = X.t[0], cy = X.t[1], reach = 0;
  for (int i = 0; i < 3; ++i) {
    cx += X.r[i] * 0.5 * (lo[i] + hi[i]);
    cy += X.r[3 + i] * 0.5 * (lo[i] + hi[i]);
  }
  double corner_max = 0;
  for (int k = 0; k < 8; ++k) {
    double x = X.t[0], y = X.t[1];
    for (int i = 0; i < 3; ++i) {
      const double l = (k >> i) & 1 ? hi[i] : lo[i];
      x += X.r[i] * l;
      y += X.r[3 + i] * l;
    }
    reach = std::max(reach, std::hypot(x - cx, y - cy));
    corner_max = std::max(corner_max, std::hypot(x, y));
  }
  const double c = std::hypot(cx, cy);
  e.lo[3] = std::max(0., c - reach);
  e.hi[3] = corner_max;
  const bool upright = std::fabs(X.r[2]) < 1e-12 && std::fabs(X.r[5]) < 1e-12 && std::fabs(X.r[6]) < 1e-12 &&
                       std::fabs(X.r[7]) < 1e-12 && std::fabs(std::fabs(X.r[8]) - 1.) < 1e-12;
  if (upright) {
    // The rectangle's nearest point to the axis, in the local frame.
    const double ax = -(X.r[0] * X.t[0] + X.r[3] * X.t[1]), ay = -(X.r[1] * X.t[0] + X.r[4] * X.t[1]);
    const double dx = std::max({0., lo[0] - ax, ax - hi[0]}), dy = std::max({0., lo[1] - ay, ay - hi[1]});
    e.lo[3] = std::max(e.lo[3], std::hypot(dx, dy));
    if (radial) {
      const double d = std::hypot(X.t[0], X.t[1]);
      e.lo[3] = std::max({e.lo[3], rlo - d, d - rhi});
      e.hi[3] = std::min(e.hi[3], d + rhi);
    }
  }
  e.safe = type == VG_ORB || (type == VG_BOX && upright);
  if (type == VG_TUBE && upright && X.t[0] == 0. && X.t[1] == 0.)
    e.safe = reinterpret_cast<const TubeP *>(blk)->hasPhi == 0;
  // The float box may reach beyond the shape (1e-3 padding); rho bounds the
  // shape itself, which is what distances and containment depend on.
  return e;
}

namespace {

// Slices per coordinate: about eight a daughter, fewer where the masks of
// very many daughters would take too much memory.
int Slices(int nd) {
  const int words = (nd + 63) / 64;
  int n = kMinSlices;
  while (n < kMaxSlices && n < 8 * nd) n *= 2;
  while (n > kMinSlices && (double)n * words > 64 * 1024) n /= 2;
  return n;
}

}  // namespace

size_t DaughterIndexWords(int nd) {
  return (size_t)kIndexAxes * Slices(nd) * 2 * (size_t)((nd + 63) / 64);
}

DaughterIndex BuildDaughterIndex(const std::vector<DaughterExtent> &d, std::vector<uint64_t> &masks, IndexAxes *axes) {
  DaughterIndex ix{};
  *axes = IndexAxes{};
  const int nd = (int)d.size();
  const int words = (nd + 63) / 64;
  for (const auto &e : d)
    for (int c = 0; c < kIndexCoords; ++c)
      if (!(std::fabs(e.lo[c]) < 1e30 && std::fabs(e.hi[c]) < 1e30)) return ix;  // no coordinate is looked up
  double lo[kIndexCoords], hi[kIndexCoords];
  for (int c = 0; c < kIndexCoords; ++c) {
    lo[c] = kInfinity;
    hi[c] = -kInfinity;
    for (const auto &e : d) {
      lo[c] = std::min(lo[c], e.lo[c]);
      hi[c] = std::max(hi[c], e.hi[c]);
    }
  }
  double diag = 0, size = 0;
  for (int c = 0; c < 3; ++c) {
    diag += (hi[c] - lo[c]) * (hi[c] - lo[c]);
    size = std::max({size, std::fabs(lo[c]), std::fabs(hi[c])});
  }
  diag = std::sqrt(diag);
  const int n = Slices(nd);
  ix.first = (float)std::max(diag * kFirst, 1e-6);
  ix.near = (float)std::max(diag * kNearShare / std::cbrt((double)nd), 1e-6);
  axes->safe = true;
  for (const auto &e : d) axes->safe &= e.safe;
  for (int c = 0; c < 3; ++c) {
    const double pad = 1e-3 + 1e-6 * size;
    ix.lo[c] = (float)(lo[c] - pad);
    ix.hi[c] = (float)(hi[c] + pad);
  }

  // Tables of every coordinate, by running ORs over the slices.
  const size_t row = 2 * (size_t)words, table = row * n;
  std::vector<uint64_t> t[kIndexCoords];
  float flo[kIndexCoords], finv[kIndexCoords];
  for (int c = 0; c < kIndexCoords; ++c) {
    const double range = std::max(hi[c] - lo[c], 1e-3);
    flo[c] = (float)lo[c];
    finv[c] = (float)(n / range);
    // Rounding of the slice arithmetic (a few 1e-7 of n slices), of lo and
    // inv themselves and of a coordinate of magnitude up to `size`.
    const double pad = 1e-5 + 4e-6 * size + 1e-5 * range;
    t[c].assign(table, 0);
    for (int k = 0; k < nd; ++k) {
      const uint64_t bit = 1ull << (k & 63);
      const double b = std::floor((d[k].lo[c] - pad - lo[c]) / range * n);
      const double e = std::floor((d[k].hi[c] + pad - lo[c]) / range * n);
      const int i0 = b > 0 ? std::min((int)b, n - 1) : 0, i1 = e < n - 1 ? std::max((int)e, 0) : n - 1;
      t[c][i1 * row + (k >> 6)] |= bit;          // ends here ...
      t[c][i0 * row + words + (k >> 6)] |= bit;  // begins here ...
    }
    for (int i = n - 1; i > 0; --i)  // ... or beyond
      for (int w = 0; w < words; ++w) t[c][(i - 1) * row + w] |= t[c][i * row + w];
    for (int i = 1; i < n; ++i)  // ... or before
      for (int w = 0; w < words; ++w) t[c][i * row + words + w] |= t[c][(i - 1) * row + words + w];
  }

  // Take the coordinates that tell daughters apart: greedily, each must cut
  // the mean number of daughters a point can be in by a tenth.
  // Measured at points of a fixed low-discrepancy sequence in the extent of
  // the daughters, on the first 64 of them.
  struct Samples {
    double f[kSamples][3];
    Samples() {
      static const double g[3] = {0.8191725133961645, 0.6710436067037893, 0.5497004779019703};
      for (int s = 0; s < kSamples; ++s)
        for (int i = 0; i < 3; ++i) f[s][i] = std::fmod(0.5 + g[i] * (s + 1), 1.);
    }
  };
  static const Samples samples;
  std::vector<uint64_t> at[kIndexCoords];  // the masks at every sample
  for (int c = 0; c < kIndexCoords; ++c) {
    at[c].resize(kSamples);
    for (int s = 0; s < kSamples; ++s) {
      double p[3];
      for (int i = 0; i < 3; ++i) p[i] = lo[i] + (hi[i] - lo[i]) * samples.f[s][i];
      const double u = c < 3 ? p[c] : std::sqrt(p[0] * p[0] + p[1] * p[1]);
      const size_t i = (size_t)std::min<double>(n - 1, std::max(0., (u - lo[c]) * finv[c]));
      at[c][s] = t[c][i * row] & t[c][i * row + words];
    }
  }
  bool taken[kIndexCoords] = {};
  double left = std::min(nd, 64);
  std::vector<uint64_t> cur(kSamples, ~0ull);
  while (axes->count < kIndexAxes) {
    int best = -1;
    double best_mean = 0.9 * left;
    for (int c = 0; c < kIndexCoords; ++c) {
      if (taken[c]) continue;
      double mean = 0;
      for (int s = 0; s < kSamples; ++s) mean += __builtin_popcountll(cur[s] & at[c][s]);
      mean /= kSamples;
      if (mean < best_mean) {
        best_mean = mean;
        best = c;
      }
    }
    if (best < 0) break;
    taken[best] = true;
    ix.axis[axes->count] = DaughterAxis{flo[best], finv[best], (int32_t)masks.size(), n};
    axes->coord[axes->count++] = best;
    masks.insert(masks.end(), t[best].begin(), t[best].end());
    for (int s = 0; s < kSamples; ++s) cur[s] &= at[best][s];
    left = best_mean;
  }
  return ix;
}

}  // namespace vga
