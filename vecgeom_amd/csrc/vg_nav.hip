// Device navigation for gfx950: LocatePoint, FindNextBoundaryAndStep of the
// ABBox and Simple navigators, GetSafety and the TraceTrack loop, one track
// per lane.
//
// Reference behaviour followed (file:line):
//   NavigationState::TopMatrix      navigation/NavigationState.h:398-408
//   SimpleNavigator::LocatePoint    navigation/SimpleNavigator.h:205-241
//   LocatePointExclVolume           navigation/SimpleNavigator.h:246-289
//   RelocatePointFromPath           navigation/SimpleNavigator.h:292-321
//   SimpleNavigator FNBAS           navigation/SimpleNavigator.h:341-482
//   ABBoxNavigator FNBAS            navigation/ABBoxNavigator.h:201-424
//   ABBoxNavigator::GetSafety       navigation/ABBoxNavigator.h:428-452
//   GetHitCandidates (float boxes)  source/ABBoxManager.cpp:80-126
//   IntersectCachedKernel2          volumes/kernel/BoxImplementation.h:334-384
//   track loop                      test/globalbenchmarks/TraceTrack.cpp:170-220
//
// Layout and execution:
//  * what bounds it: a wave's tracks are in different volumes, so each lane
//    gathers its own volume records and the kernel lives on the texture
//    pipe and on latency, not on HBM (100 B per track) or FP64 issue.  Each
//    volume is therefore one 128-byte record (NavRec) of which only the
//    parts that matter are loaded, the daughters a step can meet come from
//    bit masks (vg_daughter_index.hpp: 1.0 box tests a step on the nested
//    geometry instead of 47), and each kernel carries the code of one
//    navigator and of the shapes the geometry uses.  Against full daughter
//    scans of 128-byte placements and parameter blocks, 524,288 nested
//    tracks went from 72.0 to 7.1 ms, 1,000 from 18.9 to 1.8 ms;
//  * a track's path lives in registers (template depth D, unrolled selects
//    instead of indexed private memory); the global-to-local matrix is
//    recomputed from the path every step, as TopMatrix does;
//  * the shape of a volume is dispatched at run time by a switch over the
//    record's form (the reference makes a virtual call);
//  * ABBox daughter loop.  The reference sorts the boxes hit by the ray by
//    entry distance and walks them in that order until a box starts beyond
//    the current step.  A lane cannot hold a sorted list of up to
//    hundreds of hits, so it first takes the daughters on its way in any
//    order, computing DistanceToIn for every hit box with stepMax = the
//    initial step.  The result equals the sorted walk when (a) no hit box
//    with a negative entry distance contains the point, (b) every
//    DistanceToIn result is >= 0 and >= its box entry distance (boxes bound
//    their shapes, so a box skipped by the sorted walk cannot hold a nearer
//    surface), (c) the smallest distance is reached by one daughter only,
//    and (d) that distance is the same under every larger stepMax.  The lane
//    checks (a)-(d) and otherwise redoes the step in exact sorted order by
//    repeated selection of the next (distance, index) pair.  (d) can fail for
//    the Parallelepiped (and for a Box by the rounding of a corner): its
//    early exit compares a sheared safety, which is no lower bound of the
//    distance, with stepMax.
#include <hip/hip_runtime.h>

#include <cstring>

#include "vg_nav_impl.hpp"

namespace vga {

namespace {

using namespace nav;

constexpr int kNavBlock = 128;

// ------------------------------------------------------------------ kernels
template <int D>
VGA_NAV void LoadState(const vg_nav_states &s, uint64_t i, DPath<D> &p) {
  p.level = s.level[i];
  p.boundary = s.boundary[i];
#pragma unroll
  for (int l = 0; l < D; ++l) p.v[l] = (l < s.depth && l < p.level) ? s.path[(uint64_t)l * s.capacity + i] : -1;
}

// A caller-supplied state is navigated only if its level fits the path
// array and every id on its path is a placed volume of this geometry.
template <int D>
VGA_NAV bool ValidState(const NavDev &g, const DPath<D> &p) {
  if (p.level < 1 || p.level > D) return false;
  bool ok = true;
#pragma unroll
  for (int l = 0; l < D; ++l) ok = ok && (l >= p.level || (p.v[l] >= 0 && p.v[l] < g.n_placed));
  return ok;
}

template <int D>
VGA_NAV void StoreState(const vg_nav_states &s, uint64_t i, const DPath<D> &p) {
  s.level[i] = p.level;
  s.boundary[i] = (uint8_t)p.boundary;
  for (int l = 0; l < s.depth; ++l) s.path[(uint64_t)l * s.capacity + i] = l < D ? p.Get(l) : -1;
}

// Occupancy floors of the fused trace kernel.  Its 168 VGPRs over the basic
// shapes hold three waves per SIMD; a fourth spills 47 registers, and the
// spills cost more of the memory pipe (which the gathers of volume records
// already keep busy) than the wave hides: 524,288 nested tracks 7.1 ms with
// 3, 9.4 with 4, 16.4 with 5.  With every shape the kernel would take 330
// registers and run one wave; two with some spills take the zoo geometry's
// 200,001 tracks from 350 to 260 us.
constexpr int TraceWaves(uint32_t m) { return (m & ~(kBasicShapes | kPhiTube)) == 0 ? 3 : 2; }

// The single-step kernels: with every shape two waves as above; over the
// basic shapes four at the price of a few spills (262,144 tracks: one ABBox
// step of the nested geometry 27 -> 23 us, among four daughters with phi tubes
// 36 -> 32, Simple 34 -> 29; 65,536 nested tracks 15 -> 16).
constexpr int StepWaves(uint32_t m) { return (m & ~(kBasicShapes | kPhiTube)) == 0 ? 4 : 2; }

template <int D, uint32_t M>
__global__ __launch_bounds__(kNavBlock) void LocateKernel(const NavDev g, const double *__restrict__ x,
                                                          const double *__restrict__ y, const double *__restrict__ z,
                                                          uint64_t n, const vg_nav_states s, int shift) {
  const uint64_t i = TrackOf((uint64_t)blockIdx.x * kNavBlock + threadIdx.x, shift, n);
  if (i >= n) return;
  DPath<D> p;
  p.Clear();
  const Target t = FromWorld<D, M>(g, V3{x[i], y[i], z[i]}, p);
  Descend<D, M>(g, t, p);
  StoreState(s, i, p);
}

struct StepArgs {
  const double *x, *y, *z, *dx, *dy, *dz, *pstep;
  double *step;
  uint64_t n;
  int32_t shift;  // LanesShift(n)
  int32_t pad;
};

template <int D, uint32_t M, int Way>
__global__ __launch_bounds__(kNavBlock) __attribute__((amdgpu_waves_per_eu(StepWaves(M)))) void StepKernel(
    const NavDev g, const StepArgs a, const vg_nav_states cur, const vg_nav_states nxt) {
  const uint64_t i = TrackOf((uint64_t)blockIdx.x * kNavBlock + threadIdx.x, a.shift, a.n);
  if (i >= a.n) return;
  DPath<D> o;
  LoadState(cur, i, o);
  double step = 0;
  const double ps = a.pstep ? a.pstep[i] : kInfinity;
  bool valid = ValidState(g, o);
  int vol = o.Top();
  if constexpr (Way == kWayBasket) {
    // The basket's current volume: the top of the first track's state.
    DPath<D> c0;
    LoadState(cur, 0, c0);
    valid = valid && ValidState(g, c0);
    vol = c0.Top();
  }
  if (valid)
    FindNextBoundaryAndStep<D, M, Way>(g, V3{a.x[i], a.y[i], a.z[i]}, V3{a.dx[i], a.dy[i], a.dz[i]}, o, ps, step, vol);
  else if (o.level != 0)
    // A state outside the world has no volume to step in and stays outside
    // (step 0); a malformed state is left as it is, with step NaN.
    step = __builtin_nan("");
  StoreState(nxt, i, o);
  a.step[i] = step;
}

template <int D, uint32_t M>
__global__ __launch_bounds__(kNavBlock) void SafetyKernel(
    const NavDev g, const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z, uint64_t n,
    const vg_nav_states s, double *__restrict__ out, int shift) {
  const uint64_t i = TrackOf((uint64_t)blockIdx.x * kNavBlock + threadIdx.x, shift, n);
  if (i >= n) return;
  DPath<D> c;
  LoadState(s, i, c);
  out[i] = ValidState(g, c) ? GetSafety<D, M>(g, V3{x[i], y[i], z[i]}, c) : (c.level == 0 ? 0. : __builtin_nan(""));
}

struct TraceArgs {
  const double *x, *y, *z, *dx, *dy, *dz;
  int32_t *nsteps;
  double *fx, *fy, *fz, *travelled;
  uint64_t *hash;
  int32_t *exact;
  uint64_t n;
  double pstep;
  int32_t max_steps;
  int32_t shift;  // LanesShift(n)
};


template <int D, uint32_t M, int Way>
__global__ __launch_bounds__(kNavBlock) __attribute__((amdgpu_waves_per_eu(TraceWaves(M)))) void TraceKernel(
    const NavDev g, const TraceArgs a) {
  const uint64_t i = TrackOf((uint64_t)blockIdx.x * kNavBlock + threadIdx.x, a.shift, a.n);
  if (i >= a.n) return;
  V3 p{a.x[i], a.y[i], a.z[i]};
  const V3 d{a.dx[i], a.dy[i], a.dz[i]};
  double dist;
  uint64_t h;
  int nexact;
  const int k = TraceOne<D, M, Way>(g, p, d, a.pstep, a.max_steps, dist, h, nexact);
  a.nsteps[i] = k;
  a.fx[i] = p.x;
  a.fy[i] = p.y;
  a.fz[i] = p.z;
  a.travelled[i] = dist;
  a.hash[i] = h;
  if (a.exact) a.exact[i] = nexact;
}

unsigned Blocks(uint64_t n, int shift) {
  const uint64_t per = (uint64_t)(kNavBlock / 64) << shift;
  return (unsigned)((n + per - 1) / per);
}

}  // namespace

int NavLocate(const vg_geometry *g, const double *x, const double *y, const double *z, uint64_t n,
              const vg_nav_states &s, hipStream_t st) {
  if (n == 0) return VG_OK;
  const int shift = LanesShift(n);
  WithVariant(g, [&](auto D, auto M) {
    hipLaunchKernelGGL((LocateKernel<D.value, M.value>), dim3(Blocks(n, shift)), dim3(kNavBlock), 0, st, DeviceNav(g),
                       x, y, z, n, s, shift);
  });
  return CheckHip(hipGetLastError(), "locate launch");
}

int NavStep(const vg_geometry *g, int kind, const double *x, const double *y, const double *z, const double *dx,
            const double *dy, const double *dz, const double *pstep, uint64_t n, const vg_nav_states &cur,
            const vg_nav_states &nxt, double *step, hipStream_t st) {
  if (n == 0) return VG_OK;
  const bool abbox = kind != VG_NAV_SIMPLE && kind != VG_NAV_SIMPLE_BASKET;
  const int walks = WalkBit(abbox, n < kBigStep ? kWalkStep : kWalkBigStep);
  // The Simple navigators' loop over the world's daughters evaluates all of
  // them, all lanes the same one at a time: full waves, as for the safety.
  const NavRec &world = g->nav[g->world];
  const bool loop = !abbox && world.nd >= 3 && !(world.code & walks);
  const StepArgs a{x, y, z, dx, dy, dz, pstep, step, n, loop ? 6 : LanesShift(n), 0};
  const dim3 blocks(Blocks(n, a.shift)), threads(kNavBlock);
  if (kind == VG_NAV_SIMPLE)
    WithVariant(g, [&](auto D, auto M) {
      hipLaunchKernelGGL((StepKernel<D.value, M.value, kWaySimple>), blocks, threads, 0, st, DeviceNav(g, walks), a, cur, nxt);
    });
  else if (kind == VG_NAV_SIMPLE_BASKET)
    WithVariant(g, [&](auto D, auto M) {
      hipLaunchKernelGGL((StepKernel<D.value, M.value, kWayBasket>), blocks, threads, 0, st, DeviceNav(g, walks), a, cur, nxt);
    });
  else
    WithVariant(g, [&](auto D, auto M) {
      hipLaunchKernelGGL((StepKernel<D.value, M.value, kWayAbbox>), blocks, threads, 0, st, DeviceNav(g, walks), a, cur, nxt);
    });
  return CheckHip(hipGetLastError(), "step launch");
}

int NavSafety(const vg_geometry *g, const double *x, const double *y, const double *z, uint64_t n,
              const vg_nav_states &s, double *out, hipStream_t st) {
  if (n == 0) return VG_OK;
  // Where lanes look at every daughter, all the same one at a time, a wave
  // costs the whole loop however few its tracks: full waves (4,096 points in a
  // world of 96 cones 298 us with two tracks a wave, 93 with 64).
  const int shift = g->safety_scans ? 6 : LanesShift(n);
  WithVariant(g, [&](auto D, auto M) {
    hipLaunchKernelGGL((SafetyKernel<D.value, M.value>), dim3(Blocks(n, shift)), dim3(kNavBlock), 0, st, DeviceNav(g),
                       x, y, z, n, s, out, shift);
  });
  return CheckHip(hipGetLastError(), "safety launch");
}

int NavTrace(const vg_geometry *g, int kind, const double *x, const double *y, const double *z, const double *dx,
             const double *dy, const double *dz, uint64_t n, double pstep, int max_steps, int32_t *nsteps, double *fx,
             double *fy, double *fz, double *travelled, uint64_t *hash, int32_t *exact, hipStream_t st) {
  if (n == 0) return VG_OK;
  const TraceArgs a{x, y, z, dx, dy, dz, nsteps, fx, fy, fz, travelled, hash, exact, n, pstep, max_steps, LanesShift(n)};
  const dim3 blocks(Blocks(n, a.shift)), threads(kNavBlock);
  if (kind == VG_NAV_SIMPLE)
    WithVariant(g, [&](auto D, auto M) {
      hipLaunchKernelGGL((TraceKernel<D.value, M.value, kWaySimple>), blocks, threads, 0, st, DeviceNav(g, WalkBit(kind != VG_NAV_SIMPLE, kWalkTrace)), a);
    });
  else
    WithVariant(g, [&](auto D, auto M) {
      hipLaunchKernelGGL((TraceKernel<D.value, M.value, kWayAbbox>), blocks, threads, 0, st, DeviceNav(g, WalkBit(kind != VG_NAV_SIMPLE, kWalkTrace)), a);
    });
  return CheckHip(hipGetLastError(), "trace launch");
}

}  // namespace vga
