// Kernels of the Boolean basket queries, for one set of operand shapes; each
// set is compiled in a file of its own (vg_boolean.hip, vg_boolean_torus.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "shapes_boolean.hpp"
#include "vg_internal.hpp"

namespace vga {

namespace {

constexpr int kBoolBlock = 128;

// Bound by latency and occupancy: the largest operand shape sets the
// registers of the whole switch.  With the Torus's quartic the distances take
// 280 VGPRs and run one wave per SIMD; without it 199, and floors of three
// waves (168) and two with the Torus, at the price of some spills, took the
// 30 queries on the five test volumes (262,144 points each) from 444 to
// 355 us of kernel time (DistanceToIn of the Polyhedron intersection 133 -> 77).
template <int Q, uint32_t M>
__global__ __launch_bounds__(kBoolBlock) __attribute__((amdgpu_waves_per_eu(M == kBoolAll ? 2 : 3))) void BooleanQueryKernel(
    const double *__restrict__ blk, const Xf X, int xfkind, const QArgs a) {
  const uint64_t i = (uint64_t)blockIdx.x * kBoolBlock + threadIdx.x;
  if (i >= a.n) return;
  using B = BooleanT<M>;
  const BooleanP P{blk};
  const V3 p{a.x[i], a.y[i], a.z[i]};
  V3 d{0, 0, 0};
  if constexpr (Q == kQDistIn || Q == kQDistInMin || Q == kQDistOut || Q == kQPlacedDistOut)
    d = V3{a.dx[i], a.dy[i], a.dz[i]};
  double *od = reinterpret_cast<double *>(a.out);
  if constexpr (Q == kQContains) {
    reinterpret_cast<uint8_t *>(a.out)[i] = B::Contains(P, XfPointRt(X, xfkind, p)) ? 1 : 0;
  } else if constexpr (Q == kQInside) {
    reinterpret_cast<int32_t *>(a.out)[i] = B::Inside(P, XfPointRt(X, xfkind, p));
  } else if constexpr (Q == kQDistIn) {
    const double sm = a.sm ? a.sm[i] : kInfinity;
    od[i] = B::DistanceToIn(P, XfPointRt(X, xfkind, p), XfDirRt(X, xfkind, d), sm);
  } else if constexpr (Q == kQDistInMin) {
    const double cur = od[i];
    const double r = B::DistanceToIn(P, XfPointRt(X, xfkind, p), XfDirRt(X, xfkind, d), cur);
    if (r < cur) {
      od[i] = r;
      a.next[i] = a.did;
    }
  } else if constexpr (Q == kQDistOut) {
    const double sm = a.sm ? a.sm[i] : kInfinity;
    const double r = B::DistanceToOut(P, p, d, sm);
    od[i] = r;
    if (a.next) a.next[i] = (r < sm) ? -1 : -2;
  } else if constexpr (Q == kQPlacedDistOut) {
    const double sm = a.sm ? a.sm[i] : kInfinity;
    od[i] = B::DistanceToOut(P, XfPointRt(X, xfkind, p), XfDirRt(X, xfkind, d), sm);
  } else if constexpr (Q == kQSafeIn) {
    od[i] = B::SafetyToIn(P, XfPointRt(X, xfkind, p));
  } else if constexpr (Q == kQSafeInMin) {
    const double cur = od[i], r = B::SafetyToIn(P, XfPointRt(X, xfkind, p));
    od[i] = (r < cur) ? r : cur;
  } else if constexpr (Q == kQSafeOut) {
    od[i] = B::SafetyToOut(P, p);
  } else {  // kQSafeOutMin
    const double cur = od[i], r = B::SafetyToOut(P, p);
    od[i] = (r < cur) ? r : cur;
  }
}

template <int Q, uint32_t M>
int LaunchBooleanKernel(const double *blk, const PlacedRec &pr, const QArgs &a, hipStream_t s) {
  const unsigned blocks = (unsigned)((a.n + kBoolBlock - 1) / kBoolBlock);
  hipLaunchKernelGGL((BooleanQueryKernel<Q, M>), dim3(blocks), dim3(kBoolBlock), 0, s, blk, pr.xf, (int)pr.xfkind, a);
  return CheckHip(hipGetLastError(), "Boolean query launch");
}

template <uint32_t M>
int LaunchBooleanSet(int q, const double *blk, const PlacedRec &pr, const QArgs &a, hipStream_t s) {
  switch (q) {
    case kQContains: return LaunchBooleanKernel<kQContains, M>(blk, pr, a, s);
    case kQInside: return LaunchBooleanKernel<kQInside, M>(blk, pr, a, s);
    case kQDistIn: return LaunchBooleanKernel<kQDistIn, M>(blk, pr, a, s);
    case kQDistInMin: return LaunchBooleanKernel<kQDistInMin, M>(blk, pr, a, s);
    case kQDistOut: return LaunchBooleanKernel<kQDistOut, M>(blk, pr, a, s);
    case kQPlacedDistOut: return LaunchBooleanKernel<kQPlacedDistOut, M>(blk, pr, a, s);
    case kQSafeIn: return LaunchBooleanKernel<kQSafeIn, M>(blk, pr, a, s);
    case kQSafeInMin: return LaunchBooleanKernel<kQSafeInMin, M>(blk, pr, a, s);
    case kQSafeOut: return LaunchBooleanKernel<kQSafeOut, M>(blk, pr, a, s);
    case kQSafeOutMin: return LaunchBooleanKernel<kQSafeOutMin, M>(blk, pr, a, s);
  }
  return SetError(VG_ERR_INVALID, "unknown query");
}

}  // namespace

// Booleans with a Torus operand (vg_boolean_torus.hip).
int LaunchBooleanTorus(int q, const double *blk, const PlacedRec &pr, const QArgs &a, hipStream_t s);

}  // namespace vga
