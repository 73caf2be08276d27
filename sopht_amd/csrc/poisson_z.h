// What the z passes of the Poisson solver share (poisson_3d.hip, poisson_zrows.hip).
#pragma once

#include "poisson_slab.h"

// Line lengths 2 nz of the three-pass schedule (longer z lines leave the z pass without
// registers for its next rows).
#define SOPHT_ZROW_LENGTHS(X) \
  X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

namespace sopht {

inline bool zrow_length_supported(int64_t L) {
#define X(n) if (L == n) return true;
  SOPHT_ZROW_LENGTHS(X)
#undef X
  return false;
}

// The z pass of the three-pass schedule over all components; jobs per workgroup as tuned.
int poisson_z_rows(int64_t LZ, SlabGeom g, Cplx<float>* H, const float* ghat, const Cplx<float>* tw, hipStream_t s,
                   int jobs);
int poisson_z_rows(int64_t LZ, SlabGeom g, Cplx<double>* H, const double* ghat, const Cplx<double>* tw, hipStream_t s,
                   int jobs);

// Jobs per workgroup where nothing was timed.
#ifndef SOPHT_ZROW_JOBS
#define SOPHT_ZROW_JOBS 6
#endif
constexpr int kZrowJobs = SOPHT_ZROW_JOBS;

namespace {

// Waves per SIMD the z pass is compiled for (its VGPR budget: 128 in FP32; a budget of 80,
// for three 512-thread workgroups per CU, spills).
template <typename T>
constexpr int kZconvWaves = sizeof(T) == 4 ? 4 : 2;
// more elements per thread need more registers: twelve (L = 384, 768) one wavefront less per
// SIMD, sixteen (L = 1024) two less
template <typename T, int L>
constexpr int kZconvWavesFor = sizeof(T) != 4 ? kZconvWaves<T>
                               : (LinePlan<L>::E >= 16 ? 2 : (LinePlan<L>::E > 8 ? 3 : kZconvWaves<T>));
// Three-stage line plans: the twiddles of a thread's butterflies in the second and last stages
// depend on the thread only, so a z-pass workgroup computes them once for all its pencils.
template <typename R>
struct Plan3 {
  static constexpr bool ok = false;
  static constexpr int r0 = 0, r1 = 0, r2 = 0;
};
template <int A, int B, int C>
struct Plan3<rfft::Radices<A, B, C>> {
  static constexpr bool ok = true;
  static constexpr int r0 = A, r1 = B, r2 = C;
};
template <int L>
constexpr bool last_twiddles_hoisted() {  // the E = 8 plans (L = 128, 256, 512): 24-28 VGPRs
  using P = Plan3<typename LinePlan<L>::R>;
  return P::ok && LinePlan<L>::E == 8;
}
constexpr int at_least_1(int v) { return v > 0 ? v : 1; }

}  // namespace
}  // namespace sopht
