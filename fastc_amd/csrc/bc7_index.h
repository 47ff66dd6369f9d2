// The scalar index arithmetic of BC7's pixel pass (bc7_encode.hip): index
// weights, the scaled reciprocal of an endpoint distance and the neighbouring
// indices of a projection.  Also compiled for the host, where
// tests/cpp/index_test.cpp walks it over every distance; there the hardware's
// approximate reciprocal is the exact one moved by host_rcp_ulps.
#pragma once

#include <stdint.h>

#if defined(__HIP__)
#define FH_INDEX_FN __host__ __device__ __forceinline__
#else
#include <math.h>
#define FH_INDEX_FN inline
#endif

namespace fh {
namespace bc7 {

#if !defined(__HIP__)
static int host_rcp_ulps = 0;
#endif

// Within 1 ulp of 1 / x on the device.
FH_INDEX_FN float approx_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#elif defined(__HIP__)
  return 1.0f / x;
#else
  float r = 1.0f / x;
  for (int k = 0; k < host_rcp_ulps; k++) r = nextafterf(r, 2.0f);
  for (int k = 0; k > host_rcp_ulps; k--) r = nextafterf(r, 0.0f);
  return r;
#endif
}

FH_INDEX_FN float clamp01(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f);
#else
  return x < 0.0f ? 0.0f : (x > 1.0f ? 1.0f : x);
#endif
}

// Weight of the second endpoint at index j for nb = 4, 8, 16 entries:
// (64 j + (nb - 1) / 2) / (nb - 1) by a multiply-shift, equal to
// kInterpolationValues (Compressor.cpp:159-168).  weight_word holds the
// weight in its high half, where the packed multiply of interp_diff reads it
// without a shift.
struct WeightFn {
  uint32_t m, b;
};
FH_INDEX_FN WeightFn weight_fn(int nb) {
  if (nb == 4) return {64u * 21846u, 21846u};
  if (nb == 8) return {64u * 9363u, 3u * 9363u};
  return {64u * 4370u, 7u * 4370u};
}
FH_INDEX_FN uint32_t weight_word(WeightFn fn, uint32_t j) {
#if defined(__HIP_DEVICE_COMPILE__)
  // both factors are below 2^24: the full-rate 24-bit multiply-add, which
  // the compiler only finds where it can see the factors' ranges
  uint32_t w;
  asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(w) : "v"(j), "v"(fn.m), "v"(fn.b));
  return w;
#else
  return fn.m * j + fn.b;
#endif
}
FH_INDEX_FN uint32_t weight_of(WeightFn fn, uint32_t j) { return weight_word(fn, j) >> 16; }

// 1 / (64 l), correctly rounded, for a squared endpoint distance 0 < l <=
// 4 * 255^2: one Newton step from a reciprocal within 2 ulp.
FH_INDEX_FN float scaled_rcp(int l) {
  const float lf = (float)l, r = approx_rcp(lf);
  return __builtin_fmaf(__builtin_fmaf(-lf, r, 1.0f), r, r) * 0x1p-6f;
}

// QuantizedError's neighbouring indices (RGBAEndpoints.cpp:240-300) of a
// pixel: j1 = floor(t), j2 = ceil(t), both clamped to the index range, of the
// reference's t = fl(fl(d / l) * kf) (float, d the integer projection, l the
// integer squared distance, kf = nb - 1).  Those equal the floor and ceiling
// of the rational d kf / l: its distance to an integer, when nonzero, is at
// least 1 / l >= 1 / (4 * 255^2) = 3.8e-6, more than the float error of at
// most 2^-23 |t| <= 1.9e-6 for |t| <= 16 (larger |t| is clamped away), and
// fl(fl(k / kf) kf) = k for every integer 0 <= k <= kf in {3, 7, 15}.
//
// Here u = fl(64 d * rl) clamped to [0, 1] (64 d is below 2^24, so its
// conversion is exact; a d below 0 or above l clamps to the end index), and
// the floor and ceiling are truncations of fma(u, kf, 1.9e-6) and
// fma(u, kf, 1 - 1.9e-6).  Exact for every l up to 4 * 255^2, d and kf: the
// host test walks them all at the steps of both functions of d, which are
// monotone.
constexpr float kIndexSlack = 1.9e-6f;

FH_INDEX_FN void index_bounds(int d64, float rl, float kf, uint32_t &j1, uint32_t &j2) {
  const float u = clamp01((float)d64 * rl);
  j1 = (uint32_t)__builtin_fmaf(u, kf, kIndexSlack);
  j2 = (uint32_t)__builtin_fmaf(u, kf, 1.0f - kIndexSlack);
}

}  // namespace bc7
}  // namespace fh
