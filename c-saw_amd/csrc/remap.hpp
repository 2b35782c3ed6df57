// The pick of the region-remap mode (heur_normalize, functions.cuh:743-868) as
// a search of the CDF itself.
//
// A draw r picks the first i whose normalised CDF value
// p_i = fl32(fl64(C_i) / fl64(T)) exceeds r.  p is a nondecreasing function of
// C_i alone, so that i is the first one with C_i >= c*, the smallest key whose
// quotient exceeds r.  fl32(q) > r exactly when q lies above the midpoint m of
// r and the next float (or on it, where the tie rounds up), so c* is m * T to
// within a unit or two of rounding; the predicate itself settles it.  The
// search then runs on plain keys (the 16-ary index or a binary search) with
// two divisions in all, where a search over p_i divides at every probe.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

namespace csaw {

__host__ __device__ __forceinline__ float f32_of_bits(uint32_t b) {
  float f;
  memcpy(&f, &b, 4);
  return f;
}
__host__ __device__ __forceinline__ uint32_t bits_of_f32(float f) {
  uint32_t b;
  memcpy(&b, &f, 4);
  return b;
}

constexpr int kRemapSteps = 4;  // corrections of the estimate before giving up on it

// smallest c in [1, T] with fl32(fl64(c) / fl64(T)) > r, for 0 <= r < 1 and T >= 1
__host__ __device__ __forceinline__ bool remap_key(float r, uint32_t T, uint32_t* key) {
  const double m = 0.5 * ((double)r + (double)f32_of_bits(bits_of_f32(r) + 1u));
  const double t = (double)T;
  uint32_t c = (uint32_t)(m * t) + 1u;
  if (c > T) c = T;
  auto above = [&](uint32_t x) { return (float)((double)x / t) > r; };
  bool hi = above(c), lo = above(c - 1u);
  for (int k = 0; k < kRemapSteps && !(hi && !lo); ++k) {
    if (lo) {
      hi = true;
      lo = above(--c - 1u);
    } else {
      lo = false;
      hi = above(++c);
    }
  }
  *key = c;
  return hi && !lo;
}

// The same over FP32 keys: smallest c in (0, T], T a normal number well inside
// the range.  *below: the float before it, so the pick is the first C_i > *below.
__host__ __device__ __forceinline__ bool remap_key(float r, float T, float* below) {
  if (!(T >= 1e-30f && T <= 1e38f)) return false;
  const double m = 0.5 * ((double)r + (double)f32_of_bits(bits_of_f32(r) + 1u));
  const double t = (double)T;
  float e = (float)(m * t);
  if (e > T) e = T;
  uint32_t c = bits_of_f32(e);
  if (c == 0u) c = 1u;
  auto above = [&](uint32_t x) { return (float)((double)f32_of_bits(x) / t) > r; };
  bool hi = above(c), lo = above(c - 1u);
  for (int k = 0; k < kRemapSteps && !(hi && !lo); ++k) {
    if (lo) {
      hi = true;
      lo = above(--c - 1u);
    } else {
      lo = false;
      hi = above(++c);
    }
  }
  *below = f32_of_bits(c - 1u);
  return hi && !lo;
}

}  // namespace csaw
