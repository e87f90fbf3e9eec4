// swe_device.hpp -- scalar device primitives of the erosion hot path.
//
// Every function here is a sequence of IEEE-754 float32 operations (plus one
// float64 multiply/subtract in the drag factor, wind.hpp:87) written in the
// operation order of the reference and of glm 0.9.9, so that with
// -ffp-contract=off and correctly-rounded division/sqrt the device produces
// the same bits as any other IEEE implementation of the same steps.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/swe.h"

namespace swe {

// ---------------------------------------------------------------------------
// Bits and fixed point (int64, resolution 2^-32)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float u2f(uint32_t u) { return __uint_as_float(u); }
__device__ __forceinline__ uint32_t f2u(float f) { return __float_as_uint(f); }

// round_half_even(v * 2^32) as int64; NaN -> 0, |v| >= 2^31 saturates.
// Below 2^18 the product is formed exactly in float64 (a power-of-two scale
// of v) and 1.5 * 2^52 added: that sum's last bit is worth 1, so the addition
// rounds to an integer, ties to even, and the integer is the sum's encoding
// minus the constant's -- four instructions in place of the fourteen of a
// float -> int64 conversion.
__device__ __forceinline__ int64_t fx_from_small_f32(float v) {  // |v| < 2^18
  const double d = (double)(v * 4294967296.0f) + 6755399441055744.0;
  return (int64_t)((uint64_t)__double_as_longlong(d) - 0x4338000000000000ull);
}
__device__ __forceinline__ int64_t fx_from_f32(float v) {
  if (__builtin_expect(__builtin_fabsf(v) < 262144.0f, 1)) return fx_from_small_f32(v);
  if (!(__builtin_fabsf(v) < 2147483648.0f)) return v != v ? 0 : (v < 0.0f ? INT64_MIN : INT64_MAX);
  return (int64_t)(v * 4294967296.0f);  // a float of 2^18 or more is a multiple of 2^-5
}

// round_half_even(m * 2^-32) to float32: the int64 -> float32 conversion
// rounds to nearest even, and the power-of-two scale is exact (|m| >= 1
// keeps the result far from the denormal range).
__device__ __forceinline__ float f32_from_fx(int64_t m) { return (float)m * 2.3283064365386963e-10f; }

// The same for |m| < 2^47: the part above the lowest 24 bits and those 24
// bits each convert exactly, and one fused multiply-add rounds their scaled
// sum (six instructions, none 64-bit, for eleven).
__device__ __forceinline__ float f32_from_small_fx(int64_t m) {
  const float hi = (float)(int32_t)__builtin_amdgcn_alignbit((uint32_t)(m >> 32), (uint32_t)m, 24);
  const float lo = (float)((uint32_t)m & 0xffffffu);
  return __builtin_fmaf(hi, 0x1p-8f, lo * 0x1p-32f);
}
__device__ __forceinline__ bool small_fx(int64_t m) {  // -2^39 <= m < 2^39
  return (uint32_t)((int32_t)(m >> 32) + 128) < 256u;
}

// exp for float32: Cody-Waite reduction with a two-part ln2, degree-7
// Taylor polynomial in Horner form, exact power-of-two scaling (two steps,
// the first by 1 except below 2^-125).  The special cases are selected at
// the end, without branches.
__device__ __forceinline__ float exp_f32(float x) {
  const float log2e = 1.44269502162933349609375f;
  const float ln2_hi = 0.693145751953125f;
  const float ln2_lo = 1.428606765330187045e-06f;
  const float kf = __builtin_rintf(x * log2e);
  const float r = (x - kf * ln2_hi) - kf * ln2_lo;
  float p = 1.0f / 5040.0f;
  p = p * r + 1.0f / 720.0f;
  p = p * r + 1.0f / 120.0f;
  p = p * r + 1.0f / 24.0f;
  p = p * r + 1.0f / 6.0f;
  p = p * r + 0.5f;
  p = p * r + 1.0f;
  p = p * r + 1.0f;
  const int k = (int)kf;
  const int k1 = k < -125 ? -64 : 0;
  p = p * u2f((uint32_t)(127 + k1) << 23);
  p = p * u2f((uint32_t)(k - k1 + 127) << 23);
  p = x < -104.0f ? 0.0f : p;
  p = x > 88.72283935546875f ? u2f(0x7f800000u) : p;
  return x != x ? x : p;
}

// s = sqrt(d) and r = 1 / s, both correctly rounded.  In the normal range one
// v_rsq_f32 seeds Goldschmidt's coupled iteration g -> sqrt, h -> 1 / (2 sqrt),
// whose final residual rounds s; one residual step from v_rcp_f32 rounds r
// (from 2h in its place 450 of the range's quotients come out one ulp low, at
// s with all mantissa bits set).  Equal to the IEEE square root and quotient
// for every float (tests/test_gpu_primitives.py): 13 instructions in place of
// 26.  Zero, tiny, huge, negative and NaN take the IEEE operations.
struct Root {
  float s, r;
};
__device__ __forceinline__ Root root_of(float d) {
  if (__builtin_expect(d >= 0x1p-90f && d <= 0x1p90f, 1)) {
    const float y = __builtin_amdgcn_rsqf(d);
    float g = d * y, h = 0.5f * y;
    const float e = __builtin_fmaf(-h, g, 0.5f);
    g = __builtin_fmaf(g, e, g);
    h = __builtin_fmaf(h, e, h);
    const float s = __builtin_fmaf(__builtin_fmaf(-g, g, d), h, g);
    const float z = __builtin_amdgcn_rcpf(s);
    return Root{s, __builtin_fmaf(__builtin_fmaf(-s, z, 1.0f), z, z)};
  }
  const float s = __builtin_sqrtf(d);
  return Root{s, 1.0f / s};
}

// ---------------------------------------------------------------------------
// Counter RNG (SplitMix64 output function over (seed, cycle, particle, call))
// ---------------------------------------------------------------------------
constexpr uint64_t kGolden = 0x9E3779B97F4A7C15ull;
constexpr uint64_t kPart = 0xD1B54A32D192ED03ull;

__host__ __device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
__host__ __device__ __forceinline__ uint64_t cycle_key(uint64_t seed, uint64_t cycle) {
  return mix64(seed + kGolden * (cycle + 1));
}
__host__ __device__ __forceinline__ uint64_t particle_key(uint64_t ck, uint64_t particle) {
  return mix64(ck ^ (kPart * (particle + 1)));
}

// ---------------------------------------------------------------------------
// glm vec3 arithmetic (operation order of glm 0.9.9)
// ---------------------------------------------------------------------------
struct f3 {
  float x, y, z;
};
__device__ __forceinline__ f3 mk(float x, float y, float z) { return f3{x, y, z}; }
__device__ __forceinline__ f3 add(f3 a, f3 b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ f3 sub(f3 a, f3 b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ f3 mul(f3 a, f3 b) { return mk(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ f3 smul(float s, f3 a) { return mk(s * a.x, s * a.y, s * a.z); }
__device__ __forceinline__ f3 muls(f3 a, float s) { return mk(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ f3 divs(f3 a, float s) { return mk(a.x / s, a.y / s, a.z / s); }
__device__ __forceinline__ f3 subs(f3 a, float s) { return mk(a.x - s, a.y - s, a.z - s); }
__device__ __forceinline__ float dot(f3 a, f3 b) { return (a.x * b.x + a.y * b.y) + a.z * b.z; }
__device__ __forceinline__ f3 cross(f3 a, f3 b) {
  return mk(a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y);
}
__device__ __forceinline__ f3 normalize(f3 a) { return muls(a, root_of(dot(a, a)).r); }
__device__ __forceinline__ f3 mix(f3 x, f3 y, float a) { return add(muls(x, 1.0f - a), muls(y, a)); }

// quad::_normal (cellpool.h:200-223) from the five stencil heights.  gNE,
// gSW, gSE, gNW gate the four planes (diagonal in bounds).
__device__ __forceinline__ f3 surface_normal(float hp, float hyp, float hxp, float hym, float hxm,
                                             bool g1, bool g2, bool g3, bool g4, float mapscale) {
  const f3 s = mk(1.0f, mapscale, 1.0f);
  f3 n = mk(0.0f, 0.0f, 0.0f);
  if (g1) n = add(n, cross(mul(s, mk(0.0f, hyp - hp, 1.0f)), mul(s, mk(1.0f, hxp - hp, 0.0f))));
  if (g2) n = add(n, cross(mul(s, mk(0.0f, hym - hp, -1.0f)), mul(s, mk(-1.0f, hxm - hp, 0.0f))));
  if (g3) n = add(n, cross(mul(s, mk(1.0f, hxp - hp, 0.0f)), mul(s, mk(0.0f, hym - hp, -1.0f))));
  if (g4) n = add(n, cross(mul(s, mk(-1.0f, hxm - hp, 0.0f)), mul(s, mk(0.0f, hyp - hp, 1.0f))));
  const Root l = root_of(dot(n, n));
  if (l.s > 0.0f) n = muls(n, l.r);
  return n;
}

// Euclidean remainder of v by n (n > 0) for |v| <= 2^30: two rounds of a
// float quotient estimate (the first leaves at most a few hundred multiples
// of n, the second less than one) and a correction by one step.
__device__ __forceinline__ int32_t wrap(int32_t v, int32_t n, float rcp_n) {
  if ((uint32_t)v < (uint32_t)n) return v;
  int32_t r = v - (int32_t)__builtin_floorf((float)v * rcp_n) * n;
  r -= (int32_t)__builtin_floorf((float)r * rcp_n) * n;
  if (r < 0) r += n;
  if (r >= n) r -= n;
  return r;
}

// The same for -n <= v < 2n: as unsigned numbers the wanted one of v, v + n
// (v - n) is the smaller.
__device__ __forceinline__ int32_t wrap_near(int32_t v, int32_t n) {
  const uint32_t a = (uint32_t)v, b = a + (uint32_t)n, c = a < b ? a : b, d = c - (uint32_t)n;
  return (int32_t)(c < d ? c : d);
}

}  // namespace swe
