// swe_cascade.hpp -- one cell's cascade of a snapshot window on the device.
#pragma once

#include "swe_device.hpp"

namespace swe {

// Settling factor of a cell's `events` cascade events in one window:
// settling for one event, else 1 - (1 - settling)^events by binary
// exponentiation (least significant bit first) in float.
__device__ __forceinline__ float settle_factor_dev(float settling, uint32_t events) {
  if (events <= 1u) return settling;
  float b = 1.0f - settling, r = 1.0f;
  uint32_t e = events;
  while (e) {
    if (e & 1u) r = r * b;
    b = b * b;
    e >>= 1;
  }
  return 1.0f - r;
}

// Neighbour offsets of World::cascade (world.hpp:83-92), k = 0..7:
// (-1,-1) (-1,0) (-1,1) (0,-1) (0,1) (1,-1) (1,0) (1,1), packed two bits per
// k as offset + 1; bit k of kDiagMask marks the diagonals (distance sqrt 2).
constexpr uint32_t kOffXPacked = 0xa940u, kOffYPacked = 0x9224u, kDiagMask = 0xa5u;
__device__ __forceinline__ int32_t off_x(int32_t k) { return (int32_t)((kOffXPacked >> (2 * k)) & 3u) - 1; }
__device__ __forceinline__ int32_t off_y(int32_t k) { return (int32_t)((kOffYPacked >> (2 * k)) & 3u) - 1; }

// Sort key of a neighbour: descending order of the key is descending height,
// ties in ascending offset order -- the order the stable insertion sort of
// world.hpp:118-120 leaves eight elements in.  The key is the height as a
// float64 (exact; -0 first folded into +0, which the float comparison treats
// as equal) with the offset in the three lowest of its 29 spare bits, so
// that a compare-exchange is one v_max_f64 and one v_min_f64.  Those bits
// grow the magnitude, so a negative height holds k and a positive 7 - k;
// rounding the key to float32 gives the height back.  Map heights are
// finite; out-of-map neighbours get -infinity.
__device__ __forceinline__ double cascade_key(float h, int32_t k, bool valid) {
  const float z = h + 0.0f;
  const uint64_t u = (uint64_t)__double_as_longlong((double)z) | (uint32_t)(z < 0.0f ? k : 7 - k);
  return valid ? __longlong_as_double((long long)u) : -__builtin_inf();
}
__device__ __forceinline__ int32_t cascade_key_offset(double key) {
  const int32_t lo = (int32_t)(__double_as_longlong(key) & 7);
  return key < 0.0 ? lo : 7 - lo;
}

// One cell's cascade of the window: World::cascade (world.hpp:79-153)
// against the snapshot with the window's settling factor.  hn[k]: neighbour
// k's height in the fixed offset order; sed_of(k): its sediment (two-layer
// maps only); hc / sc: the centre's; bit k of validmask set for in-map
// neighbours.  The neighbours are sorted by a sorting network on their keys
// and walked in that order with the centre evolving; emit(k, amount) is
// called with the fixed-point amount neighbour k receives (the centre loses
// the same amount; zero for no transfer).  A wave's time is the dependent
// chain: 230 cycles for the sort on float64 keys (760 with 64-bit integer
// ones) and some 70 a walk step.
template <int LAYERS, class SedOf, class Emit>
__device__ __forceinline__ void cascade_cell_dev(const float hn[8], const SedOf& sed_of, float hc, float sc,
                                                 uint32_t validmask, float settling, float maxdiff, Emit&& emit) {
  double key[8];
#pragma unroll
  for (int k = 0; k < 8; k++) key[k] = cascade_key(hn[k], k, (validmask >> k) & 1u);
#define SWE_CAS(i, j)                      \
  {                                        \
    const double a = key[i], b = key[j];   \
    key[i] = __builtin_fmax(a, b);         \
    key[j] = __builtin_fmin(a, b);         \
  }
  SWE_CAS(0, 2) SWE_CAS(1, 3) SWE_CAS(4, 6) SWE_CAS(5, 7)
  SWE_CAS(0, 4) SWE_CAS(1, 5) SWE_CAS(2, 6) SWE_CAS(3, 7)
  SWE_CAS(0, 1) SWE_CAS(2, 3) SWE_CAS(4, 5) SWE_CAS(6, 7)
  SWE_CAS(2, 4) SWE_CAS(3, 5)
  SWE_CAS(1, 4) SWE_CAS(3, 6)
  SWE_CAS(1, 2) SWE_CAS(3, 4) SWE_CAS(5, 6)
#undef SWE_CAS
  // the walk's inputs in its order, read before it so that the reads overlap
  // (each would otherwise wait its turn in the chain); an out-of-map
  // neighbour's NaN compares false and takes nothing
  const float dd = __builtin_sqrtf(2.0f);
  int32_t kk[8];
  float hh[8], sn[8], thr[8], ts[8];
#pragma unroll
  for (int r = 0; r < 8; r++) {
    kk[r] = cascade_key_offset(key[r]);
    const bool in = key[r] != -__builtin_inf();
    hh[r] = in ? (float)key[r] : __builtin_nanf("");
    sn[r] = LAYERS == 2 && in ? sed_of(kk[r]) : 0.0f;
    const float d = ((kDiagMask >> kk[r]) & 1u) ? dd : 1.0f;
    thr[r] = (d * maxdiff) * 1.0f;
  }
  // the serial chain, without branches: a neighbour that takes nothing (no
  // difference, or none beyond the threshold) moves zero.  Transfers are
  // signed: positive from the centre to the neighbour.
  bool big = false;
#pragma unroll
  for (int r = 0; r < 8; r++) {
    const float diff = hc - hh[r], ad = __builtin_fabsf(diff);
    const float excess = ad - thr[r];
    float t = settling * excess / 2.0f;
    if (LAYERS == 2) {
      const float avail = diff > 0.0f ? sc : sn[r];
      if (t > avail) t = avail;
      t = t > 0.0f ? t : 0.0f;
    }
    t = __builtin_fminf(excess, ad) > 0.0f ? t : 0.0f;
    ts[r] = __builtin_copysignf(t, diff);
    if (t < 0.0f) ts[r] = -ts[r];  // a negative settling factor moves material uphill
    hc -= ts[r];
    if (LAYERS == 2) sc -= ts[r];
    big = big || !(__builtin_fabsf(t) < 262144.0f);
  }
  int64_t amt[8];
#pragma unroll
  for (int r = 0; r < 8; r++) amt[r] = fx_from_small_f32(ts[r]);
  // an amount that may saturate is rounded before its direction is applied:
  // what the loser gives is what the taker gets, also at -2^63.  (The sign of
  // ts is the direction, reversed by a negative settling factor.)
  if (__builtin_expect(big, 0)) {
#pragma unroll
    for (int r = 0; r < 8; r++) {
      const uint64_t m = (uint64_t)fx_from_f32(__builtin_copysignf(ts[r], settling));
      amt[r] = (int64_t)((ts[r] < 0.0f) != (settling < 0.0f) ? 0 - m : m);
    }
  }
#pragma unroll
  for (int r = 0; r < 8; r++) emit(kk[r], amt[r]);
}

}  // namespace swe
