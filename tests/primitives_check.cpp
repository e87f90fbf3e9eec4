// CPU check of the device primitives that are plain float and integer
// arithmetic (csrc/swe_device.hpp, swe_fly.hpp, swe_cascade.hpp compiled for the
// host) against the oracle and exact integer forms.  Prints one line a check:
// its name and the number of mismatches.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <hip/hip_runtime.h>  // the host stand-in written by the test

#include "SWE_CSRC/swe_cascade.hpp"
#include "SWE_CSRC/swe_fly.hpp"

extern "C" {
int64_t or_fx(float v);
float or_unfx(int64_t m);
float or_expf(float x);
}

using namespace swe;

static bool same(float a, float b) { return f2u(a) == f2u(b) || (a != a && b != b); }
static void report(const char* name, long bad) { printf("%s %ld\n", name, bad); }

int main() {
  long bad = 0;
#pragma omp parallel for reduction(+ : bad)
  for (int64_t i = 0; i < ((int64_t)1 << 32); i++) bad += !same(exp_f32(u2f((uint32_t)i)), or_expf(u2f((uint32_t)i)));
  report("exp_f32", bad);
  bad = 0;
#pragma omp parallel for reduction(+ : bad)
  for (int64_t i = 0; i < ((int64_t)1 << 32); i++) {
    const float v = u2f((uint32_t)i);
    const int64_t want = or_fx(v);
    bad += fx_from_f32(v) != want;
    if (__builtin_fabsf(v) < 262144.0f) bad += fx_from_small_f32(v) != want;
  }
  report("fx_from_f32", bad);
  // every 24-bit window of a master, with sticky bits below it and both signs
  bad = 0;
#pragma omp parallel for reduction(+ : bad)
  for (int64_t i = 0; i < ((int64_t)1 << 25); i++)
    for (int sh = 0; sh <= 22; sh++)
      for (int64_t low : {(int64_t)0, (int64_t)1, ((int64_t)1 << sh) - 1, (int64_t)1 << (sh ? sh - 1 : 0)}) {
        const int64_t m = (i << sh) + (low & (((int64_t)1 << sh) - 1));
        for (int64_t v : {m, -m}) {
          bad += !same(f32_from_fx(v), or_unfx(v));
          if (v < ((int64_t)1 << 47) && v >= -((int64_t)1 << 47)) bad += !same(f32_from_small_fx(v), or_unfx(v));
        }
      }
  report("f32_from_fx", bad);
  bad = 0;
  for (int64_t v : {-((int64_t)1 << 39) - 1, -((int64_t)1 << 39), ((int64_t)1 << 39) - 1, (int64_t)1 << 39})
    bad += small_fx(v) != (v >= -((int64_t)1 << 39) && v < ((int64_t)1 << 39));
  report("small_fx", bad);
  bad = 0;
  for (uint32_t v = 0; v < (1u << 21); v++) bad += mod1001(v) != (float)(v % 1001u);
  report("mod1001", bad);
  // wrap: small and large axes, every residue near the ends of the range
  bad = 0;
  std::vector<int32_t> axes;
  for (int32_t n = 1; n <= 300; n++) axes.push_back(n);
  for (int32_t n : {511, 512, 1000, 1001, 4096, 5003, 16384, 46340, 65537, 1 << 20, 3 << 20, 1 << 24, (1 << 24) + 1, 1 << 28})
    axes.push_back(n);
#pragma omp parallel for reduction(+ : bad) schedule(dynamic)
  for (size_t a = 0; a < axes.size(); a++) {
    const int32_t n = axes[a];
    const float rcp = 1.0f / (float)n;
    auto check = [&](int64_t v) {
      if (v < -((int64_t)1 << 30) || v > ((int64_t)1 << 30)) return;
      const int64_t want = ((v % n) + n) % n;
      bad += wrap((int32_t)v, n, rcp) != want;
      if (v >= -n && v < 2 * (int64_t)n) bad += wrap_near((int32_t)v, n) != want;
    };
    for (int64_t c : {(int64_t)0, (int64_t)n, -(int64_t)n, (int64_t)1 << 23, -((int64_t)1 << 23), (int64_t)1 << 24,
                      (int64_t)1 << 30, -((int64_t)1 << 30), (int64_t)1 << 29, (((int64_t)1 << 30) / n) * n})
      for (int64_t d = -3000; d <= 3000; d++) check(c + d);
    for (int64_t v = -((int64_t)1 << 30); v <= ((int64_t)1 << 30); v += 4093) check(v);
  }
  report("wrap", bad);
  // cascade keys: descending key is descending height, ties in ascending
  // offset; height and offset come back
  bad = 0;
  std::vector<float> hs = {0.0f, -0.0f, 1e-45f, -1e-45f, 2.3283064e-10f, 1.0f, -1.0f, 3.4e38f, -3.4e38f, 2.1e9f, -2.1e9f};
  srand(3);
  for (int i = 0; i < 3000; i++) hs.push_back(u2f(((uint32_t)rand() << 16 ^ (uint32_t)rand()) & 0xfeffffffu));
  for (int i = 0; i < 300; i++) hs.push_back(hs[(size_t)i + 11] * (1.0f + 0x1p-23f));
  for (size_t i = 0; i < hs.size(); i++)
    for (size_t j = 0; j < hs.size(); j++)
      for (int k = 0; k < 8; k += 7) {
        const int q = (int)(j % 8);
        const double a = cascade_key(hs[i], k, true), b = cascade_key(hs[j], q, true);
        const bool before = hs[i] > hs[j] || (hs[i] == hs[j] && k < q);
        bad += (a > b) != before;
        bad += !((float)a == hs[i]) || cascade_key_offset(a) != k;
        bad += !(cascade_key(hs[i], k, false) < a);
      }
  report("cascade_key", bad);
  return 0;
}
