"""The device primitives that replaced longer forms (csrc/swe_device.hpp,
swe_fly.hpp, swe_cascade.hpp) on the CPU, over every input or every window of
one: exp_f32 and the fixed-point conversions against the oracle, the turbulence
draws' remainder, the periodic wraps, and the cascade's sort keys.  (The square
root needs the GPU's seeds: test_gpu_primitives.py.)"""
import os
import shutil
import subprocess

import pytest

from simplewinderosion_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))

# what the headers use of the HIP runtime and the GPU's builtins
STAND_IN = """#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __host__
#define __forceinline__ inline
static inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static inline uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static inline long long __double_as_longlong(double d) { long long u; memcpy(&u, &d, 8); return u; }
static inline double __longlong_as_double(long long u) { double d; memcpy(&d, &u, 8); return d; }
static inline uint32_t __builtin_amdgcn_alignbit(uint32_t hi, uint32_t lo, uint32_t n) {
  return (uint32_t)((((uint64_t)hi << 32) | lo) >> n);
}
static inline float __builtin_amdgcn_rsqf(float x) { return 1.0f / std::sqrt(x); }
static inline float __builtin_amdgcn_rcpf(float x) { return 1.0f / x; }
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is needed to build the check")
def test_primitives_match_their_references(tmp_path):
    os.makedirs(str(tmp_path / "hip"))
    (tmp_path / "hip" / "hip_runtime.h").write_text(STAND_IN)
    text = open(os.path.join(HERE, "primitives_check.cpp")).read().replace("SWE_CSRC", B.CSRC)
    (tmp_path / "check.cpp").write_text(text)
    oracle = str(tmp_path / "oracle.o")
    flags = ["-O2", "-fopenmp", "-ffp-contract=off"]
    subprocess.run(["gcc", "-std=gnu11"] + flags + ["-c", "-o", oracle, os.path.join(HERE, "..", "oracle", "swe_oracle.c")],
                   check=True)
    if "fma" in open("/proc/cpuinfo").read():
        flags.append("-mfma")
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++17", "-w"] + flags + ["-I", str(tmp_path), "-o", exe, str(tmp_path / "check.cpp"),
                                                          oracle, "-lm"], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=900)
    assert res.returncode == 0, res.stderr
    got = dict(line.split() for line in res.stdout.splitlines())
    assert got == {k: "0" for k in ("exp_f32", "fx_from_f32", "f32_from_fx", "small_fx", "mod1001", "wrap",
                                    "cascade_key")}
