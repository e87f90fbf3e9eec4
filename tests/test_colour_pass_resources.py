"""Register budget of the colour classes' launches (k_colour_pass and its
batch form), read from the gfx950 metadata hipcc emits.  A launch reads every
cell of its class and most have nothing to do, so its time is the waves in
flight: four a SIMD (128 registers) with one layer or a bounded map, three
(168) with two layers on a periodic one, and no scratch."""
import os
import subprocess

import pytest

from simplewinderosion_amd import build as B
from test_kernel_resources import _kernels


def test_colour_pass_registers(tmp_path):
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    out = str(tmp_path / "kernels.s")
    subprocess.run([cc] + B.HIP_FLAGS + ["--cuda-device-only", "-S", "-o", out, os.path.join(B.CSRC, "swe_kernels.hip")],
                   check=True, capture_output=True)
    passes = {k: v for k, v in _kernels(open(out).read()).items() if "k_colour_pass" in k}
    assert len(passes) == 8  # periodic x layers, single and batch
    for name, f in passes.items():
        budget = 168 if "ILb1ELi2E" in name else 128
        assert f["vgpr_count"] <= budget, (name, f["vgpr_count"])
        assert f["private_segment_fixed_size"] == 0, name
