"""Resource budget of the step kernel, read from the gfx950 code-object
metadata that hipcc emits, for every compiled tile shape: no private
(scratch) memory, the VGPRs of the shape's waves per SIMD (96 for five, 128
for four) and LDS for the workgroups those waves make per CU.  A kernel that
breaks one of these still computes the right bits but several times slower,
so the budget is checked at build time, without a GPU."""
import os
import re
import subprocess

import pytest

from simplewinderosion_amd import build as B

LDS_PER_CU = 160 * 1024


def _kernels(text):
    kernels = {}
    for block in text.split("  - .agpr_count:")[1:]:
        m = re.search(r"\.name:\s+(\S+)", block)
        if not m:
            continue
        fields = dict(re.findall(r"\.(\w+):\s+(\d+)\s*$", block, re.M))
        kernels[m.group(1)] = {k: int(v) for k, v in fields.items()}
    return kernels


# the shape table of csrc/swe_step.h: (cells x, cells y, threads, waves per SIMD)
SHAPES = [(16, 32, 256, 5), (32, 16, 256, 5), (16, 16, 128, 5), (16, 32, 256, 4), (32, 32, 512, 4)]


def test_shape_table_matches_the_source():
    text = open(os.path.join(B.CSRC, "swe_step.h")).read()
    table = text[text.index("kStepShape[kStepShapes] = {"):]
    got = [tuple(int(v) for v in m) for m in re.findall(r"\{(\d+), (\d+), (\d+), (\d+)\}", table)][:len(SHAPES)]
    assert got == SHAPES and B.N_SHAPES == len(SHAPES)


@pytest.fixture(scope="module")
def metadata(tmp_path_factory):
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("isa")
    from concurrent.futures import ThreadPoolExecutor

    def one(i):
        out = str(d / ("shape%d.s" % i))
        cmd = [cc] + B.HIP_FLAGS + ["-DSWE_STEP_SHAPE=%d" % i, "--cuda-device-only", "-S", "-o", out,
                                    os.path.join(B.CSRC, B.SHAPE_SOURCE)]
        subprocess.run(cmd, check=True, capture_output=True)
        return _kernels(open(out).read())

    with ThreadPoolExecutor(max_workers=len(SHAPES)) as ex:
        return list(ex.map(one, range(len(SHAPES))))


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_step_kernel_budget(metadata, shape):
    """Every instance of a shape: no scratch, the VGPRs of its waves per SIMD,
    LDS for the workgroups those waves make per CU."""
    sx, sy, threads, waves = SHAPES[shape]
    steps = {k: v for k, v in metadata[shape].items() if "k_step" in k}
    assert len(steps) == 48  # periodic x track x layers x deposit x mode (step + relax, relax only, step only)
    vgpr_max = (512 // waves) // 8 * 8
    groups_per_cu = 4 * waves // (threads // 64)
    for name, f in steps.items():
        assert f["private_segment_fixed_size"] == 0, name
        assert f["vgpr_count"] <= vgpr_max, (name, f["vgpr_count"])
        assert f.get("vgpr_spill_count", 0) == 0, name
        assert groups_per_cu * f["group_segment_fixed_size"] <= LDS_PER_CU, (name, f["group_segment_fixed_size"])


@pytest.mark.parametrize("shape", range(len(SHAPES)))
def test_colour_kernel_budget(metadata, shape):
    """Every instance of k_colour_step: no scratch, the VGPRs of four waves per
    SIMD."""
    colour = {k: v for k, v in metadata[shape].items() if "k_colour_step" in k}
    assert len(colour) == 32  # periodic x track x layers x deposit x mode (step + relax, relax only)
    for name, f in colour.items():
        assert f["private_segment_fixed_size"] == 0, (name, f["private_segment_fixed_size"])
        assert f.get("vgpr_spill_count", 0) == 0, name
        assert f["vgpr_count"] <= 128, (name, f["vgpr_count"])


def test_colour_residency(metadata, tmp_path):
    """The workgroups that colour_resident (csrc/swe_step.h) says the chip
    holds of k_colour_step: what the compiled kernels' static LDS and registers
    leave room for, for every shape, halo and number of layers."""
    src = tmp_path / "resident.cpp"
    src.write_text('''#include <cstdio>
#include "%s/swe_step.h"
using namespace swe;
int main() {
  const ColourHalo hs[] = {kColourHalo, kColourHaloSeam, kColourHaloMax};
  for (int i = 0; i < kStepShapes; i++)
    for (int h = 0; h < 3; h++)
      for (int t = 0; t < 2; t++)
        for (int l = 1; l <= 2; l++)
          printf("%%d %%d %%d %%d %%ld %%ld\\n", i, h, t, l, (long)colour_lds(kStepShape[i], hs[h], t, l),
                 (long)colour_resident(kStepShape[i], hs[h], t, l));
}
''' % B.CSRC)
    exe = str(tmp_path / "resident")
    subprocess.run([B.hipcc(), "-std=c++17", "--offload-arch=gfx950", "-x", "hip", str(src), "-o", exe], check=True,
                   capture_output=True)
    rows = [tuple(int(v) for v in line.split()) for line in
            subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(rows) == 60
    for i, h, t, layers, lds, resident in rows:
        _, _, threads, _ = SHAPES[i]
        mine = [f for k, f in metadata[i].items() if "k_colour_step" in k and "ELi%dE" % layers in k.split("Lb")[2]]
        assert len(mine) == 16
        static = max(f["group_segment_fixed_size"] for f in mine)
        regs = max(f["vgpr_count"] for f in mine)
        by_lds = LDS_PER_CU // (-(-(static + lds) // 1280) * 1280)
        by_waves = 4 * min(512 // (-(-regs // 8) * 8), 8) // (threads // 64)
        assert resident == 256 * min(by_lds, by_waves), (i, h, t, layers)


def test_network_kernel_scratch(tmp_path):
    """The surrogate's kernels use no scratch but one shape of the wide
    convolution: 256 pixels x 64 channels a workgroup keeps two workgroups on a
    CU at 256 registers with some 20 spilled."""
    out = str(tmp_path / "nn.s")
    subprocess.run([B.hipcc()] + B.HIP_FLAGS + ["--cuda-device-only", "-S", "-o", out,
                                                os.path.join(B.CSRC, B.NN_SOURCES[0])], check=True, capture_output=True)
    kernels = _kernels(open(out).read())
    assert sum("k_conv_tile" in k for k in kernels) == 36 and sum("k_conv_wide" in k for k in kernels) == 66
    assert sum("k_wgrad" in k for k in kernels) == 6
    for name, f in kernels.items():
        assert f["vgpr_count"] <= 512 and f["private_segment_fixed_size"] <= (88 if "k_conv_wideILi4ELi4E" in name else 0), (
            name, f["vgpr_count"], f["private_segment_fixed_size"])
