"""Which way a window's colour-ordered relax runs (colour_fused in
csrc/swe_step.h): inside the step kernel, or as one launch per colour class.
The rule is compiled and asked about measured maps: it must take the side that
was clearly faster on each (times of a 66-window cycle, fused / classes), and
not the slower."""
import subprocess

from simplewinderosion_amd import build as B

# nx, ny, periodic, layers, particles a cell, ms fused, ms classes (16 x 32 tiles)
MEASURED = [
    (512, 512, 1, 2, 1.0, 6.10, 12.06), (512, 512, 1, 1, 0.02, 1.78, 10.23), (513, 513, 1, 2, 0.25, 3.63, 6.29),
    (725, 725, 1, 2, 0.25, 10.18, 12.91), (900, 900, 1, 2, 0.25, 9.39, 8.64), (900, 900, 1, 2, 0.08, 0.79, 1.0),
    (1024, 1024, 1, 1, 0.25, 7.25, 9.71), (1024, 1024, 1, 2, 0.25, 10.83, 12.26), (1024, 1024, 1, 2, 1.0, 11.67, 13.51),
    (1024, 1024, 0, 1, 1.0, 6.65, 8.32), (1026, 1026, 1, 2, 0.25, 11.44, 9.33), (1026, 1026, 1, 1, 0.25, 7.90, 7.34),
    (1026, 1026, 1, 2, 0.02, 5.88, 8.79), (1280, 1280, 1, 1, 0.25, 13.03, 14.56), (1280, 1280, 1, 2, 0.25, 21.31, 18.11),
    (1281, 1281, 1, 2, 0.25, 15.30, 12.28), (1281, 1281, 1, 1, 0.15, 0.90, 1.0), (1448, 1448, 1, 2, 0.25, 25.70, 19.23),
    (1449, 1449, 1, 1, 0.25, 11.80, 9.22), (1449, 1449, 1, 2, 0.04, 0.87, 1.0), (2048, 2048, 1, 2, 0.25, 45.16, 27.32),
    (2048, 2048, 1, 2, 1.0, 51.66, 34.54), (2048, 2048, 1, 1, 0.25, 26.18, 19.68), (2048, 2048, 0, 2, 0.25, 31.68, 21.72),
    (2049, 2049, 1, 1, 0.25, 21.13, 15.29), (2050, 2050, 1, 2, 0.25, 32.89, 24.93), (2050, 2050, 1, 1, 0.02, 10.80, 13.28),
]


def test_the_faster_way_is_taken(tmp_path):
    src = tmp_path / "rule.cpp"
    src.write_text('''#include <cstdio>
#include <cstdlib>
#include "%s/swe_step.h"
using namespace swe;
int main(int, char** v) {
  const int nx = atoi(v[1]), ny = atoi(v[2]), periodic = atoi(v[3]), layers = atoi(v[4]);
  const StepShape sh = kStepShape[0];
  const long tiles = (long)((nx + sh.sx - 1) / sh.sx) * ((ny + sh.sy - 1) / sh.sy);
  const int classes = (3 + (periodic ? nx %% 3 : 0)) * (3 + (periodic ? ny %% 3 : 0));
  printf("%%d\\n", colour_fused(tiles, colour_resident(sh, colour_halo(nx, ny, periodic), true, layers), classes, layers,
                               atof(v[5])));
}
''' % B.CSRC)
    exe = str(tmp_path / "rule")
    subprocess.run([B.hipcc(), "-std=c++17", "--offload-arch=gfx950", "-x", "hip", str(src), "-o", exe], check=True,
                   capture_output=True)
    for *case, fused, classes in MEASURED:
        got = subprocess.run([exe] + [str(v) for v in case], check=True, capture_output=True, text=True).stdout
        assert bool(int(got)) == (fused < classes), case
