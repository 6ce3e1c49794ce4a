"""What the launchers' rules take, asked without a device (so nothing is ever
launched) by a small program that calls them and prints the answer.

* Counts of the launches after a step: cells are numbered in 32 bits, and what
  would overflow must be refused, and only that (hipErrorInvalidValue where the
  launcher refused, another error where it went on to launch).
* Which steps the FP32 full-row kernel serves (for 256 compute units).
"""
import os
import subprocess

import pytest

import test_gpu_batch
import test_gpu_slab
from rtm3d_demo_amd import build

REFUSED = 1  # hipErrorInvalidValue

PROGRAM = r"""
#include "rtm_internal.hpp"
#include "rtm_slab_launch.hpp"
#include "rtm_tail.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
using namespace rtmhip;
static Grid grid(int nx, int ny, int nz)
{
    Grid g{};
    g.nx = nx;
    g.ny = ny;
    g.nz = nz;
    g.sy = nz;
    g.sx = (long long)ny * nz;
    return g;
}
int main(int argc, char **argv)
{
    int n = 0;
    if (hipGetDeviceCount(&n) == hipSuccess && n > 0) return 2;
    (void)hipGetLastError();
    const auto arg = [&](int i) { return atoi(argv[i]); };
    const Grid g = grid(arg(2), arg(3), arg(4));
    const int b = arg(5), R = arg(6), taps = arg(7);
    float *p = reinterpret_cast<float *>(4096);
    const TailSource src{p, (long long)g.nx / 2 * g.sx + g.ny / 2 * g.sy + g.nz / 2, 0};
    if (!strcmp(argv[1], "full-row")) {  // R: the stencil radius, taps: the taper's form
        const ImageFuse fz{};
        const TaperFuse tf{p, b, 1, taps, 0};
        printf("%d\n",
               slab_plan(R, g, arg(8) ? &fz : nullptr, taps ? &tf : nullptr, arg(9)).nyt);
        return 0;
    }
    hipError_t e;
    if (!strcmp(argv[1], "all")) {
        e = launch_tail_all<float>(p, p, g, b, R, taps, nullptr, &src, nullptr);
    } else {
        const bool layer = arg(8), image = arg(9);
        const TailLayer<float> w{taps, 0, nullptr, p, layer ? p : nullptr};
        e = launch_tail_upper<float>(p, p, g, b, R, w, nullptr, &src, image ? p : nullptr, p,
                                     nullptr);
    }
    printf("%d\n", (int)e);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("limits")
    src, exe = d / "limits.hip", d / "limits"
    src.write_text(PROGRAM)
    subprocess.run([build.HIPCC, *build.HIP_FLAGS, "-I" + build.CSRC, "--cuda-host-only",
                    "-c", str(src), "-o", str(d / "limits.o")], check=True, capture_output=True)
    subprocess.run([build.HIPCC, str(d / "limits.o"), "-o", str(exe), "-L" + build.LIBDIR,
                    "-lrtm3d_hip", "-Wl,-rpath," + build.LIBDIR], check=True, capture_output=True)
    return str(exe)


def _result(program, *args):
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="")
    r = subprocess.run([program, *map(str, args)], env=env, capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r
    return int(r.stdout)


@pytest.mark.parametrize("grid, R, layer, refused", [
    ((23171, 23170, 9), 4, 0, True),   # 2^31 + 4632 cells with z < R
    ((23171, 23170, 9), 4, 1, True),
    ((23000, 23000, 9), 4, 0, False),  # 2.116e9
    ((46340, 46340, 9), 1, 0, True),   # 2^31 - 88048 with z < R, 556068 on the rims
    ((46340, 46300, 9), 1, 0, False),  # 2145542000 and 555828
])
def test_slab_frame_bound(program, grid, R, layer, refused):
    b = 4
    assert (_result(program, "upper", *grid, b, R, 2, layer, 0) == REFUSED) == refused


# parts that fit one by one go on, together past 2^31 items or not
@pytest.mark.parametrize("args, refused", [
    # layer 4e8 rows, frame 4e8 rows + 3.2e5 cells, imaged frame 1.6e9 cells
    (("upper", 20000, 20000, 5000, 5, 4, 2, 1, 1), False),
    # the imaged frame alone: 2.2e9
    (("upper", 20000, 20000, 7000, 5, 4, 0, 0, 1), True),
    # frame 2.076e9 cells, front-right edge 1.5e8
    (("all", 240, 16000, 16000, 100, 4, 2), False),
    # the frame alone: 2.176e9
    (("all", 1000, 16000, 16000, 100, 4, 2), True),
])
def test_parts_that_fit_by_themselves(program, args, refused):
    assert (_result(program, *args) == REFUSED) == refused


# taper: 0 none, 1 the upper taper on load, 2 taper3D and 3 the upper taper on
# the output
@pytest.mark.parametrize("grid, b, radius, taper, image, served", [
    ((592, 592, 336), 40, 4, 0, 0, True),
    ((592, 592, 336), 40, 4, 2, 0, True),
    ((592, 592, 336), 40, 4, 3, 0, True),
    ((592, 592, 336), 40, 4, 0, 1, True),
    ((592, 592, 336), 40, 4, 3, 1, True),
    ((592, 592, 336), 40, 4, 1, 0, False),
    ((592, 592, 336), 40, 4, 2, 1, False),   # no imaging with taper3D
    ((592, 592, 336), 40, 3, 0, 0, False),
    ((592, 592, 128), 40, 4, 0, 0, False),   # rows of 129 to 512 cells
    ((592, 592, 129), 40, 4, 0, 0, False),   # a second wave of one cell
    ((592, 592, 513), 40, 4, 0, 0, False),
    ((301, 277, 259), 21, 4, 0, 1, True),
    ((192, 192, 192), 24, 4, 0, 0, False),
    ((40, 44, 90), 12, 4, 0, 0, False),
    # either side of the lines: the other kernels were faster on the second
    ((302, 278, 256), 20, 4, 0, 0, True),
    ((240, 200, 400), 20, 4, 0, 0, False),
    ((400, 260, 161), 20, 4, 0, 0, True),
    ((350, 350, 160), 20, 4, 0, 0, False),
    ((448, 448, 300), 20, 4, 0, 0, True),
    ((592, 592, 161), 20, 4, 0, 0, False),
    ((330, 330, 256), 20, 4, 3, 0, True),
    ((280, 280, 256), 20, 4, 3, 0, False),
    ((330, 330, 256), 20, 4, 2, 0, True),
    ((302, 278, 256), 20, 4, 2, 0, False),
    ((528, 528, 400), 20, 4, 2, 0, True),
    ((336, 336, 400), 20, 4, 2, 0, False),
    ((300, 300, 180), 20, 4, 3, 1, True),
    ((640, 300, 140), 20, 4, 3, 1, False),
])
def test_full_row_steps(program, grid, b, radius, taper, image, served):
    assert (_result(program, "full-row", *grid, b, radius, taper, image, 3) > 0) == served


# a grid whose forward loop stays in the cache and whose backward loop does not
@pytest.mark.parametrize("arrays, served", [(3, False), (6, True)])
def test_full_row_steps_count_the_loops_arrays(program, arrays, served):
    assert (_result(program, "full-row", 250, 250, 300, 20, 4, 0, 0, arrays) > 0) == served


@pytest.mark.parametrize("taper, image", [(0, 0), (2, 0), (3, 0), (0, 1), (3, 1)])
def test_windows_of_the_full_row_kernel_run_it(program, taper, image):
    """The grids of test_gpu_slab.py, and of the mixed batch, lie where those
    tests say."""
    rows = set()
    for grid, b in test_gpu_slab.SHAPES:
        taken = _result(program, "full-row", *grid, b, 4, taper, image, 3) > 0
        assert taken or (taper and not image), grid
        if taken:
            rows.add((-(-grid[2] // 128), grid[2] % 2))
    assert rows == {(waves, odd) for waves in (2, 3, 4) for odd in (0, 1)}
    served = [_result(program, "full-row", *shot[0], test_gpu_batch.B, 4, taper, image, 3) > 0
              for shot in test_gpu_batch.MIXED]
    assert served == [False, True, False]
