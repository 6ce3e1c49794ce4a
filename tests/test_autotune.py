"""The tile-shape autotuner's bookkeeping, with a stand-in for the library: the
shape recorded and installed for the forward steps is one whose kernel ran.
"""
from types import SimpleNamespace

import pytest

from rtm3d_demo_amd import autotune

TILINGS = [(1, 4, 4), (64, 1, 6), (64, 1, 8), (128, 1, 4)]


class Library:
    """Times every class 1 ms a launch, but `fast` 0.5 ms in class 2."""

    TILINGS = TILINGS

    def __init__(self, mode, fast):
        self.mode, self.fast, self.tiling = mode, fast, {}

    def set_tiling(self, cls, tz, by=0, ry=0, xchunk=0):
        self.tiling[cls] = (tz, by, ry)

    def get_taper_fusion(self, fmt):
        return self.mode

    def timing_read(self, cls):
        return 10, 5.0 if cls == 2 and self.tiling[2] == self.fast else 10.0

    def forward_steps(self, *a):
        pass

    backward_steps = synchronize = timing_enable = forward_steps


# format, row length, border, taper mode, fastest by the clock -> shape recorded
@pytest.mark.parametrize("fmt, nze, blen, mode, fast, want", [
    (0, 90, 12, -1, (1, 4, 4), (128, 1, 4)),
    (0, 91, 12, -1, (1, 4, 4), (64, 1, 8)),
    (0, 90, 12, -1, (0, 0, 0), (0, 0, 0)),
    (0, 90, 12, 1, (1, 4, 4), (1, 4, 4)),
    (1, 90, 12, -1, (1, 4, 4), (128, 1, 4)),
    (1, 90, 12, -1, (0, 0, 0), (128, 1, 4)),
    (2, 90, 12, -1, (64, 1, 6), (64, 1, 6)),
    (1, 91, 12, -1, (1, 4, 4), (1, 4, 4)),      # a pass of its own: plain steps
    (1, 91, 12, 4, (128, 1, 4), (64, 1, 8)),
    (1, 90, 7, -1, (1, 4, 4), (1, 4, 4)),
    (1, 90, 12, 0, (1, 4, 4), (1, 4, 4)),
])
def test_forward_shape_is_one_that_ran(fmt, nze, blen, mode, fast, want):
    lib = Library(mode, fast)
    shot = SimpleNamespace(nt=40, wave_format=fmt, order=8, nze=nze, blen=blen, sze=blen + 2)
    field = SimpleNamespace(zero=lambda: None)
    pair = SimpleNamespace(a=field, b=field)
    best = autotune.tune(lib, shot, None, None, None, None, pair, pair, None, None, field)
    assert best[2][0] == want
    assert lib.tiling[2] == want
