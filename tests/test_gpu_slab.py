"""The FP32 order-8 step on full-row blocks (k_slab), which the loops use by
default on grids large enough for it: modeling, HBC and RBC migration windows
on dense random states against the oracle's operators in the reference's
order, bit for bit, at the edges of the kernel's range -- rows of two to four
128-cell waves, odd and even, just past and just at a wave; last blocks of
one row and of every row; odd and even borders.  test_launch_limits.py checks
that every shape here takes the kernel for the plain and the imaging step, and
the tapered forms for each number of waves, odd and even.
"""
import pytest

import windows

pytestmark = pytest.mark.gpu

SHAPES = [
    ((160, 600, 250), 21),  # two waves per row, even rows, odd border
    ((160, 602, 251), 10),  # odd rows: the last pair is half outside
    ((160, 603, 256), 32),  # two whole waves; last block of one row
    ((128, 592, 336), 40),  # three waves
    ((128, 585, 337), 24),  # last block of one row
    ((160, 587, 383), 8),
    ((128, 592, 384), 16),
    ((104, 503, 500), 40),  # four waves; whole blocks
    ((104, 504, 509), 12),
    ((104, 500, 512), 9),
    # grids past the Infinity Cache, where even rows take the tapered forms too
    ((200, 603, 250), 13),
    ((152, 592, 336), 40),
    ((160, 585, 384), 15),  # last block of one row
    ((136, 503, 500), 10),
    ((130, 500, 512), 33),
]


@pytest.mark.parametrize("shape,blen", SHAPES)
def test_modeling_window(gpu, oracle, shape, blen):
    windows.modeling(gpu, oracle, windows.setup(oracle, shape, blen, 1))


@pytest.mark.parametrize("hbc", [1, 0])
@pytest.mark.parametrize("shape,blen", SHAPES)
def test_migration_window(gpu, oracle, shape, blen, hbc):
    windows.migration(gpu, oracle, windows.setup(oracle, shape, blen, 2), hbc)


# one step is a call's first and last: both tapers in place before it
@pytest.mark.parametrize("shape,blen", SHAPES[:2])
@pytest.mark.parametrize("n", [1, 2])
def test_short_migration_window(gpu, oracle, shape, blen, n):
    windows.migration(gpu, oracle, windows.setup(oracle, shape, blen, 4), 1, n)


# taper3D on the output with and without the older field's taper
@pytest.mark.parametrize("shape,blen", [SHAPES[1], SHAPES[5], SHAPES[10], SHAPES[13]])
def test_frequency_window(gpu, oracle, shape, blen):
    windows.frequency(gpu, oracle, windows.setup(oracle, shape, blen, 5))


# the upper taper on the output of the whole border
@pytest.mark.parametrize("shape,blen", [SHAPES[1], SHAPES[4], SHAPES[10], SHAPES[14]])
def test_snapshot_window(gpu, oracle, shape, blen):
    windows.snapshots(gpu, oracle, windows.setup(oracle, shape, blen, 6))
