"""The launch that follows a step (k_tail_all, k_tail_upper: border frame,
upper-border layer, receivers, image frame, source together) where its parts
meet: the source on a receiver's cell, in the upper-border layer, on the
border; receivers on the border; rows that cannot be moved in fours; borders
narrower than the two frames of an output-tapered step.  Modeling, HBC and RBC
migration windows against the oracle's operators in the reference's order, bit
for bit.
"""
import pytest

import test_gpu_slab as windows

pytestmark = pytest.mark.gpu

# (grid, border, source cell, receivers (x0, y0, z, dx, dy, nx, ny) counted
# from the border)
CASES = [
    ((44, 40, 48), 12, (15, 14, 13), (0, 0, 1, 3, 2, 6, 8)),  # source on a receiver
    ((44, 40, 48), 12, (15, 14, 10), (1, 0, 3, 3, 2, 6, 8)),  # source in the layer
    ((43, 41, 47), 11, (14, 13, 9), (0, 0, 0, 3, 2, 6, 8)),   # odd rows and border
    ((44, 40, 48), 8, (20, 20, 8), (0, 0, 0, 1, 1, 28, 24)),  # every cell, b = 2R
    ((44, 40, 48), 7, (20, 20, 5), (0, 0, 1, 2, 2, 12, 12)),  # b < 2R
    ((44, 40, 48), 12, (3, 14, 13), (1, 1, 2, 3, 2, 11, 18)),  # on the borders
]


@pytest.fixture
def window(monkeypatch):
    setup = windows._setup

    def use(cell, geo):
        def patched(gpu, po, shape, blen, seed):
            import numpy as np
            c = setup(gpu, po, shape, blen, seed)
            rng = np.random.default_rng(seed + 10)
            rcv = rng.standard_normal((geo[5], geo[6], c["nt"])).astype(np.float32)
            return dict(c, cell=cell, geo=geo, rcv=rcv)
        monkeypatch.setattr(windows, "_setup", patched)
    return use


@pytest.mark.parametrize("shape,blen,cell,geo", CASES)
def test_modeling(gpu, oracle, window, shape, blen, cell, geo):
    window(cell, geo)
    windows.test_modeling_window(gpu, oracle, shape, blen)


@pytest.mark.parametrize("hbc", [1, 0])
@pytest.mark.parametrize("shape,blen,cell,geo", CASES)
def test_migration(gpu, oracle, window, shape, blen, cell, geo, hbc):
    window(cell, geo)
    windows.test_migration_window(gpu, oracle, shape, blen, hbc)
