"""The launch that follows a step (k_tail_all, k_tail_upper: border frame,
upper-border layer, receivers, image frame, source together) where its parts
meet: the source on a receiver's cell, in the upper-border layer, on the
border; receivers on the border; rows that cannot be moved in fours; borders
narrower than the two frames of an output-tapered step.  Modeling, HBC and RBC
migration windows against the oracle's operators in the reference's order, bit
for bit.
"""
import numpy as np
import pytest

import windows

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


def _window(oracle, shape, blen, cell, geo, seed):
    c = windows.setup(oracle, shape, blen, seed, cell, geo)
    rng = np.random.default_rng(seed + 10)
    c["rcv"] = rng.standard_normal((geo[5], geo[6], c["nt"])).astype(np.float32)
    return c


@pytest.mark.parametrize("shape,blen,cell,geo", CASES)
def test_modeling(gpu, oracle, shape, blen, cell, geo):
    windows.modeling(gpu, oracle, _window(oracle, shape, blen, cell, geo, 1))


@pytest.mark.parametrize("hbc", [1, 0])
@pytest.mark.parametrize("shape,blen,cell,geo", CASES)
def test_migration(gpu, oracle, shape, blen, cell, geo, hbc):
    windows.migration(gpu, oracle, _window(oracle, shape, blen, cell, geo, 2), hbc)


# borders down to the stencil's radius: the layer and the z frame share cells
NARROW = [((44, 40, 48), 4), ((43, 41, 47), 5), ((44, 40, 48), 6), ((33, 36, 131), 7),
          ((160, 600, 250), 4), ((160, 602, 251), 5), ((128, 585, 337), 6),
          ((104, 503, 500), 7)]


@pytest.mark.parametrize("shape,blen", NARROW)
def test_narrow_borders(gpu, oracle, shape, blen):
    nx, ny, nz = shape
    cell = (nx // 2, ny // 2, blen)
    geo = (0, 0, 0, 3, 2, (nx - 2 * blen) // 3, (ny - 2 * blen) // 2)
    windows.migration(gpu, oracle, _window(oracle, shape, blen, cell, geo, 2), 1)


@pytest.mark.parametrize("fmt,mode", [("f32", -1), ("f16", 4)])
@pytest.mark.parametrize("blen", [4, 5, 6, 7, 8])
def test_narrow_borders_keep_the_output_form(gpu, oracle, blen, fmt, mode):
    """A forward window with the upper taper on the output runs every step but
    the last as the tapered kernel class (2) and the last as the plain one (0);
    with tapers on load or in a pass of their own every step is of one class."""
    shape, nt, n = (40, 44, 90), 8, 5
    wd = gpu.WAVE_FORMATS[fmt][1]
    V = gpu.DeviceArray(shape).zero()
    g = gpu.DeviceArray.from_host(oracle.taper_table(blen, np.float32(0.9)))
    src = gpu.DeviceArray((nt,)).zero()
    F = gpu.FieldPair(shape, wd)
    upb = gpu.DeviceArray((nt, shape[0], shape[1], 4), wd)
    shot = gpu.make_shot(*shape, blen, 8, nt, nt, (20, 22, blen), gpu.RcvGeom(0, 0, 0, 2, 2, 3, 3),
                         fmt=fmt)
    gpu.timing_enable(True)
    gpu.set_taper_fusion(fmt, mode)
    try:
        for cls in (0, 2):
            gpu.timing_read(cls)
        gpu.forward_steps(shot, 1, V, oracle.stencil_coefs(8, 10.0, 11.0, 9.0), g, src, F, upb,
                          0, n)
        runs = [gpu.timing_read(cls)[0] for cls in (0, 2)]
    finally:
        gpu.timing_enable(False)
        gpu.set_taper_fusion(fmt, -1)
        for d in (V, g, src, F, upb):
            d.free()
    assert runs == [1, n - 1]
