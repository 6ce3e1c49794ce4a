"""The upper tapers of 16-bit forward windows in every form: the default (on
the step's output for even rows, in a pass of their own for odd ones), on the
output whatever the row (mode 4: one-z waves for odd rows), and a pass before
each step (mode 0).  Each against the oracle's operators in the reference's
order, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# rows that fill whole and partial 128- and 64-cell tiles, even and odd; borders
# narrower than the frames of z and of the history layer (b < 8)
SHAPES = [((40, 36, 130), 8), ((40, 36, 131), 8), ((33, 41, 62), 11), ((33, 41, 255), 11),
          ((40, 36, 130), 4), ((33, 41, 62), 5), ((40, 36, 130), 6), ((33, 41, 131), 7)]


@pytest.fixture(scope="module")
def expected(oracle):
    """Start fields, inputs and the oracle's result, once per (fmt, shape, b)."""
    known = {}

    def of(fmt, shape, b, nt, it0, n, cell):
        key = (fmt, shape, b)
        if key not in known:
            rng = np.random.default_rng(8)
            start = [oracle.to_format(rng.uniform(-1, 1, shape).astype(np.float32), fmt)
                     for _ in range(2)]
            v2 = rng.uniform(0, 0.15, shape).astype(np.float32)
            g = oracle.taper_table(b, np.float32(0.5))
            src = rng.uniform(-1, 1, nt).astype(np.float32)
            coefs = oracle.stencil_coefs(8, 10.0, 11.0, 9.0)
            P, PP = (a.copy() for a in start)
            upb = np.zeros((nt, shape[0], shape[1], 4), np.uint16)
            for it in range(it0, it0 + n):
                P, PP = PP, P
                oracle.taper(P, g, b, True, fmt)
                oracle.taper(PP, g, b, True, fmt)
                oracle.step(P, PP, v2, coefs, 8, fmt)
                oracle.apply_source(PP, *cell, src[it], fmt)
                oracle.upb(PP, upb, b, 8, it, False, fmt)
            known[key] = (start, v2, g, src, coefs, [P, PP, upb])
        return known[key]
    return of


@pytest.mark.parametrize("fmt", ["f16", "bf16"])
@pytest.mark.parametrize("mode", [-1, 4, 0], ids=["default", "output", "separate"])
@pytest.mark.parametrize("shape, b", SHAPES)
def test_forward_window(gpu, expected, shape, b, mode, fmt):
    nx, ny, nz = shape
    nt, it0, n = 12, 2, 5
    cell = (nx // 2, ny // 2, b + 1)
    start, v2, g, src, coefs, want = expected(fmt, shape, b, nt, it0, n, cell)
    V, dg, ds = (gpu.DeviceArray.from_host(a) for a in (v2, g, src))
    shot = gpu.make_shot(nx, ny, nz, b, 8, nt, nt, cell, gpu.RcvGeom(0, 0, 0, 2, 2, 3, 3),
                         fmt=fmt)
    F = gpu.FieldPair(shape, dtype=np.uint16)
    F.a.upload(start[0])
    F.b.upload(start[1])
    upb = gpu.DeviceArray((nt, nx, ny, 4), np.uint16).zero()
    gpu.set_taper_fusion(fmt, mode)
    try:
        gpu.forward_steps(shot, 1, V, coefs, dg, ds, F, upb, it0, n)
        got = [F.P.download(), F.PP.download(), upb.download()]
    finally:
        gpu.set_taper_fusion(fmt, -1)
        for d in (F, upb, V, dg, ds):
            d.free()
    for name, a, w in zip(("P", "PP", "history"), got, want):
        assert np.array_equal(a, w), name
