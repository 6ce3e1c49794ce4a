"""The 16-bit default of the upper tapers: on the step's output for even rows,
in a pass of their own for odd ones.  A forward window in the default mode equals mode 0 (a pass before each step) bit for bit: the same
operators in the same order on stored values.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _narrow(a, fmt):
    if fmt == "f16":
        return a.astype(np.float16).view(np.uint16)
    return (a.view(np.uint32) >> 16).astype(np.uint16)


@pytest.mark.parametrize("fmt", ["f16", "bf16"])
@pytest.mark.parametrize("shape, b", [((40, 36, 130), 8), ((40, 36, 131), 8), ((33, 41, 62), 11),
                                      ((33, 41, 255), 11)])
def test_default_equals_separate_pass(gpu, oracle, shape, b, fmt):
    rng = np.random.default_rng(8)
    nx, ny, nz = shape
    nt, n = 12, 5
    start = [_narrow(rng.uniform(-1, 1, shape).astype(np.float32), fmt) for _ in range(2)]
    V = gpu.DeviceArray.from_host(rng.uniform(0, 0.15, shape).astype(np.float32))
    g = gpu.DeviceArray.from_host(oracle.taper_table(b, np.float32(0.5)))
    src = gpu.DeviceArray.from_host(rng.uniform(-1, 1, nt).astype(np.float32))
    coefs = oracle.stencil_coefs(8, 10.0, 11.0, 9.0)
    shot = gpu.make_shot(nx, ny, nz, b, 8, nt, nt, (nx // 2, ny // 2, b + 1),
                         gpu.RcvGeom(0, 0, 0, 2, 2, 3, 3), fmt=fmt)
    got = {}
    for mode in (-1, 0):
        gpu.set_taper_fusion(fmt, mode)
        F = gpu.FieldPair(shape, dtype=np.uint16)
        F.a.upload(start[0])
        F.b.upload(start[1])
        upb = gpu.DeviceArray((nt, nx, ny, 4), np.uint16).zero()
        try:
            gpu.forward_steps(shot, 1, V, coefs, g, src, F, upb, 2, n)
            got[mode] = [F.P.download(), F.PP.download(), upb.download()]
        finally:
            gpu.set_taper_fusion(fmt, -1)
            F.a.free()
            F.b.free()
            upb.free()
    for a, w in zip(got[-1], got[0]):
        assert np.array_equal(a, w)
    for d in (V, g, src):
        d.free()
