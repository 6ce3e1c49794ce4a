"""The step on planes of exactly 4 GB (2^30 FP32 cells): the buffer views of the
waves hold a plane's size in 32 bits.  Impulses in a field of zeros, near the
plane's corners and in it, against the step's definition: 2p - 0 + v lap with
one term, or the three centre terms, in the sum.  Three fields of 39 GB.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (9, 32768, 32768)
POINTS = [(4, 4, 4), (4, 100, 200), (4, 16384, 16384), (4, 32763, 32763), (4, 32763, 4),
          (4, 20000, 31000)]


def _row(gpu, field, x, y, z, n):
    """n cells of a row as an array of their own (not freed by itself)."""
    a = gpu.DeviceArray.__new__(gpu.DeviceArray)
    a.shape, a.dtype, a.nbytes = (n,), np.dtype(np.float32), 4 * n
    a.ptr = C.c_void_p(field.ptr.value + 4 * ((x * SHAPE[1] + y) * SHAPE[2] + z))
    return a


def test_step(gpu, oracle):
    fields = []
    try:
        try:
            for _ in range(3):
                fields.append(gpu.DeviceArray(SHAPE).zero())
        except gpu.RtmError as e:
            pytest.skip("116 GB of device memory: %s" % e)
        P, PP, V = fields
        gpu.check(gpu.load().rtmhip_fill(V.ptr, V.size, C.c_float(0.1)))
        c = oracle.stencil_coefs(8, 10.0, 11.0, 9.0).reshape(3, 9)
        for p in POINTS:
            _row(gpu, P, *p, 1).upload(np.ones(1, np.float32))
        gpu.step(P, PP, V, c.ravel(), 8)
        v = np.float32(0.1)
        for x, y, z in POINTS:
            for y1 in range(y - 4, y + 5):
                z0, z1 = max(z - 4, 0), min(z + 5, SHAPE[2])
                want = np.zeros(z1 - z0, np.float32)
                for k in range(z0, z1):
                    if not (4 <= y1 < SHAPE[1] - 4 and 4 <= k < SHAPE[2] - 4):
                        continue  # not updated
                    if y1 == y and k == z:
                        want[k - z0] = np.float32(2) + v * (c[0, 4] + c[1, 4] + c[2, 4])
                    elif y1 == y:
                        want[k - z0] = v * c[2, 4 - (k - z)]
                    elif k == z:
                        want[k - z0] = v * c[1, 4 - (y1 - y)]
                got = _row(gpu, PP, x, y1, z0, z1 - z0).download()
                assert np.array_equal(got, want), (x, y1, z0)
    finally:
        for f in fields:
            f.free()
