"""The FP32 order-8 step on full-row blocks (k_slab), which the loops use by
default on grids large enough for it: modeling, HBC and RBC migration windows
on dense random states against the oracle's operators in the reference's
order, bit for bit, at the edges of the kernel's range -- rows of one to four
128-cell waves, odd and even, just past and just at a wave; last blocks of
one row and of every row; odd and even borders.
"""
import numpy as np
import pytest

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
]


def _setup(gpu, po, shape, blen, seed):
    rng = np.random.default_rng(seed)
    nx, ny, nz = shape

    def dense():
        a = np.zeros(shape, np.float32)
        a[4:-4, 4:-4, 4:-4] = rng.standard_normal((nx - 8, ny - 8, nz - 8), np.float32)
        return a

    order, nt, d = 8, 40, 10.0
    vel = rng.uniform(1500.0, 4500.0, shape).astype(np.float32)
    v2 = po.v2dt2(vel, np.float32(0.4 * d / 4500.0))
    coefs = po.stencil_coefs(order, d, 12.0, 11.0)
    g = po.taper_table(blen, np.float32(0.9))
    src = po.ricker(nt, np.float32(1e-3), np.float32(25.0))
    geo = (1, 0, 1, 3, 2, (nx - 2 * blen) // 3, (ny - 2 * blen) // 2)
    rcv = rng.standard_normal((geo[5], geo[6], nt)).astype(np.float32)
    return dict(order=order, nt=nt, v2=v2, coefs=coefs, g=g, src=src, geo=geo, rcv=rcv,
                fields=[dense() for _ in range(4)], b=blen, shape=shape,
                cell=(nx // 2, ny // 2, blen + 2))


def _device(gpu, c, names):
    dev = {k: gpu.DeviceArray.from_host(c[k]) for k in ("v2", "g", "src", "rcv")}
    for n, (i, j) in names.items():
        f = gpu.FieldPair(c["shape"])
        f.a.upload(c["fields"][i])
        f.b.upload(c["fields"][j])
        dev[n] = f
    dev["shot"] = gpu.make_shot(*c["shape"], c["b"], c["order"], c["nt"], c["nt"], c["cell"],
                                gpu.RcvGeom(*c["geo"]))
    return dev


def _same(got, want, what):
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), what


def _free(dev):
    for k, d in dev.items():
        if k != "shot":
            d.free()


@pytest.mark.parametrize("shape,blen", SHAPES)
def test_modeling_window(gpu, oracle, shape, blen):
    c = _setup(gpu, oracle, shape, blen, 1)
    n, it0 = 4, 7
    dev = _device(gpu, c, {"S": (0, 1)})
    gpu.model_steps(dev["shot"], dev["v2"], c["coefs"], dev["g"], dev["src"], dev["S"],
                    dev["rcv"], it0, n)
    P, PP = (c["fields"][i].copy() for i in (0, 1))
    rcv = c["rcv"].copy()
    geo = oracle.RcvGeom(*c["geo"])
    for it in range(it0, it0 + n):
        P, PP = PP, P
        oracle.taper(P, c["g"], blen, False)
        oracle.taper(PP, c["g"], blen, False)
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        oracle.apply_source(PP, *c["cell"], c["src"][it])
        oracle.receivers(PP, rcv, blen, geo, c["nt"], it, False)
    _same(dev["S"].P.download(), P, "P")
    _same(dev["S"].PP.download(), PP, "PP")
    _same(dev["rcv"].download(), rcv, "record")
    _free(dev)


@pytest.mark.parametrize("hbc", [1, 0])
@pytest.mark.parametrize("shape,blen", SHAPES)
def test_migration_window(gpu, oracle, shape, blen, hbc):
    c = _setup(gpu, oracle, shape, blen, 2)
    n, it0 = 4, 7
    nx, ny, nz = shape
    dev = _device(gpu, c, {"S": (0, 1), "R": (2, 3)})
    dev["img"] = gpu.DeviceArray(shape).zero()
    dev["upb"] = gpu.DeviceArray((c["nt"], nx, ny, 4)).zero()
    args = (dev["v2"], c["coefs"], dev["g"])
    gpu.forward_steps(dev["shot"], hbc, *args, dev["src"], dev["S"], dev["upb"], it0, n)
    P, PP, Pr, PPr = (f.copy() for f in c["fields"])
    upb = np.zeros((c["nt"], nx, ny, 4), np.float32)
    geo = oracle.RcvGeom(*c["geo"])
    for it in range(it0, it0 + n):
        P, PP = PP, P
        if hbc:
            oracle.taper(P, c["g"], blen, True)
            oracle.taper(PP, c["g"], blen, True)
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        oracle.apply_source(PP, *c["cell"], c["src"][it])
        if hbc:
            oracle.upb(PP, upb, blen, 8, it, False)
    _same(dev["S"].P.download(), P, "forward P")
    _same(dev["S"].PP.download(), PP, "forward PP")
    _same(dev["upb"].download(), upb, "history")
    hi = it0 + n - 1
    gpu.backward_steps(dev["shot"], hbc, *args, dev["S"], dev["R"], dev["upb"], dev["rcv"],
                       dev["img"], hi, n, True)
    img = np.zeros(shape, np.float32)
    for it in range(hi, hi - n, -1):
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        if hbc:
            oracle.upb(PP, upb, blen, 8, it, True)
        P, PP = PP, P
        if hbc:
            oracle.taper(Pr, c["g"], blen, True)
            oracle.taper(PPr, c["g"], blen, True)
        assert oracle.step(Pr, PPr, c["v2"], c["coefs"], 8) == 0
        oracle.receivers(PPr, c["rcv"], blen, geo, c["nt"], it, True)
        oracle.image(img, P, PPr, blen)
        Pr, PPr = PPr, Pr
    for name, d, want in (("S.P", dev["S"].P, P), ("S.PP", dev["S"].PP, PP),
                          ("R.P", dev["R"].P, Pr), ("R.PP", dev["R"].PP, PPr),
                          ("image", dev["img"], img)):
        _same(d.download(), want, name)
    _free(dev)
