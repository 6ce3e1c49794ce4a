"""Windows of the FP32 order-8 loops on dense random states against the
oracle's operators in the reference's order, bit for bit: inputs and the
comparison, shared by the tests of the kernels that those loops run.
"""
import numpy as np

NT = 40


def setup(po, shape, blen, seed, cell=None, geo=None):
    """Inputs of a window.  cell: the source's (extended grid); geo: receivers
    (x0, y0, z, dx, dy, nx, ny) counted from the border."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = shape

    def dense():
        a = np.zeros(shape, np.float32)
        a[4:-4, 4:-4, 4:-4] = rng.standard_normal((nx - 8, ny - 8, nz - 8), np.float32)
        return a

    order, nt, d = 8, NT, 10.0
    vel = rng.uniform(1500.0, 4500.0, shape).astype(np.float32)
    v2 = po.v2dt2(vel, np.float32(0.4 * d / 4500.0))
    coefs = po.stencil_coefs(order, d, 12.0, 11.0)
    g = po.taper_table(blen, np.float32(0.9))
    src = po.ricker(nt, np.float32(1e-3), np.float32(25.0))
    geo = geo or (1, 0, 1, 3, 2, (nx - 2 * blen) // 3, (ny - 2 * blen) // 2)
    rcv = rng.standard_normal((geo[5], geo[6], nt)).astype(np.float32)
    return dict(order=order, nt=nt, v2=v2, coefs=coefs, g=g, src=src, geo=geo, rcv=rcv,
                fields=[dense() for _ in range(4)], b=blen, shape=shape,
                cell=cell or (nx // 2, ny // 2, blen + 2))


def device(gpu, c, names):
    dev = {k: gpu.DeviceArray.from_host(c[k]) for k in ("v2", "g", "src", "rcv")}
    for n, (i, j) in names.items():
        f = gpu.FieldPair(c["shape"])
        f.a.upload(c["fields"][i])
        f.b.upload(c["fields"][j])
        dev[n] = f
    dev["shot"] = gpu.make_shot(*c["shape"], c["b"], c["order"], c["nt"], c["nt"], c["cell"],
                                gpu.RcvGeom(*c["geo"]))
    return dev


def same(got, want, what):
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), what


def free(dev):
    for k, d in dev.items():
        if k != "shot":
            d.free()


def modeling(gpu, oracle, c, n=4, it0=7):
    b = c["b"]
    dev = device(gpu, c, {"S": (0, 1)})
    gpu.model_steps(dev["shot"], dev["v2"], c["coefs"], dev["g"], dev["src"], dev["S"],
                    dev["rcv"], it0, n)
    P, PP = (c["fields"][i].copy() for i in (0, 1))
    rcv = c["rcv"].copy()
    geo = oracle.RcvGeom(*c["geo"])
    for it in range(it0, it0 + n):
        P, PP = PP, P
        oracle.taper(P, c["g"], b, False)
        oracle.taper(PP, c["g"], b, False)
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        oracle.apply_source(PP, *c["cell"], c["src"][it])
        oracle.receivers(PP, rcv, b, geo, c["nt"], it, False)
    same(dev["S"].P.download(), P, "P")
    same(dev["S"].PP.download(), PP, "PP")
    same(dev["rcv"].download(), rcv, "record")
    free(dev)


def migration(gpu, oracle, c, hbc, n=4, it0=7):
    """A forward window, then the backward window over the same steps."""
    b, shape = c["b"], c["shape"]
    nx, ny, nz = shape
    dev = device(gpu, c, {"S": (0, 1), "R": (2, 3)})
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
            oracle.taper(P, c["g"], b, True)
            oracle.taper(PP, c["g"], b, True)
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        oracle.apply_source(PP, *c["cell"], c["src"][it])
        if hbc:
            oracle.upb(PP, upb, b, 8, it, False)
    same(dev["S"].P.download(), P, "forward P")
    same(dev["S"].PP.download(), PP, "forward PP")
    same(dev["upb"].download(), upb, "history")
    hi = it0 + n - 1
    gpu.backward_steps(dev["shot"], hbc, *args, dev["S"], dev["R"], dev["upb"], dev["rcv"],
                       dev["img"], hi, n, True)
    img = np.zeros(shape, np.float32)
    for it in range(hi, hi - n, -1):
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        if hbc:
            oracle.upb(PP, upb, b, 8, it, True)
        P, PP = PP, P
        if hbc:
            oracle.taper(Pr, c["g"], b, True)
            oracle.taper(PPr, c["g"], b, True)
        assert oracle.step(Pr, PPr, c["v2"], c["coefs"], 8) == 0
        oracle.receivers(PPr, c["rcv"], b, geo, c["nt"], it, True)
        oracle.image(img, P, PPr, b)
        Pr, PPr = PPr, Pr
    for name, d, want in (("S.P", dev["S"].P, P), ("S.PP", dev["S"].PP, PP),
                          ("R.P", dev["R"].P, Pr), ("R.PP", dev["R"].PP, PPr),
                          ("image", dev["img"], img)):
        same(d.download(), want, name)
    free(dev)


def frequency(gpu, oracle, c, n=3):
    """Steps of the frequency-domain loop, one frequency at a time."""
    b, shape, nt = c["b"], c["shape"], c["nt"]
    hi = nt - 1
    rng = np.random.default_rng(3)
    inner = (1,) + tuple(s - 2 * b for s in shape)
    acc = [rng.uniform(-1, 1, inner).astype(np.float32) for _ in range(4)]
    w2, kre, kim = oracle.freq_tables(nt, np.float32(0.004), np.float32(2.0), np.float32(40.0))
    w2, kre, kim = (np.ascontiguousarray(a[:1]) for a in (w2, kre, kim))
    img = rng.uniform(-1, 1, shape).astype(np.float32)
    dev = device(gpu, c, {"S": (0, 1), "R": (2, 3)})
    dacc = [gpu.DeviceArray.from_host(a) for a in acc]
    tabs = [gpu.DeviceArray.from_host(a) for a in (kre, kim, w2)]
    dev["img"] = gpu.DeviceArray.from_host(img)
    gpu.freq_steps(dev["shot"], dev["v2"], c["coefs"], dev["g"], dev["src"], dev["S"], dev["R"],
                   dev["rcv"], dev["img"], dacc, *tabs, 1, 0, 1, hi, n)
    Ps, PPs, Pr, PPr = (f.copy() for f in c["fields"])
    geo = oracle.RcvGeom(*c["geo"])
    for rt in range(hi, hi - n, -1):
        st = nt - 1 - rt
        assert oracle.step(Ps, PPs, c["v2"], c["coefs"], 8) == 0
        assert oracle.step(Pr, PPr, c["v2"], c["coefs"], 8) == 0
        for f in (Ps, PPs, Pr, PPr):
            oracle.taper(f, c["g"], b, False)
        oracle.apply_source(PPs, *c["cell"], c["src"][st])
        oracle.receivers(PPr, c["rcv"], b, geo, nt, rt, True)
        oracle.freq_image(img, PPs, PPr, acc, kre, kim, w2, b, 1, 0, nt, st)
        Ps, PPs = PPs, Ps
        Pr, PPr = PPr, Pr
    for name, d, want in [("S.P", dev["S"].P, Ps), ("S.PP", dev["S"].PP, PPs),
                          ("R.P", dev["R"].P, Pr), ("R.PP", dev["R"].PP, PPr),
                          ("image", dev["img"], img)] + list(zip("abcd", dacc, acc)):
        same(d.download(), want, name)
    free(dev)
    for d in dacc + tabs:
        d.free()


def snapshots(gpu, oracle, c, n=4, k=2):
    """The last n steps forward with FP32 snapshots every k, then backward
    (receiver field only, imaged with them)."""
    b, shape, nt = c["b"], c["shape"], c["nt"]
    z = slice(b, shape[2] - b)
    dev = device(gpu, c, {"S": (0, 1), "R": (2, 3)})
    snaps = gpu.snap_buffer(dev["shot"], "f32", k)
    dev["img"] = gpu.DeviceArray(shape).zero()
    args = (dev["v2"], c["coefs"], dev["g"])
    gpu.snap_forward_steps(dev["shot"], *args, dev["src"], dev["S"], snaps, "f32", k, nt - n, n)
    P, PP, Pr, PPr = (f.copy() for f in c["fields"])
    geo = oracle.RcvGeom(*c["geo"])
    kept = {}
    for it in range(nt - n, nt):
        P, PP = PP, P
        oracle.taper(P, c["g"], b, True)
        oracle.taper(PP, c["g"], b, True)
        assert oracle.step(P, PP, c["v2"], c["coefs"], 8) == 0
        oracle.apply_source(PP, *c["cell"], c["src"][it])
        if (nt - 1 - it) % k == 0:
            kept[it] = PP[:, :, z].copy()
    same(dev["S"].P.download(), P, "forward P")
    same(dev["S"].PP.download(), PP, "forward PP")
    gpu.snap_backward_steps(dev["shot"], *args, dev["R"], snaps, "f32", k, dev["rcv"],
                            dev["img"], nt - 1, n)
    img = np.zeros(shape, np.float32)
    for it in range(nt - 1, nt - 1 - n, -1):
        oracle.taper(Pr, c["g"], b, True)
        oracle.taper(PPr, c["g"], b, True)
        assert oracle.step(Pr, PPr, c["v2"], c["coefs"], 8) == 0
        oracle.receivers(PPr, c["rcv"], b, geo, nt, it, True)
        if it in kept:
            img[:, :, z] = img[:, :, z] + np.float32(k) * (kept[it] * PPr[:, :, z])
        Pr, PPr = PPr, Pr
    for name, d, want in (("R.P", dev["R"].P, Pr), ("R.PP", dev["R"].PP, PPr),
                          ("image", dev["img"], img)):
        same(d.download(), want, name)
    snaps.free()
    free(dev)
