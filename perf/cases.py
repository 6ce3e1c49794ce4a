"""Workloads whose time is followed from version to version.

Every case is one pass through the library's public entry points
(rtm3d_demo_amd.hip and rtm3d_demo_amd.ae, the bindings of include/rtm_hip.h)
as a migration program calls them: a window of time steps of a shot that is
under way, or one snapshot through the coder, or a few training steps.  The
wavefields are dense (a smooth random field stands for the state in mid-shot,
when the wave has filled the aperture) and go on propagating from pass to pass,
as the chunks of a shot do.  The velocity model is v(z) = 1500 + 0.8 z[m],
capped at 4500, with a smooth 5 % perturbation and an ellipsoidal salt body;
12.5 m cells, CFL 0.4.

listed() holds the cases, draw() gives others of the same ranges, prepare()
makes what the program holds before the call, run() is the call, work() says
what a pass cannot do without and exact() gives its result in 64 bits from
plain torch.
"""
import ctypes
import math
import random

import numpy as np
import torch
import torch.nn.functional as F

from rtm3d_demo_amd import ae, hip

SPACING, VMAX, COURANT = 12.5, 4500.0, 0.4
WAVES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
TAPS = {2: [-2.0, 1.0], 4: [-5 / 2, 4 / 3, -1 / 12], 6: [-49 / 18, 3 / 2, -3 / 20, 1 / 90],
        8: [-205 / 72, 8 / 5, -1 / 5, 8 / 315, -1 / 560]}


# --------------------------------------------------------------- the cases
def _shot(name, kind, nx, ny, nz, blen, steps, wave="f32", order=8, stride=4, **more):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, blen=blen, steps=steps, wave=wave,
                order=order, stride=stride, **more)


def listed():
    return [
        # a small survey model with odd sides and a low stencil order, as the
        # reference's own small inputs have them: launches and latency count
        _shot("model_small_o4", "model", 33, 39, 37, 6, 25, order=4, stride=2),
        # the three-layer modeling workload (128^3 and a border of 32): fits
        # the caches, many short steps
        _shot("model_192", "model", 192, 192, 192, 32, 25, stride=2),
        # the benchmark's shot (512 x 512 x 256 and a border of 40), its
        # forward pass with the upper-border history ...
        _shot("hbc_forward_592", "hbc_forward", 592, 592, 336, 40, 10),
        # ... and its backward pass: source reconstruction, receiver step,
        # imaging
        _shot("hbc_backward_592", "hbc_backward", 592, 592, 336, 40, 10),
        # random-border migration on a grid of odd sides, both directions
        _shot("rbc_301", "rbc", 301, 277, 259, 20, 8, stride=3),
        # the 800 x 800 x 400 model with 16-bit wavefields, both directions
        _shot("hbc_880_f16", "hbc", 880, 880, 480, 40, 6, wave="f16"),
        # snapshot migration with 16-bit wavefields and FP16 snapshots of
        # every 4th step, both directions
        _shot("snap_592_f16", "snap", 592, 592, 336, 40, 16, wave="f16", every=4),
        # snapshot migration of the largest batch window with
        # transform-coded snapshots, both directions
        _shot("snap_dct_528", "snap_dct", 528, 528, 400, 40, 8, every=4),
        # frequency-domain migration, a group of 4 frequencies
        _shot("freq_592", "freq", 592, 592, 336, 40, 4, nw=4),
        # uneven apertures of one survey migrated together, both directions
        dict(name="batch_6", kind="batch", shots=6, lo=256, hi=448, zlo=256, zhi=320, mix=64,
             blen=40, steps=18, wave="f32"),
        # the learned code of one snapshot of the benchmark's shot: bricks,
        # encoding and decoding
        dict(name="codes_592", kind="codes", nx=592, ny=592, nz=336, blen=40),
        # training that code: Adam steps on batches of 64 bricks
        dict(name="train_64", kind="train", bricks=64, iters=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["model", "model", "hbc_forward", "hbc_backward", "rbc", "hbc", "snap",
                       "snap_dct", "freq", "batch", "codes", "train"])
    if kind == "train":
        return dict(kind=kind, bricks=_log(rng, 8, 128), iters=rng.randint(3, 10))
    if kind == "batch":
        lo = rng.choice([64, 128, 192, 256])
        return dict(kind=kind, shots=rng.randint(2, 6), lo=lo, hi=lo + rng.choice([64, 128, 192]),
                    zlo=lo, zhi=lo + 64, mix=rng.randint(1, 10000), blen=rng.choice([16, 24, 40]),
                    steps=2 * rng.randint(5, 10), wave=rng.choice(["f32", "f32", "f16"]))
    lo = 33 if kind == "model" else 80
    nx, ny, nz = (_log(rng, lo, 640) for _ in range(3))
    nz = min(nz, 520)
    blen = max(5, min(rng.choice([6, 10, 16, 21, 32, 40]), (min(nx, ny, nz) - 8) // 3))
    if rng.random() < 0.5:  # half of the grids with even sides, as most configurations
        nx, ny, nz, blen = (v + v % 2 for v in (nx, ny, nz, blen))
    if kind == "codes":
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, blen=blen)
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz, blen=blen, steps=2 * rng.randint(2, 12),
                wave="f32", order=8, stride=rng.choice([1, 2, 3, 4, 5]))
    if kind in ("model", "rbc"):
        case["order"] = rng.choice([8, 8, 8, 2, 4, 6])
    if case["order"] == 8 and kind != "freq":
        case["wave"] = rng.choice(["f32", "f32", "f16", "bf16"])
    if kind in ("snap", "snap_dct"):
        case["every"] = rng.choice([2, 4, 5])
    if kind == "freq":
        case["nw"] = rng.randint(1, 7)
    return case


def draw(rng):
    most = max(work(c)["bytes"] for c in listed())
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= most:
            return case


# ---------------------------------------------------------------- the inputs
def _noise(shape, gen, step=4, amplitude=1.0):
    """A smooth random field: normal values every `step` cells, interpolated."""
    coarse = torch.randn([1, 1] + [max(2, n // step + 1) for n in shape], generator=gen,
                         device="cuda")
    return F.interpolate(coarse, size=tuple(shape), mode="trilinear",
                         align_corners=True)[0, 0] * amplitude


def _velocity(shape, blen, gen):
    """v^2 dt^2 of the model on the extended grid."""
    nx, ny, nz = shape
    ax = [torch.arange(n, device="cuda", dtype=torch.float32) for n in shape]
    vz = torch.clamp(1500.0 + 0.8 * SPACING * torch.clamp(ax[2] - blen, min=0.0), max=VMAX)
    v = vz * (1.0 + 0.02 * _noise(shape, gen, 8).clamp(-2.5, 2.5))
    r2 = (((ax[0] - 0.45 * nx) / (0.17 * nx)) ** 2)[:, None, None] + \
         (((ax[1] - 0.55 * ny) / (0.15 * ny)) ** 2)[None, :, None] + \
         (((ax[2] - 0.55 * nz) / (0.12 * nz)) ** 2)[None, None, :]
    v = torch.where(r2 < 1.0, VMAX, v).clamp(max=VMAX)
    dt = COURANT * SPACING / VMAX
    return (v * dt) ** 2


def _wave(shape, order, gen, wave):
    """A wavefield in mid-shot; the frame that no step updates is zero."""
    r = order // 2
    out = torch.zeros(shape, device="cuda")
    inner = tuple(slice(r, n - r) for n in shape)
    out[inner] = _noise(shape, gen)[inner]
    return out.to(WAVES[wave])


def _coefs(order):
    t = TAPS[order]
    return np.array([t[:0:-1] + t] * 3, np.float32) / np.float32(SPACING ** 2)


def _tables(blen, nt):
    dt = COURANT * SPACING / VMAX
    a = (math.pi * 25.0 * (np.arange(nt) * dt - 0.05)) ** 2
    ricker = ((1.0 - 2.0 * a) * np.exp(-a)).astype(np.float32)
    g = (1.0 - 0.1 * ((np.arange(blen) + 1.0) / blen) ** 2).astype(np.float32)
    return torch.from_numpy(ricker).cuda(), torch.from_numpy(g).cuda()


#: time steps of a shot and of one receiver chunk, and the step a pass starts at
def _times(case):
    kind, n = case["kind"], case["steps"]
    if kind in ("snap", "snap_dct", "batch"):
        return n + 8, n + 8, 4
    return 100 * n, 2 * n, 50 * n


class Shot:
    """One shot's inputs as tensors on the GPU (everything from the seed)."""

    def __init__(self, case, seed, shape=None):
        gen = torch.Generator("cuda").manual_seed(seed)
        self.kind, self.wave = case["kind"], case["wave"]
        self.order, self.blen, self.steps = case.get("order", 8), case["blen"], case["steps"]
        self.shape = shape or (case["nx"], case["ny"], case["nz"])
        self.nt, self.ntstep, self.it0 = _times(case)
        nx, ny, nz = self.shape
        b, d = self.blen, case.get("stride", 4)
        self.rcv_geom = (0, 0, 0, d, d, -(-(nx - 2 * b) // d), -(-(ny - 2 * b) // d))
        self.src = (nx // 2, ny // 2, b + 2)
        self.every = case.get("every", 0)
        self.V = _velocity(self.shape, b, gen)
        self.coefs = _coefs(self.order)
        self.ricker, self.g = _tables(b, self.nt)
        record = (self.rcv_geom[5], self.rcv_geom[6], self.ntstep)
        back = self.kind != "model"
        self.rcv = torch.randn(record, generator=gen, device="cuda") if back else \
            torch.zeros(record, device="cuda")
        self.R = self.img = self.upb = self.snaps = None
        self.S = [_wave(self.shape, self.order, gen, self.wave)]
        self.S.append(self.S[0].clone())
        if self.kind not in ("model", "hbc_forward"):
            self.R = [_wave(self.shape, self.order, gen, self.wave)]
            self.R.append(self.R[0].clone())
            self.img = torch.zeros(self.shape, device="cuda")
        if self.kind.startswith("hbc") or self.kind == "batch":
            layers = self.nt if self.kind == "batch" else self.ntstep
            self.upb = torch.zeros((layers, nx, ny, self.order // 2), device="cuda",
                                   dtype=WAVES[self.wave])
            if self.kind == "hbc_backward":
                for l in range(layers):
                    self.upb[l] = self.S[0][:, :, b - self.order // 2:b] * (1.0 - 0.01 * l)
        if self.kind == "freq":
            inner = tuple(n - 2 * b for n in self.shape)
            nw = case["nw"]
            self.nw = nw
            # angular frequencies from 2 Hz on, times at the shot's steps
            w = 2.0 * math.pi * (2.0 + 2.0 * np.arange(nw)) * COURANT * SPACING / VMAX
            ph = w[:, None] * np.arange(self.nt)[None, :]
            self.kre = torch.from_numpy(np.cos(ph).astype(np.float32)).cuda()
            self.kim = torch.from_numpy(np.sin(ph).astype(np.float32)).cuda()
            self.w2 = torch.from_numpy((w * w).astype(np.float32)).cuda()
            self.acc = [_noise(inner, gen)[None].repeat(nw, 1, 1, 1) for _ in range(4)]
        if self.kind == "snap":
            nsnap = (self.nt - 1) // self.every + 1
            self.snaps = torch.zeros((nsnap, nx, ny, nz - 2 * b), device="cuda",
                                     dtype=torch.float16)


def _window(case, i):
    """Extended grid of shot i of a batch: sides in steps of 32."""
    r = random.Random(case["mix"] * 1000 + i)
    n = r.randrange(case["lo"], case["hi"] + 1, 32)
    z = r.randrange(case["zlo"], case["zhi"] + 1, 32)
    return tuple(v + 2 * case["blen"] for v in (n, n, z))


def _borrow(t):
    """The library's view of a tensor (it borrows device pointers)."""
    d = hip.DeviceArray.__new__(hip.DeviceArray)
    d.shape, d.base = tuple(t.shape), t
    d.dtype = np.dtype({4: np.float32, 2: np.uint16, 1: np.uint8}[t.element_size()])
    d.nbytes = t.numel() * t.element_size()
    d.ptr = ctypes.c_void_p(t.data_ptr())
    return d


def _pair(ts):
    f = hip.FieldPair.__new__(hip.FieldPair)
    f.a, f.b = _borrow(ts[0]), _borrow(ts[1])
    f.p, f.pp = ctypes.c_void_p(f.a.ptr.value), ctypes.c_void_p(f.b.ptr.value)
    return f


class State:
    """What a program holds for one case; library objects end with it."""

    def __init__(self):
        self.close = []

    def __del__(self):
        for f in self.close:
            f()


def _handles(s):
    """The library's arguments for a shot."""
    h = State()
    h.shot = hip.make_shot(*s.shape, s.blen, s.order, s.nt, s.ntstep, s.src,
                           hip.RcvGeom(*s.rcv_geom), s.wave)
    h.V, h.ricker, h.g, h.rcv = (_borrow(t) for t in (s.V, s.ricker, s.g, s.rcv))
    h.S = _pair(s.S)
    h.R = _pair(s.R) if s.R else None
    h.img = _borrow(s.img) if s.img is not None else None
    h.upb = _borrow(s.upb) if s.upb is not None else None
    h.snaps = _borrow(s.snaps) if s.snaps is not None else None
    h.inputs = s
    return h


def _glorot(seed):
    """Weights of the snapshot autoencoder (its four layers, flat)."""
    rng = np.random.default_rng(seed)
    out = []
    for k, n in ((8, 8), (512, 32), (32, 512), (8, 8)):
        lim = math.sqrt(6.0 / (k + n))
        out += [rng.uniform(-lim, lim, k * n), 0.05 * rng.standard_normal(n)]
    return np.concatenate(out).astype(np.float32)


def _brick_index():
    """Cell (x*32 + y)*32 + z of every element of a brick, in brick order."""
    e = np.arange(32768)
    l, m, a = e & 7, (e >> 3) & 63, e >> 9
    x = 8 * (a >> 4) + 2 * (m >> 4) + (l >> 2)
    y = 8 * ((a >> 2) & 3) + 2 * ((m >> 2) & 3) + ((l >> 1) & 1)
    z = 8 * (a & 3) + 2 * (m & 3) + (l & 1)
    return torch.from_numpy((x * 32 + y) * 32 + z).cuda()


def _train_pool(case, seed):
    gen = torch.Generator("cuda").manual_seed(seed)
    n = case["bricks"]
    coarse = torch.randn((n, 1, 9, 9, 9), generator=gen, device="cuda")
    cells = F.interpolate(coarse, size=(32, 32, 32), mode="trilinear", align_corners=True)
    cells = cells.reshape(n, -1)
    cells = cells / cells.abs().amax(1, keepdim=True)
    return cells[:, _brick_index()].to(torch.float16).contiguous()


def prepare(case, seed):
    hip.init(0)
    kind = case["kind"]
    if kind == "train":
        st = State()
        st.pool = _borrow(_train_pool(case, seed))
        st.codec = ae.Codec(max_bricks=case["bricks"], seed=1)
        st.codec.set_params(_glorot(seed))
        st.close.append(st.codec.destroy)
    elif kind == "codes":
        st = State()
        gen = torch.Generator("cuda").manual_seed(seed)
        shape = (case["nx"], case["ny"], case["nz"])
        st.field = _borrow(_wave(shape, 8, gen, "f32"))
        st.region = ae.region_of(shape, case["blen"])
        n = st.n = ae.region_bricks(st.region)
        dev = dict(device="cuda")
        st.bricks = _borrow(torch.zeros((n, 32768), dtype=torch.float16, **dev))
        st.scales = _borrow(torch.zeros(n, **dev))
        st.codes = _borrow(torch.zeros((n, 2048), dtype=torch.float16, **dev))
        st.out = _borrow(torch.zeros(shape, **dev))
        st.codec = ae.Codec(max_bricks=256, seed=1)
        st.codec.set_params(_glorot(seed))
        st.close.append(st.codec.destroy)
    elif kind == "batch":
        st = State()
        st.shots = [_handles(Shot(case, seed * 100 + i, _window(case, i)))
                    for i in range(case["shots"])]
        torch.cuda.synchronize()
        st.batch = hip.Batch([vars(h) for h in st.shots], st.shots[0].inputs.coefs, st.shots[0].g)
        st.close.append(st.batch.destroy)
    else:
        st = _handles(Shot(case, seed))
        if kind == "freq":
            s = st.inputs
            st.tab = [_borrow(t) for t in (s.kre, s.kim, s.w2)]
            st.acc = [_borrow(t) for t in s.acc]
        if kind == "snap_dct":
            st.dct = hip.DctSnapshots(st.shot, case["every"])
            st.close.append(st.dct.free)
    st.case = dict(case)
    torch.cuda.synchronize()  # the library works on a stream of its own
    return st


# ------------------------------------------------------------------ the call
def _fields(h, *names):
    out = {}
    for n in names:
        f = getattr(h, n)
        out[n] = [f.P.base, f.PP.base]
    return out


def run(st):
    case = st.case
    kind, n = case["kind"], case.get("steps", 0)
    if kind == "train":
        losses = st.codec.train(st.pool, case["bricks"], case["iters"], batch=case["bricks"],
                                lr=1e-3, seed=7)
        return {"losses": losses, "params": st.codec.params()}
    if kind == "codes":
        ae.cut_bricks(st.field, st.region, st.bricks, st.scales)
        st.codec.encode(st.bricks, st.n, st.codes)
        st.codec.decode(st.codes, st.scales, st.n, st.out, st.region)
        return {"bricks": st.bricks.base, "scales": st.scales.base, "codes": st.codes.base,
                "field": st.out.base}
    if kind == "batch":
        it0 = st.shots[0].inputs.it0
        st.batch.forward_steps(it0, n)
        st.batch.backward_steps(it0 + n - 1, n)
        return [dict(_fields(h, "S", "R"), img=h.img.base) for h in st.shots]
    s = st.inputs
    it0, hi = s.it0, s.it0 + n - 1
    head = (st.shot, st.V, s.coefs, st.g)
    if kind == "model":
        hip.model_steps(*head, st.ricker, st.S, st.rcv, it0, n)
        return dict(_fields(st, "S"), rcv=s.rcv)
    if kind == "freq":
        kre, kim, w2 = st.tab
        hip.freq_steps(*head, st.ricker, st.S, st.R, st.rcv, st.img, st.acc, kre, kim, w2, s.nw,
                       0, s.nw, hi, n)
        return dict(_fields(st, "S", "R"), img=s.img, acc=s.acc)
    if kind == "snap":
        hip.snap_forward_steps(*head, st.ricker, st.S, st.snaps, "f16", s.every, it0, n)
        hip.snap_backward_steps(*head, st.R, st.snaps, "f16", s.every, st.rcv, st.img, hi, n)
        return dict(_fields(st, "S", "R"), img=s.img, snaps=s.snaps)
    if kind == "snap_dct":
        st.dct.forward_steps(*head[1:], st.ricker, st.S, it0, n)
        st.dct.backward_steps(*head[1:], st.R, st.rcv, st.img, hi, n)
        return dict(_fields(st, "S", "R"), img=s.img)
    hbc = 0 if kind == "rbc" else 2
    out = {}
    if kind != "hbc_backward":
        hip.forward_steps(st.shot, hbc, *head[1:], st.ricker, st.S, st.upb, it0, n)
        out = _fields(st, "S")
    if kind != "hbc_forward":
        hip.backward_steps(st.shot, hbc, *head[1:], st.S, st.R, st.upb, st.rcv, st.img, hi, n)
        out = dict(_fields(st, "S", "R"), img=s.img)
    if kind != "rbc" and kind != "hbc_backward":
        out["upb"] = s.upb
    return out


# ------------------------------------------- what a pass cannot do without
def work(case):
    """Per time step of a field: P, PP and V read, PP written, the taps of
    every cell; per imaging step: both fields' values at hand in the step that
    makes one of them, the other read, the image read and written."""
    kind = case["kind"]
    if kind == "train":
        rows = case["bricks"]
        flops = 2.0 * rows * (2 * 4096 * 64 + 2 * 64 * 512 * 32) * 3 - 2.0 * rows * 4096 * 64
        return {"bytes": float(case["iters"] * rows * 65536),
                "flops": float(case["iters"] * flops)}
    if kind == "codes":
        cells = case["nx"] * case["ny"] * (case["nz"] - 2 * case["blen"])
        bricks = ae.region_bricks(ae.region_of((case["nx"], case["ny"], case["nz"]),
                                               case["blen"]))
        # the field read and written, bricks written and read, codes likewise
        return {"bytes": float(8 * cells + bricks * (2 * 65536 + 2 * 4096)),
                "flops": 2.0 * bricks * (2 * 4096 * 64 + 2 * 64 * 512 * 32)}
    if kind == "batch":
        parts = [work(dict(case, kind="hbc", nx=w[0], ny=w[1], nz=w[2]))
                 for w in (_window(case, i) for i in range(case["shots"]))]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    n, r = case["steps"], case.get("order", 8) // 2
    w = 4 if case["wave"] == "f32" else 2
    b = case["blen"]
    cells = float((case["nx"] - 2 * r) * (case["ny"] - 2 * r) * (case["nz"] - 2 * r))
    image = float(case["nx"] * case["ny"] * (case["nz"] - 2 * b))
    step, tap = 3 * w + 4, 3 * (4 * r + 2) + 6
    both = kind in ("hbc", "rbc", "snap", "snap_dct", "freq")
    fields = {"model": 1, "hbc_forward": 1, "hbc_backward": 2, "hbc": 3, "rbc": 3, "snap": 2,
              "snap_dct": 2, "freq": 2}[kind]
    total, flops = n * fields * step * cells, n * fields * tap * cells
    if kind in ("hbc", "rbc", "hbc_backward"):
        total += n * (w + 8) * image
        flops += n * 2 * image
    if kind.startswith("hbc"):
        total += n * (2 if both else 1) * w * r * case["nx"] * case["ny"]
    if kind in ("snap", "snap_dct"):
        imaged = n // case["every"]
        # the snapshot stored and read: FP16 cells, or a 32nd of them as words
        kept = 2 * 2 if kind == "snap" else 2 * 4 / 32
        total += imaged * (kept + w * (kind == "snap_dct") + 8) * image
        flops += imaged * 3 * image
    if kind == "freq":
        inner = float((case["nx"] - 2 * b) * (case["ny"] - 2 * b) * (case["nz"] - 2 * b))
        total += n * inner * (32 * case["nw"] + 8)
        flops += n * inner * 12 * case["nw"]
    return {"bytes": total, "flops": flops}


# ------------------------------------------------------- the result in 64 bits
class Exact:
    """The propagation's operators on float64 tensors [x][y][z]."""

    def __init__(self, s):
        self.s, self.r, self.b = s, s.order // 2, s.blen
        self.c = [[float(v) for v in row] for row in s.coefs]
        self.V = s.V.double()
        self.g = s.g.double()
        self.ricker, self.rcv = s.ricker.double(), s.rcv.double()
        dev = dict(device="cuda", dtype=torch.float64)
        b, (nx, ny, nz) = self.b, s.shape
        self.lat = []
        for n in s.shape:
            f = torch.ones(n, **dev)
            f[:b], f[n - b:] = self.g.flip(0), self.g
            self.lat.append(f)
        sx, sy, dz, dx, dy, cx, cy = s.rcv_geom
        self.rx = slice(b + sx, b + sx + (cx - 1) * dx + 1, dx)
        self.ry = slice(b + sy, b + sy + (cy - 1) * dy + 1, dy)
        self.rz = b + dz

    def step(self, P, PP):
        r = self.r
        inner = tuple(slice(r, n - r) for n in P.shape)
        lap = torch.zeros_like(P[inner])
        for d in range(3):
            for k in range(2 * r + 1):
                at = list(inner)
                at[d] = slice(k, P.shape[d] - 2 * r + k)
                lap.add_(P[tuple(at)], alpha=self.c[d][k])
        lap.mul_(self.V[inner])
        PP[inner] = lap.add_(P[inner], alpha=2.0).sub_(PP[inner])

    def upper(self, *fields):
        b = self.b
        for f in fields:
            v = f[:, :, :b]
            v.mul_(self.lat[0][:, None, None]).mul_(self.lat[1][None, :, None])
            v.mul_(self.lat[2][:b])

    def all(self, *fields):
        """Every border; the edge at small x and large y takes the value of
        its neighbour at x = b (between the z borders)."""
        b = self.b
        for f in fields:
            f.mul_(self.lat[0][:, None, None]).mul_(self.lat[1][None, :, None])
            f.mul_(self.lat[2])
            ny, nz = f.shape[1:]
            edge = f[b, ny - b:, b:nz - b]  # carries its y factor already
            f[:b, ny - b:, b:nz - b] = edge[None] * self.lat[0][:b, None, None] * \
                self.lat[1][None, ny - b:, None]

    def source(self, PP, it):
        PP[self.s.src] += self.ricker[it]

    def inject(self, PP, it):
        PP[self.rx, self.ry, self.rz] = self.rcv[:, :, it % self.s.ntstep]

    def image(self, img, PS, PR, weight=1.0):
        z = slice(self.b, self.s.shape[2] - self.b)
        img[:, :, z] += weight * (PS[:, :, z] * PR[:, :, z])


def _exact_forward(e, S, upb=None, store=None, it0=0, n=0):
    s, b, hf = e.s, e.b, e.r
    P, PP = S
    for it in range(it0, it0 + n):
        P, PP = PP, P
        if s.kind != "rbc":
            e.upper(P, PP)
        e.step(P, PP)
        e.source(PP, it)
        if upb is not None:
            upb[it % upb.shape[0]] = PP[:, :, b - hf:b]
        if store is not None and (s.nt - 1 - it) % s.every == 0:
            store((s.nt - 1 - it) // s.every, PP)
    return [P, PP]


def _exact_backward(e, S, R, img, upb=None, load=None, hi=0, n=0):
    s, b, hf = e.s, e.b, e.r
    Pr, PPr = R
    for it in range(hi, hi - n, -1):
        if load is None:
            Ps, PPs = S
            e.step(Ps, PPs)
            if upb is not None:
                PPs[:, :, b - hf:b] = upb[it % upb.shape[0]]
            S = [PPs, Ps]
        if s.kind != "rbc":
            e.upper(Pr, PPr)
        e.step(Pr, PPr)
        e.inject(PPr, it)
        if load is None:
            e.image(img, S[0], PPr)
        elif (s.nt - 1 - it) % s.every == 0:
            load((s.nt - 1 - it) // s.every, PPr, img)
        Pr, PPr = PPr, Pr
    return S, [Pr, PPr]


def _dct(n):
    k = torch.arange(n, device="cuda", dtype=torch.float64)
    m = torch.cos(math.pi * (2 * k[None, :] + 1) * k[:, None] / (2 * n)) * math.sqrt(2.0 / n)
    m[0] /= math.sqrt(2.0)
    return m


class ExactCoder:
    """Transform-coded snapshots: the largest coefficients of 8 x 8 x 32
    bricks, one power-of-two threshold, FP16 values over the brick's scale."""

    def __init__(self, s):
        nx, ny, nz = s.shape
        self.b, self.shape, self.kept = s.blen, s.shape, {}
        self.n = (-(-nx // 8), -(-ny // 8), -(-nz // 32))
        self.budget = max(1, nx * ny * (nz - 2 * s.blen) // 32)
        self.every = s.every

    def _bricks(self, f):
        (bx, by, bz), (nx, ny, nz) = self.n, self.shape
        p = torch.zeros((8 * bx, 8 * by, 32 * bz), device="cuda", dtype=torch.float64)
        p[:nx, :ny, self.b:nz - self.b] = f[:, :, self.b:nz - self.b]
        return p.view(bx, 8, by, 8, bz, 32)

    def store(self, j, f):
        t = self._bricks(f)
        t = torch.einsum("wk,aibjck->aibjcw", _dct(32), t)
        t = torch.einsum("vj,aibjcw->aibvcw", _dct(8), t)
        t = torch.einsum("ui,aibvcw->aubvcw", _dct(8), t)
        mag = t.abs()
        exponent = torch.frexp(mag).exponent[mag > 2.0 ** -126].long()
        counts = torch.bincount(exponent + 200, minlength=400)
        above = torch.flip(torch.cumsum(torch.flip(counts, [0]), 0), [0])
        lowest = int((above <= self.budget).nonzero()[0]) - 200
        scale = mag.amax((1, 3, 5), keepdim=True)
        kept = torch.where(mag >= 2.0 ** (lowest - 1), t / scale.clamp(min=1e-300), 0.0)
        self.kept[j] = kept.to(torch.float16).double() * scale

    def load(self, j, PR, img):
        t = torch.einsum("ui,aubvcw->aibvcw", _dct(8), self.kept[j])
        t = torch.einsum("vj,aibvcw->aibjcw", _dct(8), t)
        t = torch.einsum("wk,aibjcw->aibjck", _dct(32), t)
        nx, ny, nz = self.shape
        v = t.reshape(8 * self.n[0], 8 * self.n[1], 32 * self.n[2])[:nx, :ny]
        z = slice(self.b, nz - self.b)
        img[:, :, z] += self.every * (v[:, :, z] * PR[:, :, z])


def _exact_shot(s, kind):
    """Outputs of run() for a shot's inputs."""
    e, n, it0 = Exact(s), s.steps, s.it0
    hi = it0 + n - 1
    S = [t.double() for t in s.S]
    R = [t.double() for t in s.R] if s.R else None
    img = s.img.double() if s.img is not None else None
    upb = s.upb.double() if s.upb is not None else None
    if kind == "model":
        P, PP = S
        rcv = s.rcv.double()
        for it in range(it0, it0 + n):
            P, PP = PP, P
            e.all(P, PP)
            e.step(P, PP)
            e.source(PP, it)
            rcv[:, :, it % s.ntstep] = PP[e.rx, e.ry, e.rz]
        return {"S": [P, PP], "rcv": rcv}
    if kind == "freq":
        b = s.blen
        inner = tuple(slice(b, v - b) for v in s.shape)
        acc = [t.double() for t in s.acc]
        kre, kim, w2 = (t.double() for t in (s.kre, s.kim, s.w2))
        (Ps, PPs), (Pr, PPr) = S, R
        for it in range(hi, hi - n, -1):
            st = s.nt - 1 - it
            e.step(Ps, PPs)
            e.step(Pr, PPr)
            e.all(Ps, PPs, Pr, PPr)
            e.source(PPs, st)
            e.inject(PPr, it)
            for w in range(s.nw):
                for a, k, f in zip(acc, (kre, kim, kre, kim), (PPs, PPs, PPr, PPr)):
                    a[w] += k[w, st] * f[inner]
                img[inner] += w2[w] * (acc[0][w] * acc[2][w] - acc[1][w] * acc[3][w])
            Ps, PPs, Pr, PPr = PPs, Ps, PPr, Pr
        return {"S": [Ps, PPs], "R": [Pr, PPr], "img": img, "acc": acc}
    if kind in ("snap", "snap_dct"):
        snaps = s.snaps.double() if kind == "snap" else None
        if kind == "snap":
            z = slice(s.blen, s.shape[2] - s.blen)

            def store(j, f):
                snaps[j] = f[:, :, z]

            def load(j, PR, img):
                img[:, :, z] += s.every * (snaps[j] * PR[:, :, z])
        else:
            coder = ExactCoder(s)
            store, load = coder.store, coder.load
        S = _exact_forward(e, S, store=store, it0=it0, n=n)
        _, R = _exact_backward(e, None, R, img, load=load, hi=hi, n=n)
        out = {"S": S, "R": R, "img": img}
        if kind == "snap":
            out["snaps"] = snaps
        return out
    out = {}
    if kind != "hbc_backward":
        S = _exact_forward(e, S, upb, it0=it0, n=n)
        out = {"S": S}
    if kind != "hbc_forward":
        S, R = _exact_backward(e, S, R, img, upb, hi=hi, n=n)
        out = {"S": S, "R": R, "img": img}
    if kind not in ("rbc", "hbc_backward", "batch"):
        out["upb"] = upb
    return out


def _layers(params):
    p, out, o = torch.from_numpy(params).cuda().double(), [], 0
    for k, n in ((8, 8), (512, 32), (32, 512), (8, 8)):
        out += [p[o:o + k * n].view(k, n), p[o + k * n:o + k * n + n]]
        o += k * n + n
    return out


def _encode(x, w):
    h = torch.tanh(x.reshape(-1, 8) @ w[0] + w[1])
    return h.reshape(-1, 512) @ w[2] + w[3]


def _decode(z, w):
    h = torch.tanh(z.reshape(-1, 32) @ w[4] + w[5])
    return h.reshape(-1, 8) @ w[6] + w[7]


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        x = _train_pool(case, seed).double()
        w = [t.clone().requires_grad_(True) for t in _layers(_glorot(seed))]
        m, v = [torch.zeros_like(t) for t in w], [torch.zeros_like(t) for t in w]
        losses = []
        for it in range(1, case["iters"] + 1):
            sq = (_decode(_encode(x, w), w).reshape(x.shape) - x).square().sum()
            grads = torch.autograd.grad(0.5 * sq, w)
            losses.append(float(sq.detach()) / x.numel())
            rate = 1e-3 * math.sqrt(1.0 - 0.999 ** it) / (1.0 - 0.9 ** it)
            with torch.no_grad():
                for p, g, mi, vi in zip(w, grads, m, v):
                    mi.mul_(0.9).add_(g, alpha=0.1)
                    vi.mul_(0.999).addcmul_(g, g, value=0.001)
                    p.sub_(rate * mi / (vi.sqrt() + 1e-8))
        return {"losses": np.array(losses),
                "params": torch.cat([t.detach().reshape(-1) for t in w])}
    if kind == "codes":
        gen = torch.Generator("cuda").manual_seed(seed)
        shape, b = (case["nx"], case["ny"], case["nz"]), case["blen"]
        f = _wave(shape, 8, gen, "f32").double()[:, :, b:shape[2] - b]
        nb = [-(-n // 32) for n in f.shape]
        cells = torch.zeros([32 * n for n in nb], device="cuda", dtype=torch.float64)
        cells[:f.shape[0], :f.shape[1], :f.shape[2]] = f
        cells = cells.view(nb[0], 32, nb[1], 32, nb[2], 32).permute(0, 2, 4, 1, 3, 5)
        cells = cells.reshape(-1, 32768)
        scales = cells.abs().amax(1)
        index, w = _brick_index(), _layers(_glorot(seed))
        bricks = (cells / scales.clamp(min=1e-300)[:, None])[:, index]
        codes = _encode(bricks, w).reshape(-1, 2048)
        back = torch.empty_like(cells)
        back[:, index] = _decode(codes, w).reshape(-1, 32768) * scales[:, None]
        back = back.view(*nb, 32, 32, 32).permute(0, 3, 1, 4, 2, 5)
        back = back.reshape([32 * n for n in nb])
        out = torch.zeros(shape, device="cuda", dtype=torch.float64)
        out[:, :, b:shape[2] - b] = back[:f.shape[0], :f.shape[1], :f.shape[2]]
        return {"bricks": bricks, "scales": scales, "codes": codes, "field": out}
    if kind == "batch":
        return [_exact_shot(Shot(case, seed * 100 + i, _window(case, i)), "batch")
                for i in range(case["shots"])]
    return _exact_shot(Shot(case, seed), kind)
