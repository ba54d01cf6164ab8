"""The work that users of this library have it do, as timed cases.

A case is one pass of a user's inner loop through the public entry points:
lattice-Boltzmann steps on a sphere pack (single `lbstep` calls, runs, solves
to a residual), moment propagation of a tracer, a batch of resistance
problems, and the warm-start network (a training gradient, a warm start).
Flow fields come back as the 10 moments per node that `slb_warm_moments`
writes on the device.  `exact` restates each path in 64-bit torch.
"""
import ctypes as C
import math
import os

import numpy as np
import torch

import sunlightlb_amd as slb

DEV = "cuda"
RHO0 = 72.0  # the default


def listed():
    return [
        # the smallest calls: a reference driver's loop of single steps and a
        # measurement on the sphere-in-a-box example, where launches and host
        # work count
        dict(name="sphere32-lbstep-f64", kind="lb", i=32, j=32, k=32, prec=64, steps=20, single=True,
             radius=4.5, phi=0.0, moving=False, skip=True, stokes=False, measure=True),
        # the mobility example: a moving sphere in a small non-cubic box
        dict(name="mobility48-run-f64", kind="lb", i=48, j=32, k=32, prec=64, steps=100, single=False,
             radius=5.1, phi=0.0, moving=True, skip=False, stokes=True, measure=True),
        # odd edges, Navier-Stokes, double precision: a scanned sample's cut-out
        dict(name="ragged-run-f64", kind="lb", i=131, j=97, k=75, prec=64, steps=40, single=False,
             radius=6.0, phi=0.3, moving=False, skip=False, stokes=False, measure=False),
        # an ordinary solve to a residual with its checks: one pack of a training set
        dict(name="solve128-f32", kind="solve", i=128, j=128, k=128, prec=32, radius=6.0, phi=0.25,
             tol=2e-3, interval=100, most=1200),
        # permeability packs in single precision: the benchmark's, the largest
        dict(name="pack256-run-f32", kind="lb", i=256, j=256, k=256, prec=32, steps=50, single=False,
             radius=8.0, phi=0.35, moving=False, skip=False, stokes=True, measure=False),
        dict(name="pack512-run-f32", kind="lb", i=512, j=512, k=512, prec=32, steps=8, single=False,
             radius=16.0, phi=0.35, moving=False, skip=False, stokes=True, measure=False),
        # passive scalar: a long run with displacement moments and partial
        # adsorption; the reference driver's loop of single steps
        dict(name="tracer128-run-f32", kind="mp", i=128, j=128, k=128, prec=32, steps=400, single=False,
             radius=6.0, phi=0.25, moments=True, pads=0.01),
        dict(name="tracer-ragged-mpstep-f64", kind="mp", i=53, j=41, k=67, prec=64, steps=60, single=True,
             radius=5.0, phi=0.25, moments=False, pads=0.0),
        # resistance problems: boxes of U{32..64}, 6 right-hand sides each
        dict(name="batch32x6-f32", kind="batch", boxes=32, lo=32, hi=64, prec=32, steps=64),
        # the warm-start network: the gradient of one training sample (the
        # training set's size, and a box that is no power of two), and a warm
        # start of a solve (features, forward pass, injection)
        dict(name="net128-gradient", kind="grad", i=128, j=128, k=128),
        dict(name="net-ragged-gradient", kind="grad", i=96, j=80, k=72),
        dict(name="net64-warmstart-f32", kind="warm", i=64, j=80, k=96, prec=32, radius=5.0, phi=0.3),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _edges(rng, lo, hi, unit=1):
    """Three edges about one size of [lo, hi], one time in three with a row of a power of two."""
    e = _log(rng, lo, hi)
    d = [max(lo, min(hi, int(round(e * rng.uniform(0.75, 1.3) / unit)) * unit)) for _ in range(3)]
    if unit == 1 and rng.random() < 0.33:
        d[2] = min((64, 128, 256), key=lambda q: abs(q - d[2]))
    return d


def draw(rng):
    what = rng.choice(["lb", "lb", "lb", "lb", "solve", "mp", "mp", "batch", "grad", "warm"])
    if what == "lb":
        i, j, k = _edges(rng, 16, 320)
        prec = rng.choice([32, 32, 64])
        single = rng.random() < 0.25
        moving = i * j * k < 250000 and min(i, j, k) >= 24 and rng.random() < 0.4
        # at most the work of the largest listed case
        most = int(512 ** 3 * 8 / (i * j * k) * 32 / prec)
        return dict(kind="lb", i=i, j=j, k=k, prec=prec, steps=max(1, min(most, rng.randint(5, 60))), single=single,
                    radius=round(rng.uniform(3.5, 5.5) if moving else rng.uniform(3.5, 9.0), 2),
                    phi=0.0 if moving else round(rng.uniform(0.1, 0.4), 2), moving=moving,
                    skip=rng.random() < 0.2, stokes=rng.random() < 0.6, measure=moving or rng.random() < 0.3)
    if what == "solve":
        i, j, k = _edges(rng, 40, 120)
        return dict(kind="solve", i=i, j=j, k=k, prec=rng.choice([32, 64]), radius=round(rng.uniform(4, 6), 2),
                    phi=round(rng.uniform(0.25, 0.4), 2), tol=2e-3, interval=100, most=600)
    if what == "mp":
        i, j, k = _edges(rng, 24, 140)
        single = rng.random() < 0.4
        return dict(kind="mp", i=i, j=j, k=k, prec=rng.choice([32, 64]), steps=rng.randint(20, 60) if single else rng.randint(33, 300),
                    single=single, radius=round(rng.uniform(4, 7), 2), phi=round(rng.uniform(0.15, 0.35), 2),
                    moments=rng.random() < 0.6, pads=rng.choice([0.0, 0.01, 0.2]))
    if what == "batch":
        return dict(kind="batch", boxes=rng.randint(4, 28), lo=rng.randint(28, 36), hi=rng.randint(48, 64),
                    prec=rng.choice([32, 32, 64]), steps=rng.randint(20, 70))
    i, j, k = _edges(rng, 24, 128, 8)
    if what == "grad":
        return dict(kind="grad", i=i, j=j, k=k)
    return dict(kind="warm", i=i, j=j, k=k, prec=rng.choice([32, 64]), radius=round(rng.uniform(4, 7), 2),
                phi=round(rng.uniform(0.2, 0.4), 2))


# ---------------------------------------------------------------- geometry

def _mark(solid, rad, centres):
    """Set the nodes nearer than rad to a centre (periodic) in the device map."""
    ei, ej, ek = solid.shape
    m = int(rad) + 2
    o = torch.arange(-m, m + 1, device=DEV)
    g = torch.stack(torch.meshgrid(o, o, o, indexing="ij"), -1).reshape(1, -1, 3)
    for part in torch.as_tensor(centres, dtype=torch.float64, device=DEV).split(max(1, 20_000_000 // g.shape[1])):
        base = part.floor().long()[:, None, :]
        d = (base + g) - part[:, None, :]
        near = (d * d).sum(-1) < rad * rad
        n = (base + g)[near]
        solid[n[:, 0] % ei, n[:, 1] % ej, n[:, 2] % ek] = True


def _pack(case, seed):
    """Spheres at random (overlap allowed) to about the solid fraction phi; one central sphere for phi = 0."""
    dims = (case["i"], case["j"], case["k"])
    solid = torch.zeros(dims, dtype=torch.bool, device=DEV)
    rs = np.random.RandomState(seed % (1 << 31))
    if case["phi"] > 0:
        vol = 4 / 3 * math.pi * case["radius"] ** 3
        n = max(1, round(-math.log(1 - case["phi"]) * dims[0] * dims[1] * dims[2] / vol))
        centres = rs.rand(n, 3) * dims
    else:
        centres = [[d / 2 + rs.uniform(-0.5, 0.5) for d in dims]]
    _mark(solid, case["radius"], centres)
    return solid, np.asarray(centres)


def _force(case, seed):
    rs = np.random.RandomState((seed + 77) % (1 << 31))
    return [round(1e-3 * rs.uniform(0.5, 1.5), 9), round(1e-4 * rs.uniform(-1, 1), 10), 0.0]


class Handle:
    """A lattice (or a batch) that is released with the last reference to it."""

    def __init__(self, h, free):
        self.h, self.free = h, free

    def __del__(self):
        self.free(self.h)


def _lattice(case, solid, bf, tau=0.75, stokes=True, skip=False):
    L = slb.lib()
    os.environ["SLB_PRECISION"] = str(case.get("prec", 32))
    h = L.newlb(*solid.shape, b"null")
    s = h.contents
    s.tau, s.stokes_flow, s.skip_solid = tau, int(stokes), int(skip)
    s.objects_moving, s.vel_corrected = 0, 1
    s.dpdx, s.dpdy, s.dpdz = bf
    m = solid.to(torch.uint8).cpu().numpy().reshape(-1)
    L.slb_insert_map(h, m.ctypes.data_as(C.c_void_p))
    L.syncobjs(h)
    return Handle(h, L.slb_destroy)


def _spheres(rs, e, count):
    """`count` spheres of radius U[3, 6] wholly inside a box of edge e, apart from each other."""
    got, tried = [], 0
    while len(got) < count:
        tried += 1
        if tried % 200 == 0:
            got = []  # no room left: begin again
        r = rs.uniform(3.0, 6.0)
        p = rs.uniform(r + 1.0, e - r - 2.0, 3)
        if all(np.sum((p - q) ** 2) > (r + t + 1.5) ** 2 for t, q in got):
            got.append((r, p))
    return got


def _boxes(case, seed):
    rs = np.random.RandomState(seed % (1 << 31))
    edges = rs.randint(case["lo"], case["hi"] + 1, case["boxes"])
    return [(int(e), _spheres(rs, e, 2 + q % 6)) for q, e in enumerate(edges)]


# 6 right-hand sides: the first sphere translating and rotating about x, y, z
def _velocities(spheres):
    v = np.zeros((6, len(spheres), 6))
    for q in range(6):
        v[q, 0, q] = 1e-3 if q < 3 else 1e-3 / spheres[0][0]
    return v


# ---------------------------------------------------------------- network

LAYERS = [(16, 16, 0), (16, 16, 0), (16, 32, 1), (32, 32, 1), (32, 64, 2), (64, 64, 2), (64, 64, 3), (64, 64, 3),
          (64, 32, 2), (32, 16, 1), (16, 16, 0), (16, 16, 0)]  # channels in and out, level


def _weights(seed):
    """He-scaled weights [co][27 ci] and small biases of every layer."""
    rs = np.random.RandomState((seed + 5) % (1 << 31))
    ws = []
    for q, (ci, co, _) in enumerate(LAYERS):
        sd = (1.0 if q == len(LAYERS) - 1 else math.sqrt(2.0)) / math.sqrt(27.0 * ci)
        ws.append((rs.standard_normal((co, 27 * ci)).astype(np.float32) * np.float32(sd),
                   rs.standard_normal(co).astype(np.float32) * np.float32(0.02)))
    return ws


def _arena(ws):
    """The parameter arena: per layer W[co][27 ci rounded up to 32], then 64 bias slots."""
    parts = []
    for w, b in ws:
        kp = -(-w.shape[1] // 32) * 32
        parts.append(np.pad(w, ((0, 0), (0, kp - w.shape[1]))).reshape(-1))
        parts.append(np.pad(b, (0, 64 - b.size)))
    return np.concatenate(parts).astype(np.float32)


def _net(seed):
    L = slb.lib()
    net = L.slb_warm_new(seed)
    w = _arena(_weights(seed))
    L.slb_warm_set_params(net, w.ctypes.data_as(C.c_void_p))
    return Handle(net, L.slb_warm_free)


def _sample(case, seed):
    """A training sample: the two features and ten targets of every node, in bfloat16, and the loss weights."""
    dims = (case["i"], case["j"], case["k"])
    solid, _ = _pack(dict(case, radius=6.0, phi=0.3), seed)
    g = torch.Generator(device=DEV).manual_seed(seed)
    dist = torch.randn(dims, device=DEV, generator=g).abs() * torch.where(solid, -1.0, 1.0)
    x = torch.zeros((*dims, 16), device=DEV)
    x[..., 0], x[..., 1] = solid.float(), dist
    t = torch.randn((*dims, 10), device=DEV, generator=g) * 0.3 * (~solid)[..., None]
    n = float(solid.numel())
    return x.bfloat16(), t.bfloat16(), np.asarray([1 / (3 * n * c * 0.09) for c in (3, 3, 3, 1, 6, 6, 6, 6, 6, 6)], np.float32)


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    L = slb.lib()
    kind = case["kind"]
    if kind == "grad":
        x, t, wc = _sample(case, seed)
        net = _net(seed)
        return dict(kind=kind, net=net, x=x, t=t, wc=wc, dims=(C.c_int * 3)(case["i"], case["j"], case["k"]),
                    grad=np.zeros(L.slb_warm_nparams(net.h), np.float32))
    if kind == "batch":
        b = Handle(L.slb_batch_new(case["prec"]), L.slb_batch_free)
        objs = []
        for e, spheres in _boxes(case, seed):
            h = L.newlb(e, e, e, b"null")
            s = h.contents
            s.tau, s.stokes_flow, s.objects_moving = 1.0, 1, 1
            for r, p in reversed(spheres):  # the first sphere heads the object list
                L.insertsph(h, r, *p)
            v = np.ascontiguousarray(_velocities(spheres))
            L.slb_batch_add(b.h, h, 6, v.ctypes.data_as(C.POINTER(C.c_double)))
            L.slb_destroy(h)
            objs.append(len(spheres))
        L.slb_batch_commit(b.h)
        return dict(kind=kind, batch=b, objs=objs, steps=case["steps"], dtype=np.float32 if case["prec"] == 32 else np.float64)
    bf = _force(case, seed)
    solid, centres = _pack(case, seed)
    n = solid.numel()
    st = dict(kind=kind, steps=case.get("steps", 0), single=case.get("single", False), prec=case["prec"])
    if kind == "mp":
        # a developed flow, scaled to a mean speed of about 0.05
        lat = _lattice(case, solid, bf)
        L.slb_run(lat.h, 200)
        L.slb_scale_pops(lat.h, 30.0)
        mp = L.newmp(lat.h, b"null")
        L.mpinit(mp)
        L.mpall(mp, 1.0)
        if case["pads"]:
            L.slb_mp_set_adsorption(mp, case["pads"])
        if case["moments"]:
            L.slb_mp_track_moments(mp, 0)
        return dict(st, lat=lat, mp=mp, n=n, sums=(C.c_double * 6)())
    if kind == "warm":
        return dict(st, lat=_lattice(case, solid, bf), net=_net(seed), m=torch.zeros(n, 10, device=DEV))
    if kind == "solve":
        return dict(st, lat=_lattice(case, solid, bf), m=torch.zeros(n, 10, device=DEV), tol=case["tol"],
                    interval=case["interval"], most=case["most"], res=C.c_double(0))
    lat = _lattice(case, solid, bf, 0.75, case["stokes"], case["skip"])
    if case["moving"]:
        lat.h.contents.objects_moving = 1
        o = lat.h.contents.obj_head.contents
        o.posx, o.posy, o.posz = centres[0]
        o.velx, o.vely, o.velz, o.angx, o.angy, o.angz = _motion(seed)
        L.vspread(lat.h)
    return dict(st, lat=lat, m=torch.zeros(n, 10, device=DEV), measure=case["measure"])


def _motion(seed):
    rs = np.random.RandomState((seed + 3) % (1 << 31))
    return [1e-3 * rs.uniform(-1, 1) for _ in range(3)] + [2e-4 * rs.uniform(-1, 1) for _ in range(3)]


# ---------------------------------------------------------------- one pass

def run(st):
    L = slb.lib()
    kind = st["kind"]
    if kind == "grad":
        loss = L.slb_warm_fwd_bwd(st["net"].h, st["dims"], st["x"].data_ptr(), st["t"].data_ptr(),
                                  st["wc"].ctypes.data, None, st["grad"].ctypes.data)
        return dict(loss=np.float32(loss), grad=st["grad"])
    if kind == "batch":
        b = st["batch"].h
        L.slb_batch_run(b, st["steps"])
        L.slb_batch_measure(b)
        out = []
        for q, n in enumerate(st["objs"]):
            for r in range(6):
                f, t = np.zeros((n, 3)), np.zeros((n, 3))
                L.slb_batch_forces(b, q, r, f.ctypes.data_as(slb.RealP), t.ctypes.data_as(slb.RealP))
                out.append(np.concatenate([f, t], 1))
        return np.concatenate(out).astype(st["dtype"])
    h = st["lat"].h
    if kind == "mp":
        mp = st["mp"]
        if st["single"]:
            for _ in range(st["steps"]):
                L.mpstep(mp)
        else:
            L.slb_mp_run(mp, st["steps"])
        L.slb_mp_sums(mp, st["sums"])
        L.slb_mp_sync_host(mp)
        as_ = np.float32 if st["prec"] == 32 else np.float64
        return dict(p=slb.view(mp.contents.p, st["n"]).astype(as_), sums=np.array(st["sums"][:]).astype(as_))
    out = {}
    if kind == "warm":
        L.slb_warm_start(st["net"].h, h)
    elif kind == "solve":
        L.slb_scale_pops(h, 0.0)  # from rest
        L.slb_residual_reset(h)
        out["steps"] = L.slb_run_to_residual(h, st["tol"], st["interval"], st["most"], C.byref(st["res"]))
    else:
        if st["single"]:
            for _ in range(st["steps"]):
                L.lbstep(h)
        else:
            L.slb_run(h, st["steps"])
        if st["measure"]:
            L.measure(h)
            o = h.contents.obj_head.contents
            as_ = np.float32 if st["prec"] == 32 else np.float64
            out["force"] = np.array([o.frcx, o.frcy, o.frcz, o.trqx, o.trqy, o.trqz], as_)
            s = h.contents
            out["vmean"] = np.array([s.vmeanx, s.vmeany, s.vmeanz], as_)
    L.slb_warm_moments(h, C.cast(st["m"].data_ptr(), C.c_void_p), 10, 1.0)
    out["moments"] = st["m"]
    return out


# ---------------------------------------------------------------- work

def work(case):
    kind = case["kind"]
    if kind == "batch":
        edges = [case["lo"] + (case["hi"] - case["lo"]) * (q + 0.5) / case["boxes"] for q in range(case["boxes"])]
        n = 6 * sum(e ** 3 for e in edges)
        return dict(bytes=n * 30 * case["prec"] / 8, flops=170 * n * (case["steps"] + 2))
    n, s = case["i"] * case["j"] * case["k"], case.get("prec", 32) / 8
    if kind in ("grad", "warm"):
        f = sum(54 * ci * co * (n >> (3 * lv)) for ci, co, lv in LAYERS)
        if kind == "grad":
            return dict(bytes=n * 26 * 2, flops=3 * f - 54 * 16 * 16 * n)
        return dict(bytes=n * (2 + 15 * s), flops=f)
    if kind == "mp":
        rec = 3 if case["moments"] else 1
        return dict(bytes=n * (15 + 1 + 2 * rec) * s + 4 * n, flops=n * case["steps"] * 29 * (2 if rec == 1 else 4))
    steps = 3 * case["interval"] if kind == "solve" else case["steps"] + 2 * case["measure"]
    return dict(bytes=n * (30 * s + 2 + 40), flops=170 * n * steps)


# ---------------------------------------------------------------- 64-bit restatement

CV = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 1), (-1, 1, 1), (1, -1, 1),
      (-1, -1, 1), (1, 1, -1), (-1, 1, -1), (1, -1, -1), (-1, -1, -1)]
WL = [16] + [8] * 6 + [1] * 8
OPP = [CV.index((-x, -y, -z)) for x, y, z in CV]


def _pull(f, c):
    """f(x - c) at every x (periodic), over the last three axes."""
    return torch.roll(f, c, (-3, -2, -1)) if any(c) else f


class Flow:
    """D3Q15 in 64 bits: R problems on one solid map, walls moving with U (R, 3, i, j, k) or at rest."""

    def __init__(self, solid, tau, bf, stokes, skip, wall=None, problems=1):
        self.solid, self.om, self.stokes, self.skip, self.wall = solid, 1 / tau, stokes, skip, wall
        self.b = [f * (~solid).double() for f in bf]
        self.bf = bf
        self.a = [torch.zeros((problems, *solid.shape), dtype=torch.float64, device=DEV) for _ in CV]

    def step(self, force=None):
        got = []
        for l, c in enumerate(CV):
            v = _pull(self.a[l], c)
            if l:
                bounce = self.solid ^ _pull(self.solid, c)
                own = self.a[OPP[l]]
                if self.wall is not None:
                    cu = sum(WL[l] * c[d] * self.wall[:, d] for d in range(3))
                    cu = torch.where(self.solid, cu, _pull(cu, c))
                    if force is not None:
                        g = torch.where(bounce & self.solid, -2 * (own - v + cu), 0.0)
                    own = own + cu
                elif force is not None:
                    g = torch.where(bounce & self.solid, -2 * (own - v), 0.0)
                if force is not None:
                    for d in range(3):
                        if c[d]:
                            force[:, d] += c[d] * g
                v = torch.where(bounce, own, v)
            got.append(v)
        d, j, s = self.moments(got)
        j = [x + b for x, b in zip(j, self.b)]
        for q, (x, y) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
            s[q] = s[q] * (1 - self.om)
            if not self.stokes:
                s[q] += self.om * j[x] * j[y] / (RHO0 + d)
        tr = (s[0] + s[1] + s[2]) / 3
        for l, (x, y, z) in enumerate(CV):
            cs = x * x * s[0] + y * y * s[1] + z * z * s[2] + 2 * (x * y * s[3] + x * z * s[4] + y * z * s[5])
            new = WL[l] / 72 * (d + 3 * (x * j[0] + y * j[1] + z * j[2]) + 4.5 * (cs - tr))
            self.a[l] = torch.where(self.solid, got[l], new) if self.skip else new

    @staticmethod
    def moments(a):
        d = sum(a)
        j = [sum(c[q] * v for c, v in zip(CV, a) if c[q]) for q in range(3)]
        s = [sum(c[x] * c[y] * v for c, v in zip(CV, a) if c[x] * c[y]) for x, y in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))]
        return d, j, [v - d / 3 if q < 3 else v for q, v in enumerate(s)]

    def velocity(self):
        d, j, s = self.moments(self.a)
        return [torch.where(self.solid, 0.0, (x - f / 2) / (RHO0 + d)) for x, f in zip(j, self.bf)], d, s

    def mean(self):
        return np.array([float(x.sum()) for x in self.velocity()[0]]) / self.solid.numel()

    def scaled(self, tau):
        """What slb_warm_moments writes for a unit length."""
        u, d, s = self.velocity()
        f, eta = math.sqrt(sum(x * x for x in self.bf)), RHO0 * (tau - 0.5) / 3
        d, s = [torch.where(self.solid, 0.0, x) for x in (d,)][0], [torch.where(self.solid, 0.0, x) for x in s]
        return torch.stack([x[0].reshape(-1) for x in [x * (eta / f) for x in u] + [d * (0.125 / f)] + [x / f for x in s]], 1)


def _grid(dims):
    return torch.meshgrid(*[torch.arange(n, dtype=torch.float64, device=DEV) for n in dims], indexing="ij")


def _rigid(dims, pos, vel):
    """rho0 (v + w x r) / 12 at every node, r from pos."""
    r = [g - p for g, p in zip(_grid(dims), pos)]
    v, w = vel[:3], vel[3:]
    return torch.stack([RHO0 / 12 * (v[0] + w[1] * r[2] - w[2] * r[1]), RHO0 / 12 * (v[1] + w[2] * r[0] - w[0] * r[2]),
                        RHO0 / 12 * (v[2] + w[0] * r[1] - w[1] * r[0])])


def _torque(f, pos):
    """Sum and torque about pos of a node force (3, i, j, k)."""
    r = [g - p for g, p in zip(_grid(f.shape[1:]), pos)]
    t = [r[1] * f[2] - r[2] * f[1], r[2] * f[0] - r[0] * f[2], r[0] * f[1] - r[1] * f[0]]
    return np.array([float(x.sum()) for x in list(f) + t])


def _exact_lb(case, seed):
    solid, centres = _pack(case, seed)
    wall = None
    if case["moving"]:
        wall = (_rigid(solid.shape, centres[0], _motion(seed)) * solid)[None]
    fl = Flow(solid, 0.75, _force(case, seed), case["stokes"], case["skip"], wall)
    for _ in range(case["steps"]):
        fl.step()
    out = {}
    if case["measure"]:
        f = torch.zeros((1, 3, *solid.shape), dtype=torch.float64, device=DEV)
        v = 0.25 * fl.mean()
        fl.step(f)
        v = v + 0.5 * fl.mean()
        fl.step(f)
        v = v + 0.25 * fl.mean()
        if case["moving"]:
            pos = centres[0]
        else:
            pos = [0.0, 0.0, 0.0]  # an inserted map has no centre of its own
        out = dict(force=_torque(f[0] / 2, pos), vmean=v)
    out["moments"] = fl.scaled(0.75)
    return out


def _exact_solve(case, seed):
    solid, _ = _pack(case, seed)
    fl = Flow(solid, 0.75, _force(case, seed), True, False)
    n, before = 0, None
    while n < case["most"]:
        for _ in range(min(case["interval"], case["most"] - n)):
            fl.step()
            n += 1
        u = torch.stack(fl.velocity()[0])
        r = None if before is None else float((u - before).norm() / u.norm())
        before = u
        if r is not None and r < case["tol"]:
            break
    return dict(steps=n, moments=fl.scaled(0.75))


def _exact_mp(case, seed):
    solid, _ = _pack(case, seed)
    fl = Flow(solid, 0.75, _force(case, seed), True, False)
    for _ in range(200):
        fl.step()
    a = [30.0 * x[0] for x in fl.a]
    fluid = (~solid).double()
    rho = torch.where(solid, RHO0, RHO0 + sum(a))
    pi = [a[l] / rho + WL[l] / 72 * RHO0 / rho for l in range(15)]
    link = [_pull(pi[l] * fluid, CV[l]) for l in range(15)]      # from a fluid source
    near = sum(_pull(fluid, CV[l]) for l in range(1, 15)) > 0
    keep = sum((1 - case["pads"]) * pi[OPP[l]] * (1 - _pull(fluid, CV[l])) for l in range(1, 15)) * fluid
    frac = torch.where(solid & near, case["pads"], 0.0)
    q = [fluid.clone()] + ([torch.zeros_like(fluid), torch.zeros_like(fluid)] if case["moments"] else [])
    for _ in range(case["steps"]):
        new = [keep * x for x in q]
        for l, c in enumerate(CV):
            p = [_pull(x, c) for x in q]
            new[0] += link[l] * p[0]
            if case["moments"]:
                new[1] += link[l] * (p[1] + c[0] * p[0])
                new[2] += link[l] * (p[2] + 2 * c[0] * p[1] + c[0] * c[0] * p[0])
        q = [torch.where(solid, x + frac * y, y) for x, y in zip(q, new)]
    sums = [float((q[0] * fluid).sum()), float((q[0] * (1 - fluid)).sum()), 0.0]
    sums += [float((x * fluid).sum()) for x in q[1:]] if case["moments"] else [0.0, 0.0]
    return dict(p=q[0].reshape(-1), sums=np.array(sums + [float(fluid.sum())]))


def _exact_batch(case, seed):
    out = []
    for e, spheres in _boxes(case, seed):
        owner = torch.full((e, e, e), -1, dtype=torch.long, device=DEV)
        for q in range(len(spheres) - 1, -1, -1):
            own = torch.zeros((e, e, e), dtype=torch.bool, device=DEV)
            _mark(own, spheres[q][0], [spheres[q][1]])
            owner[own] = q
        vel = _velocities(spheres)
        wall = torch.stack([sum(_rigid((e, e, e), p, vel[r, q]) * (owner == q) for q, (_, p) in enumerate(spheres)) for r in range(6)])
        fl = Flow(owner >= 0, 1.0, [0.0, 0.0, 0.0], True, False, wall, 6)
        for _ in range(case["steps"]):
            fl.step()
        f = torch.zeros((6, 3, e, e, e), dtype=torch.float64, device=DEV)
        fl.step(f)
        fl.step(f)
        for r in range(6):
            out += [_torque(f[r] / 2 * (owner == q), p) for q, (_, p) in enumerate(spheres)]
    return np.stack(out)


TAPS = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]


def _tap(x, o):
    return torch.roll(x, (-o[0], -o[1], -o[2]), (0, 1, 2)) if any(o) else x


def _conv(x, w):
    y = 0
    for t, o in enumerate(TAPS):
        y = y + _tap(x, o) @ w[:, t * x.shape[-1]:(t + 1) * x.shape[-1]].T
    return y


def _halve(x):
    i, j, k, c = x.shape
    return x.reshape(i // 2, 2, j // 2, 2, k // 2, 2, c).mean((1, 3, 5))


def _double(x):
    for a in range(3):
        x = x.repeat_interleave(2, a)
    return x


def _forward(x, ws):
    """Outputs, and what each layer read and gave, of the network on x (i, j, k, 16)."""
    ins, outs = [], []

    def layer(x):
        q = len(ins)
        y = _conv(x, ws[q][0]) + ws[q][1]
        ins.append(x)
        outs.append(y.relu() if q < 11 else y)
        return outs[-1]

    e1 = layer(layer(x))
    e2 = layer(layer(_halve(e1)))
    e3 = layer(layer(_halve(e2)))
    y = layer(layer(_halve(e3)))
    y = layer(_double(y) + e3)
    y = layer(_double(y) + e2)
    y = layer(_double(y) + e1)
    return layer(y), ins, outs


def _exact_grad(case, seed):
    x, t, wc = _sample(case, seed)
    ws = [[torch.as_tensor(v, device=DEV).double() for v in wb] for wb in _weights(seed)]
    y, ins, outs = _forward(x.double(), ws)
    d = y[..., :10] - t.double()
    wc = torch.as_tensor(wc, device=DEV).double()
    loss = float((wc * d * d).sum())
    gy = torch.zeros_like(y)
    gy[..., :10] = 2 * wc * d
    grads = [None] * 12

    def back(q, g):
        g = g * (outs[q] > 0) if q < 11 else g
        ci = ins[q].shape[-1]
        flat = g.reshape(-1, g.shape[-1])
        gw = torch.cat([flat.T @ _tap(ins[q], o).reshape(-1, ci) for o in TAPS], 1)
        grads[q] = (gw.cpu().numpy(), flat.sum(0).cpu().numpy())
        if q == 0:
            return None
        return sum(_tap(g @ ws[q][0][:, n * ci:(n + 1) * ci], tuple(-v for v in o)) for n, o in enumerate(TAPS))

    def down(g):  # of _double
        return 8 * _halve(g)

    s1 = back(10, back(11, gy))
    s2 = back(9, down(s1))
    s3 = back(8, down(s2))
    g = back(6, back(7, down(s3)))
    g = back(4, back(5, _double(g) / 8 + s3))
    g = back(2, back(3, _double(g) / 8 + s2))
    back(0, back(1, _double(g) / 8 + s1))
    parts = []
    for w, b in grads:
        parts += [np.pad(w, ((0, 0), (0, -w.shape[1] % 32))).reshape(-1), np.pad(b, (0, 64 - b.size))]
    return dict(loss=np.float64(loss), grad=np.concatenate(parts))


def _distance(seeds):
    """Periodic Euclidean distance of every node to the nearest set node."""
    d = torch.where(seeds, 0.0, 1e9).double()
    for a in range(3):
        n = d.shape[a]
        o = torch.arange(n, device=DEV)
        best = d
        for s in range(1, n // 2 + 1):
            best = torch.minimum(best, torch.minimum(d.roll(s, a), d.roll(-s, a)) + s * s)
        d = best
    return d.sqrt()


def _exact_warm(case, seed):
    solid, _ = _pack(case, seed)
    to_solid, to_fluid = _distance(solid), _distance(~solid)
    ell = float(to_solid[~solid].mean())
    x = torch.zeros((*solid.shape, 16), dtype=torch.float64, device=DEV)
    x[..., 0], x[..., 1] = solid.double(), torch.where(solid, -to_fluid, to_solid) / ell
    ws = [[torch.as_tensor(v, device=DEV).double() for v in wb] for wb in _weights(seed)]
    y = _forward(x, ws)[0][..., :10] * (~solid)[..., None]
    y[..., :3] *= ell * ell
    y[..., 3:] *= ell
    return dict(moments=y.reshape(-1, 10))


def exact(case, seed):
    with torch.no_grad():
        return {"lb": _exact_lb, "solve": _exact_solve, "mp": _exact_mp, "batch": _exact_batch, "grad": _exact_grad,
                "warm": _exact_warm}[case["kind"]](case, seed)
