"""Runs with walls at rest take their steps two at a time (k_step2), single
lbstep calls and moving walls do not.
Populations after runs against the same number of lbstep calls, bit for bit
(one function holds the collision of both kernels, so the tolerance is zero),
at the edges of its tiles: k tiles with a remainder and rows of one node,
j and i remainders, planes that are and are not whole population tiles,
lattices of one plane, odd step counts."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def build(dims, prec, moving, stokes, skip, bf):
    import sunlightlb_amd as s
    lat = s.Lattice(*dims, precision=prec)
    L, h = lat.L, lat.h
    lat.s.tau, lat.s.stokes_flow, lat.s.skip_solid, lat.s.objects_moving = 0.7, stokes, skip, moving
    rng = np.random.default_rng(sum(dims))
    for q in range(max(3, lat.N // 4000)):
        sph = L.insertsph(h, float(rng.uniform(0.8, 4.0)), *[float(rng.uniform(-1.0, n)) for n in dims])
        if sph:
            sph.contents.velx, sph.contents.vely = 0.01, -0.004 * (q % 3)
            sph.contents.velz, sph.contents.angz = 0.006, 0.002
    if moving:
        L.vspread(h)
    L.zerobf(h)
    if bf == 2:
        lat.sync()
        solid = lat.solid()
        for nm, sc in (("bx", 2e-4), ("by", 5e-5), ("bz", 1e-4)):
            s.view(getattr(lat.s, nm), lat.N)[:] = np.where(solid, 0.0, sc * (1 + rng.random(lat.N)))
        L.slb_sync_device(h)
    elif bf == 1:
        L.addbf(h, 1e-4, 0.0, 2e-5)
    lat.set_pops(1e-3 * rng.standard_normal(lat.N * 15))
    return lat


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("dims,moving,stokes,skip,bf", [
    ((9, 32, 64), 1, 0, 1, 2),        # whole tiles per plane
    ((7, 16, 256), 0, 1, 0, 1),       # more than one k tile
    ((5, 8, 512), 1, 1, 0, 0),
    ((13, 23, 75), 0, 0, 0, 2),       # remainders in j and k
    ((4, 11, 331), 1, 0, 0, 1),       # k tiles of unequal width
    ((70, 5, 9), 0, 1, 1, 1),         # many planes
    ((1, 1, 7), 1, 0, 0, 1), ((2, 2, 2), 0, 0, 0, 1), ((3, 2, 1), 1, 1, 0, 2), ((2, 1024, 1), 0, 1, 0, 1),
    ((96, 96, 96), 0, 1, 0, 1),       # plain stores (FP32: both buffers fit the cache)
])
def test_run_is_single_steps(prec, dims, moving, stokes, skip, bf):
    print(f"pairs: {dims} prec {prec}", flush=True)
    ref, got = (build(dims, prec, moving, stokes, skip, bf) for _ in range(2))
    for n in (2, 7):
        for _ in range(n):
            ref.L.lbstep(ref.h)
        got.L.slb_run(got.h, n)
        assert np.array_equal(ref.pops(), got.pops())
    assert got.s.step == 9
    ref.free()
    got.free()


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("dims,stokes,skip,bf", [
    ((9, 32, 64), 0, 1, 2), ((9, 32, 64), 1, 0, 2), ((5, 8, 512), 1, 1, 0), ((4, 11, 331), 0, 0, 1),
    ((1, 1, 7), 0, 0, 1), ((1, 40, 50), 0, 1, 2), ((3, 2, 1), 1, 1, 2), ((300, 4, 4), 0, 0, 1),
])
def test_pairs_with_walls_at_rest(prec, dims, stokes, skip, bf, monkeypatch):
    """The shapes that test_run_is_single_steps runs with moving walls, which
    take single steps, with walls at rest, in pairs: one plane, whole tiles with
    a force per node, k tiles of unequal width, a long march."""
    monkeypatch.setenv("SLB_STEP2", "1")
    ref, got = (build(dims, prec, 0, stokes, skip, bf) for _ in range(2))
    assert got.L.slb_run_kernel(got.h) == b"k_step2"
    for n in (2, 7):
        for _ in range(n):
            ref.L.lbstep(ref.h)
        got.L.slb_run(got.h, n)
        assert np.array_equal(ref.pops(), got.pops())
    ref.free()
    got.free()


@pytest.mark.parametrize("dims,mode", [((1, 6016, 6016), 3), ((1, 6000, 6001), 3), ((4, 3072, 3072), 2)])
def test_pairs_on_buffers_over_4_gb(dims, mode, monkeypatch):
    """FP64: one plane of 4.3 GB, whose byte offsets do not fit 32 bits, of whole
    tiles and ragged; four planes of 1.1 GB.  Momentum and density of every node
    after 4 steps, bit for bit."""
    import sunlightlb_amd as s
    monkeypatch.setenv("SLB_STEP2", "1")
    n, out, d = dims[1], [], None
    for pairs in (0, 1):
        print(f"lattice {dims}, pairs {pairs}", flush=True)
        lat = s.Lattice(*dims, precision=64)
        L, h = lat.L, lat.h
        L.slbd_step2_mode.argtypes = [C.c_long, C.c_long, C.c_int]
        assert 15 * lat.N * 8 > 1 << 32
        assert L.slbd_step2_mode(dims[1] * dims[2], lat.N, 64) == mode
        lat.s.tau, lat.s.stokes_flow = 0.8, 0
        for q in range(4):
            L.insertcyl(h, b"x", 40.0, n * (0.12 + 0.25 * q), n * (0.98 - 0.27 * q))
        L.zerobf(h)
        lat.s.dpdx, lat.s.dpdy, lat.s.dpdz = 1e-5, 2e-5, -3e-5
        if pairs:
            assert L.slb_run_kernel(h) == b"k_step2"
            L.slb_run(h, 4)
        else:
            for _ in range(4):
                L.lbstep(h)
        d = d or L.slbn_malloc(lat.N * 4 * 4)
        L.slb_warm_moments(h, d, 4, 1.0)
        a = np.empty(lat.N * 4, np.float32)
        L.slbn_d2h(a.ctypes.data, d, a.nbytes)
        out.append(a)
        L.slb_destroy(h)
    L.slbn_free(d)
    last = out[0].reshape(-1, 4)[-64:]
    assert np.all(last[:, 1] != 0.0) and np.array_equal(out[0], out[1])


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("dims,nmom,axis,pads,moving", [
    ((9, 32, 64), 3, 0, 0.01, 0),
    ((7, 13, 131), 3, 1, 0.3, 0),     # remainders in j and k, more than one k tile
    ((70, 6, 11), 3, 2, 0.0, 1),      # many planes; factors with wall terms
    ((5, 40, 33), 1, 0, 0.2, 0),
    ((1, 2, 3), 3, 0, 0.01, 0), ((3, 2, 1), 1, 0, 0.0, 0), ((2, 300, 2), 3, 0, 0.01, 0),
])
def test_tracer_pairs_are_single_steps(prec, dims, nmom, axis, pads, moving, monkeypatch):
    """Two tracer steps per pass over the link factors (k_mpstep2, forced)
    against one (k_mpstep_w): P and the moment sums after 32 and 37 steps, bit
    for bit; adsorbing sites among the boundary nodes."""
    out = []
    print(f"tracer pairs: {dims} prec {prec}", flush=True)
    for on in "01":
        monkeypatch.setenv("SLB_MP_STEP2", on)
        lat = build(dims, prec, moving, 0, 0, 1)
        L, h = lat.L, lat.h
        mp = L.newmp(h, b"null")
        mp.contents.alpha, mp.contents.objects_moving = 0.1, moving
        L.mpinit(mp)
        L.mpall(mp, 1.0)
        L.adsph(mp, 2.5, dims[0] / 2, dims[1] / 2, dims[2] / 2)
        L.slb_mp_set_adsorption(mp, pads)
        if nmom > 1:
            L.slb_mp_track_moments(mp, axis)
        got = []
        for n in (32, 37):
            import sunlightlb_amd as s
            L.slb_mp_run(mp, n)
            sums = (C.c_double * 6)()
            L.slb_mp_sums(mp, sums)
            L.slb_mp_sync_host(mp)
            got += [s.view(mp.contents.p, lat.N).copy(), np.array(sums[:])]
        out.append(got)
        lat.free()
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)


BATCH = [  # dims, objects moving, stokes, skip_solid, body force
    ((33, 31, 29), 1, 1, 0, 0), ((12, 40, 64), 0, 0, 1, 1), ((5, 3, 701), 1, 0, 0, 1), ((2, 2, 2), 1, 1, 0, 1),
    ((1, 1, 7), 0, 1, 0, 1), ((70, 4, 5), 1, 0, 1, 0), ((3, 120, 1), 1, 1, 0, 1),
]


@pytest.mark.parametrize("prec", [64, 32])
def test_batch_pairs_are_single_steps(prec, monkeypatch):
    """A batch in pairs (k_bstep2, wall terms from their rows) against single
    steps (k_bstep): populations after 33 and 2 steps, bit for bit, on boxes at
    the edges of its tiles; forces of measure() to the order of their atomics."""
    out = []
    for on in "01":
        monkeypatch.setenv("SLB_BATCH_STEP2", on)
        print(f"batch pairs: prec {prec} pairs {on}", flush=True)
        b, nobj = None, []
        for q, (dims, moving, stokes, skip, bf) in enumerate(BATCH):
            lat = build(dims, prec, moving, stokes, skip, bf)
            if b is None:
                b = lat.L.slb_batch_new(prec)
            n = len(lat.objects())
            vel = np.random.default_rng(q).normal(0, 0.01, (2, n, 6)) if moving else None
            assert lat.L.slb_batch_add(b, lat.h, 2, vel.ctypes.data_as(C.POINTER(C.c_double))
                                       if moving else None) == q
            nobj.append(n)
            L = lat.L
            lat.free()
        assert L.slb_batch_commit(b) == 0
        got = []
        for n in (33, 2):
            L.slb_batch_run(b, n)
            for q, (dims, *_) in enumerate(BATCH):
                for r in range(2):
                    a = np.zeros(15 * int(np.prod(dims)))
                    L.slb_batch_get_pops(b, q, r, a.ctypes.data_as(C.POINTER(C.c_double)))
                    got.append(a)
        L.slb_batch_measure(b)
        frc = []
        for q, n in enumerate(nobj):
            f, t = np.zeros(3 * max(n, 1)), np.zeros(3 * max(n, 1))
            assert L.slb_batch_forces(b, q, 1, f.ctypes.data_as(C.POINTER(C.c_double)),
                                      t.ctypes.data_as(C.POINTER(C.c_double))) == n
            frc.append(np.concatenate([f, t]))
        out.append((got, frc))
        L.slb_batch_free(b)
    for a, c in zip(out[0][0], out[1][0]):
        assert np.all(np.isfinite(a)) and np.array_equal(a, c)
    for a, c in zip(out[0][1], out[1][1]):
        assert np.abs(a - c).max() <= 1e-12 * max(np.abs(a).max(), 1e-30)


def test_batch_pairs_many_right_hand_sides(monkeypatch):
    """More right-hand sides of one box than a launch of the wall rows takes
    (32768): populations of the problems at that edge, bit for bit."""
    import sunlightlb_amd as s
    nrhs, out = 32770, []
    for on in "01":          # 1: also where single steps are the faster way
        monkeypatch.setenv("SLB_BATCH_STEP2", on)
        print(f"batch pairs: {nrhs} right-hand sides, pairs {on}", flush=True)
        lat = s.Lattice(6, 5, 4, precision=32)
        L = lat.L
        lat.s.tau, lat.s.stokes_flow, lat.s.objects_moving = 0.7, 1, 1
        assert L.insertsph(lat.h, 1.3, 2.6, 2.2, 1.7)
        n = len(lat.objects())
        vel = np.random.default_rng(3).normal(0, 0.01, (nrhs, n, 6))
        b = L.slb_batch_new(32)
        assert L.slb_batch_add(b, lat.h, nrhs, vel.ctypes.data_as(C.POINTER(C.c_double))) == 0
        lat.free()
        assert L.slb_batch_commit(b) == 0
        L.slb_batch_run(b, 4)
        got = []
        for r in (0, 1, 32767, 32768, 32769):
            a = np.zeros(15 * 120)
            L.slb_batch_get_pops(b, 0, r, a.ctypes.data_as(C.POINTER(C.c_double)))
            assert np.abs(a).max() > 1e-6
            got.append(a)
        out.append(got)
        L.slb_batch_free(b)
    for a, c in zip(*out):
        assert np.array_equal(a, c)


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
@pytest.mark.parametrize("dims,stokes,skip,bf,nt", [
    ((9, 32, 64), 0, 1, 2, 1),        # whole tiles per plane, per-node body force
    ((1, 32, 32), 1, 0, 1, 0),        # one plane, a neighbour of itself
    ((5, 8, 512), 1, 1, 0, 1),        # more than one k tile, no body force
    ((4, 11, 331), 0, 0, 1, 1),       # k tiles of unequal width; rows off the 128-byte lines
    ((1, 1, 7), 0, 0, 1, 0), ((3, 2, 1), 1, 1, 2, 1),
])
def test_every_addressing_mode_is_single_steps(dims, stokes, skip, bf, nt, mode, prec, monkeypatch):
    """The addressing of buffers over 4 GB (modes 2 and 3) on small lattices:
    every mode that reaches the lattice, with and without non-temporal stores."""
    import sunlightlb_amd as s
    L = s.lib()
    L.slbd_step2_mode_ok.argtypes = [C.c_int, C.c_long, C.c_long, C.c_int]
    plane = dims[1] * dims[2]
    if not L.slbd_step2_mode_ok(mode, plane, dims[0] * plane, prec):
        assert mode in (0, 2) and plane % 1024
        return
    print(f"pairs: {dims} prec {prec} mode {mode} nt {nt}", flush=True)
    monkeypatch.setenv("SLB_STEP2_MODE", str(mode))
    monkeypatch.setenv("SLB_NT_STORE", str(nt))
    ref, got = (build(dims, prec, 0, stokes, skip, bf) for _ in range(2))
    for n in (2, 5):
        for _ in range(n):
            ref.L.lbstep(ref.h)
        got.L.slb_run(got.h, n)
        assert np.array_equal(ref.pops(), got.pops())
    ref.free()
    got.free()


def limited_batch(limit, env, monkeypatch):
    """A committed batch under a limit of device memory (0: none): its handle,
    the bytes it holds, and the populations after 35 steps and 3 more at
    another launch shape."""
    monkeypatch.setenv("SLB_BATCH_STEP2", env)
    lats = [build(d, 32, 1, 1, 0, 0) for d in ((33, 31, 29), (40, 24, 36))]
    L = lats[0].L
    L.slbd_batch_mem_limit.argtypes, L.slbd_batch_mem_limit.restype = [C.c_size_t], C.c_size_t
    b = L.slb_batch_new(32)
    for lat in lats:
        n = len(lat.objects())
        vel = np.random.default_rng(n).normal(0, 0.01, (3, n, 6))
        L.slb_batch_add(b, lat.h, 3, vel.ctypes.data_as(C.POINTER(C.c_double)))
        lat.free()
    try:
        L.slbd_batch_mem_limit(limit)
        assert L.slb_batch_commit(b) == 0
        held = L.slbd_batch_mem_limit(limit)
        kernel = L.slb_batch_run_kernel(b).decode()
        L.slb_batch_run(b, 35)
        L.slb_batch_set_config(b, 64, 1, 0)      # four times the tiles
        L.slb_batch_run(b, 3)
    finally:
        L.slbd_batch_mem_limit(0)
    out = []
    for q, n in enumerate((33 * 31 * 29, 40 * 24 * 36)):
        a = np.zeros(15 * n)
        L.slb_batch_get_pops(b, q, 2, a.ctypes.data_as(C.POINTER(C.c_double)))
        out.append(a)
    after = L.slb_batch_run_kernel(b).decode()
    L.slb_batch_free(b)
    return held, kernel, after, out


def test_batch_without_memory_for_pairs_runs_single_steps(monkeypatch):
    """The tables of single steps come before those of the pairs: whatever is
    left for the latter, the batch runs, with the same results."""
    single, k, _, ref = limited_batch(0, "0", monkeypatch)
    pairs, k2, after, got = limited_batch(0, "1", monkeypatch)
    assert (k, k2, after) == ("k_bstep", "k_bstep2", "k_bstep2") and pairs > single
    assert all(np.array_equal(a, c) for a, c in zip(ref, got))
    # from what single steps hold (and commit needs for the masks, and the tiles of
    # the second shape) up to a byte too few
    least = single + 4 * (33 * 31 * 29 + 40 * 24 * 36) + 40000
    assert least < pairs
    for limit in (least, (single + pairs) // 2, pairs - 1, pairs, pairs + 20000):
        held, k, after, got = limited_batch(limit, "1", monkeypatch)
        print(f"batch memory limit {limit}: holds {held}, {k}, {after}", flush=True)
        assert held <= limit and k == ("k_bstep2" if limit >= pairs else "k_bstep")
        # the second shape's tiles (18 kB more) take the pairs' memory where there is no other
        assert after == ("k_bstep2" if limit >= pairs + 20000 else "k_bstep")
        assert all(np.array_equal(a, c) for a, c in zip(ref, got))
