"""The warm-start network's weight gradient on x-rows of any length, its
input expansion, and the lattice hooks' features and moments, at the edges
of their groups and blocks.  Bars as in test_gpu_warm.py: FP32 weight
gradients within 1e-5 of the oracle relative to the largest value, features
and copies bit-exact."""
import ctypes as C

import numpy as np
import pytest

from oracle import nn as onn
from test_gpu_warm import Dev, bf_random, lib, test_conv_forward_matches_oracle as conv_matches_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (64, 32), (64, 64)])
@pytest.mark.parametrize("shape", [(3, 4, 1), (4, 3, 2), (2, 5, 7), (3, 3, 9), (5, 4, 12), (4, 2, 23),
                                   (2, 3, 36), (6, 5, 18), (2, 2, 141)])
def test_weight_gradient_on_ragged_rows(shape, cin, cout):
    L = lib()
    print(f"ragged wgrad {shape} {cin}->{cout}", flush=True)
    assert L.slbn_wgrad_blocked_ok(cin, cout, *shape)
    rng = np.random.default_rng(sum(shape) + cin + cout)
    xb, x = bf_random(rng, shape + (cin,))
    gb, g = bf_random(rng, shape + (cout,))
    kp = onn.kpad(cin)
    dX, dG, dW = Dev(host=xb), Dev(host=gb), Dev(cout * kp * 4)
    L.slbn_conv_wgrad(dX.p, cin, dG.p, cout, dW.p, *shape)
    L.slbn_sync()
    got = dW.get(np.float32, (cout, kp)).astype(np.float64)
    for d in (dX, dG, dW):
        d.free()
    ref = onn.conv3d_bwd_weight(x, g).reshape(cout, 27 * cin)
    assert np.all(got[:, 27 * cin:] == 0.0)
    assert np.abs(got[:, :27 * cin] - ref).max() < 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("cin,cout", [(16, 16), (16, 32), (32, 64), (64, 16)])
@pytest.mark.parametrize("shape", [(4, 4, 64), (16, 128, 64)])   # one, four node tiles per wave
def test_general_convolution_equals_the_staged_one(shape, cin, cout, monkeypatch):
    """Same K order and MFMA sequence: bit for bit."""
    L = lib()
    rng = np.random.default_rng(cin + cout)
    xb, _ = bf_random(rng, shape + (cin,))
    wb, _ = bf_random(rng, (cout, onn.kpad(cin)), 0.1)
    wb[:, 27 * cin:] = 0
    dX, dW, n = Dev(host=xb), Dev(host=wb), int(np.prod(shape))
    got = []
    for on in "01":
        monkeypatch.setenv("SLBN_CONV_LDS", on)
        dY, dF = Dev(n * cout * 2), Dev(n * cout * 4)
        L.slbn_conv(dX.p, cin, dW.p, None, dY.p, dF.p, cout, 1, 0, *shape)
        L.slbn_sync()
        got.append((dY.get(np.uint16, (n, cout)), dF.get(np.uint32, (n, cout))))
        dY.free()
        dF.free()
    dX.free()
    dW.free()
    assert got[0][1].any()
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("cin,cout", [(16, 16), (32, 64), (64, 32)])
@pytest.mark.parametrize("shape", [(4, 128, 64), (8, 128, 64), (16, 128, 128)])
def test_two_and_four_node_tiles_equal_the_staged_one(shape, cin, cout, monkeypatch):
    """Two node tiles per wave, and the generic channel count (32 -> 64 on 262
    thousand nodes)."""
    test_general_convolution_equals_the_staged_one(shape, cin, cout, monkeypatch)


@pytest.mark.parametrize("cin,cout", [(16, 16), (24, 8), (64, 64)])
@pytest.mark.parametrize("shape", [(13, 37, 41), (3, 79, 71)])
def test_two_node_tiles_with_a_remainder(shape, cin, cout):
    """19721 and 16827 nodes: the last wave's second tile partly and wholly past the end."""
    conv_matches_oracle(shape, cin, cout, 1)


@pytest.mark.parametrize("cs,c", [(2, 16), (16, 16), (8, 16), (10, 16), (3, 12), (24, 8)])
def test_expand(cs, c):
    L = lib()
    n = 773
    s = np.random.default_rng(cs + c).integers(0, 1 << 16, (n, cs)).astype(np.uint16)
    dS, dX = Dev(host=s), Dev(n * c * 2)
    L.slbn_expand(dS.p, cs, dX.p, c, n)
    L.slbn_sync()
    want = np.zeros((n, c), np.uint16)
    want[:, :min(cs, c)] = s[:, :min(cs, c)]
    assert np.array_equal(dX.get(np.uint16, (n, c)), want)
    dS.free()
    dX.free()


@pytest.mark.parametrize("dims", [(5, 7, 3), (2, 3, 1030), (17, 4, 33), (1, 1, 6)])
def test_features_at_odd_extents(dims):
    """Seeds as coordinates (extents up to 1024) and as node indices."""
    import sunlightlb_amd as s
    lat = s.Lattice(*dims, precision=64)
    solid = np.random.default_rng(sum(dims)).random(dims) < 0.1
    solid.reshape(-1)[0] = True
    m = np.ascontiguousarray(solid.astype(np.uint8).reshape(-1))
    lat.L.slb_insert_map(lat.h, m.ctypes.data_as(C.c_void_p))
    f, ell_ref = onn.features(solid)
    for ch in (2, 8, 16, 3):
        dF = Dev(lat.N * ch * 2)
        ell = lat.L.slb_warm_features(lat.h, dF.p, ch)
        got = dF.get(np.uint16, dims + (ch,))
        dF.free()
        assert abs(ell - ell_ref) < 1e-12 * ell_ref
        want = np.zeros(dims + (ch,), np.uint16)
        want[..., :2] = onn.bf16_bits(f)
        assert np.array_equal(got, want)
    lat.free()


@pytest.mark.parametrize("dims", [(3, 5, 7), (4, 8, 8), (5, 9, 23)])
def test_moments_of_any_channel_count(dims):
    """The moments' first channels are the same whatever the channel count."""
    import sunlightlb_amd as s
    lat = s.Lattice(*dims, precision=64)
    lat.L.insertsph(lat.h, 1.5, 1.0, 2.0, 3.0)
    lat.s.dpdx = 1e-3
    lat.set_pops(1e-3 * np.random.default_rng(3).standard_normal(lat.N * 15))
    out = {}
    for ch in (10, 16, 4, 13, 300):
        d = Dev((lat.N * ch + 64) * 4)
        lat.L.slb_warm_moments(lat.h, d.p, ch, 1.0)
        a = d.get(np.float32, (lat.N * ch + 64,))
        d.free()
        assert np.all(a[lat.N * ch:] == 0.0)
        out[ch] = a[:lat.N * ch].reshape(lat.N, ch)
        assert np.all(out[ch][:, 10:] == 0.0)
    for ch in (16, 4, 13, 300):
        q = min(10, ch)
        assert np.array_equal(out[ch][:, :q], out[10][:, :q])
    assert np.abs(out[10]).max() > 0.0
    lat.free()


@pytest.mark.parametrize("ch", [0, -8, -16])
def test_no_channels_write_nothing(ch):
    """Channel counts of zero and below leave the tensors as they are."""
    import sunlightlb_amd as s
    lat = s.Lattice(6, 7, 9, precision=64)
    lat.L.insertsph(lat.h, 2.0, 3.0, 3.0, 4.0)
    lat.s.dpdx = 1e-3
    n = 64 * lat.N
    pat = np.arange(n, dtype=np.uint32)
    d = Dev(host=pat)
    mid = d.p + 2 * n
    ell = lat.L.slb_warm_features(lat.h, mid, ch)
    assert ell > 0.0 and ell == lat.L.slb_warm_features_noalloc(lat.h, mid, ch)
    lat.L.slb_warm_moments(lat.h, mid, ch, 1.0)
    lat.L.slb_warm_targets(lat.h, mid, ch, 1.0)
    assert np.array_equal(d.get(np.uint32, (n,)), pat)
    d.free()
    lat.free()


@pytest.mark.parametrize("ch", [1, 2, 4, 5])
def test_moments_on_few_channels(ch):
    """Both sides of the line between stores from registers and through the LDS,
    FP32 and BF16, a last block that is not full; nothing past the end."""
    import sunlightlb_amd as s
    lat = s.Lattice(5, 9, 23, precision=32)
    lat.L.insertsph(lat.h, 1.5, 1.0, 2.0, 3.0)
    lat.s.dpdx = 1e-3
    lat.set_pops(1e-3 * np.random.default_rng(5).standard_normal(lat.N * 15))
    out = {}
    for c in (10, ch):
        m, t = Dev(lat.N * c * 4 + 64), Dev(lat.N * c * 2 + 64)
        lat.L.slb_warm_moments(lat.h, m.p, c, 1.0)
        lat.L.slb_warm_targets(lat.h, t.p, c, 1.0)
        a, b = m.get(np.float32, (lat.N * c + 16,)), t.get(np.uint16, (lat.N * c + 32,))
        assert not a[lat.N * c:].any() and not b[lat.N * c:].any()
        out[c] = a[:lat.N * c].reshape(lat.N, c), b[:lat.N * c].reshape(lat.N, c)
        m.free()
        t.free()
    for a, b in zip(out[ch], out[10]):
        assert a.any() and np.array_equal(a, b[:, :ch])
    lat.free()


def wgrad_data(shape, cin, cout, seed):
    rng = np.random.default_rng(seed)
    xb, x = bf_random(rng, shape + (cin,))
    gb, g = bf_random(rng, shape + (cout,))
    return Dev(host=xb), Dev(host=gb), onn.conv3d_bwd_weight(x, g).reshape(cout, 27 * cin)


def wgrad_close(got, ref, times=1):
    assert np.abs(got[:, :ref.shape[1]].astype(np.float64) - times * ref).max() < 1e-5 * times * np.abs(ref).max()


@pytest.mark.parametrize("shape", [(6, 5, 18), (4, 6, 16)])
def test_weight_gradient_without_a_workspace(shape, monkeypatch):
    L, cin, cout = lib(), 32, 16
    monkeypatch.setenv("SLBN_WGRAD_WS", "1000")
    dX, dG, ref = wgrad_data(shape, cin, cout, 4)
    dW = Dev(cout * onn.kpad(cin) * 4)
    L.slbn_conv_wgrad(dX.p, cin, dG.p, cout, dW.p, *shape)
    L.slbn_sync()
    wgrad_close(dW.get(np.float32, (cout, onn.kpad(cin))), ref)
    for d in (dX, dG, dW):
        d.free()


def test_weight_gradient_on_two_streams():
    """Calls on two streams overlap: each keeps its own workspace (fixed order
    of summation, so bit for bit the result of a call alone)."""
    import torch
    L, cin, cout, shape, reps = lib(), 32, 32, (20, 20, 18), 12
    kp = onn.kpad(cin)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    data = [wgrad_data(shape, cin, cout, q) for q in range(2)]
    alone, both = [], [[Dev(cout * kp * 4) for _ in range(reps)] for _ in streams]
    try:
        for q, (dX, dG, ref) in enumerate(data):
            dW = Dev(cout * kp * 4)
            L.slbn_conv_wgrad(dX.p, cin, dG.p, cout, dW.p, *shape)
            L.slbn_sync()
            alone.append(dW.get(np.uint32, (cout, kp)))
            wgrad_close(alone[q].view(np.float32), ref)
            dW.free()
        for r in range(reps):
            for q, st in enumerate(streams):
                L.slbn_set_stream(st.cuda_stream)
                L.slbn_conv_wgrad(data[q][0].p, cin, data[q][1].p, cout, both[q][r].p, *shape)
        torch.cuda.synchronize()
    finally:
        L.slbn_set_stream(None)
    for q in range(2):
        for d in both[q]:
            assert np.array_equal(d.get(np.uint32, (cout, kp)), alone[q])
            d.free()


def test_weight_gradient_on_many_streams():
    """More streams than workspaces."""
    import torch
    L, cin, cout, shape = lib(), 16, 16, (5, 6, 9)
    kp = onn.kpad(cin)
    dX, dG, ref = wgrad_data(shape, cin, cout, 2)
    dW = Dev(cout * kp * 4)
    streams = [torch.cuda.Stream() for _ in range(24)]
    assert len({st.cuda_stream for st in streams}) > 16
    try:
        for st in streams:
            L.slbn_set_stream(st.cuda_stream)
            L.slbn_conv_wgrad(dX.p, cin, dG.p, cout, dW.p, *shape)
            L.slbn_sync()
    finally:
        L.slbn_set_stream(None)
    wgrad_close(dW.get(np.float32, (cout, kp)), ref, len(streams))
    for d in (dX, dG, dW):
        d.free()


def test_weight_gradient_in_a_captured_graph():
    """Ragged rows captured without a call before them, and replayed between
    eager calls that grow the workspace."""
    import torch
    L, cin, cout, shape = lib(), 16, 32, (7, 6, 11)
    kp = onn.kpad(cin)
    dX, dG, ref = wgrad_data(shape, cin, cout, 9)
    dW = Dev(cout * kp * 4)
    st, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    try:
        with torch.cuda.graph(g, stream=st):
            L.slbn_set_stream(torch.cuda.current_stream().cuda_stream)
            L.slbn_conv_wgrad(dX.p, cin, dG.p, cout, dW.p, *shape)
    finally:
        L.slbn_set_stream(None)
    torch.cuda.synchronize()
    assert not dW.get(np.float32, (cout, kp)).any()
    for r in range(1, 4):
        g.replay()
        torch.cuda.synchronize()
        wgrad_close(dW.get(np.float32, (cout, kp)), ref, r)
        big = (12 * r, 20, 23)
        bX, bG, bref = wgrad_data(big, cin, cout, 20 + r)
        bW = Dev(cout * kp * 4)
        L.slbn_conv_wgrad(bX.p, cin, bG.p, cout, bW.p, *big)
        L.slbn_sync()
        wgrad_close(bW.get(np.float32, (cout, kp)), bref)
        for d in (bX, bG, bW):
            d.free()
    for d in (dX, dG, dW):
        d.free()


@pytest.mark.parametrize("C,N", [(16, 300001), (64, 40000), (8, 5000), (32, 7), (256, 3000), (4, 70000)])
def test_bias_gradient_is_the_same_at_every_call(C, N):
    """The blocks' sums in a fixed order: 8 calls bit for bit, added to what is
    there; with atomics (no workspace) to rounding."""
    L = lib()
    rng = np.random.default_rng(C + N)
    yb, y = bf_random(rng, (N, C))
    gb, g = bf_random(rng, (N, C))
    dY, dG, dP = Dev(host=yb), Dev(host=gb), Dev(N * C * 2)
    was = rng.standard_normal(C).astype(np.float32)
    ref = np.where(y > 0, g, 0.0).sum(0) + was
    scale = np.abs(g).sum(0).max()
    got = []
    for _ in range(8):
        db = Dev(host=was)
        L.slbn_relu_bwd_bias(dY.p, dG.p, dP.p, C, N, db.p)
        L.slbn_sync()
        got.append(db.get(np.uint32, (C,)))
        db.free()
    for d in (dY, dG, dP):
        d.free()
    assert all(np.array_equal(a, got[0]) for a in got)
    assert np.abs(got[0].view(np.float32) - ref).max() < 1e-5 * scale


def test_bias_gradient_without_a_workspace(monkeypatch):
    monkeypatch.setenv("SLBN_WGRAD_WS", "0")
    L, N, C = lib(), 9000, 32
    gb, g = bf_random(np.random.default_rng(8), (N, C))
    dG, db = Dev(host=gb), Dev(C * 4)
    L.slbn_bias_grad(dG.p, C, N, db.p)
    L.slbn_sync()
    assert np.abs(db.get(np.float32, (C,)) - g.sum(0)).max() < 1e-5 * np.abs(g).sum(0).max()
    dG.free()
    db.free()


@pytest.mark.parametrize("dims", [(16, 24, 32), (16, 16, 40), (24, 16, 72)])
def test_training_can_be_repeated(dims):
    """Two networks of one seed trained on the same packs: the same weights, bit
    for bit (rows that the LDS-staged, the blocked and the padded weight
    gradients take)."""
    import sunlightlb_amd as s
    L, out = lib(), []
    for _ in range(2):
        net = L.slb_warm_new(3)
        for q in range(3):
            lat = s.Lattice(*dims, precision=32)
            lat.s.tau, lat.s.stokes_flow = 0.75, 1
            rng = np.random.default_rng(q)
            for _ in range(4):
                L.insertsph(lat.h, 3.0, *[float(rng.uniform(0, n)) for n in dims])
            L.zerobf(lat.h)
            L.addbf(lat.h, 1e-6, 0.0, 0.0)
            L.slb_run(lat.h, 200)
            L.slb_warm_add_sample(net, lat.h)
            lat.free()
        L.slb_warm_train(net, 40, 1e-3, 5, None)
        w = np.empty(L.slb_warm_nparams(net), np.float32)
        L.slb_warm_get_params(net, w.ctypes.data)
        L.slb_warm_free(net)
        out.append(w)
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])
