"""Addressing of the two-step kernel (k_step2), on the host without a GPU: the
mode that slbd_step2_mode chooses for a lattice must reach every population
with the integers that the kernel computes in that mode.  The kernel's
expressions are restated with its 32-bit wrap-around, and compared with the
64-bit offset of the tiled layout at the corners of the first, second and
last planes and at random nodes."""
import ctypes as C
import os

import numpy as np
import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "sunlightlb_amd", "libsunlightlb.so")
TILE, U32 = 1024, 0xffffffff


def lib():
    L = C.CDLL(LIB)
    L.slbd_step2_mode.argtypes = [C.c_long, C.c_long, C.c_int]
    L.slbd_step2_mode_ok.argtypes = [C.c_int, C.c_long, C.c_long, C.c_int]
    return L


def pidx(l, n):
    return ((n >> 10) * 15 + l) * TILE + (n & 1023)


def kernel_byte(mode, l, p, t, plane, ts):
    """Byte of population l at node p * plane + t, as k_step2 computes it."""
    def i32(v):
        return (v + 2 ** 31 & U32) - 2 ** 31
    if mode in (0, 2):
        off = i32(i32(((t >> 10) * 15) * TILE) + (t & 1023)) * ts & U32
        if mode == 0:
            return ((p * (15 * plane & U32) + l * TILE & U32) * ts + off) & U32
        return (p * 15 * plane + l * TILE) * ts + off
    if mode == 1:
        n = (p * plane * ts + t * ts) & U32
        return (n + (n // (TILE * ts)) * 14 * TILE * ts & U32) + l * TILE * ts
    n = i32(p * plane + t)
    return i32(i32(((n >> 10) * 15 + l) * TILE) + (n & 1023)) * ts


SHAPES = [(d, prec) for prec in (32, 64) for d in [
    (1, 8192, 8192), (2, 8192, 8192), (3, 6144, 6144), (1, 8192, 9216), (1, 10240, 8192),
    (1, 7001, 8191), (2, 8193, 8191), (420, 420, 420), (340, 340, 340), (401, 401, 401),
    (512, 512, 512), (1024, 1024, 1024), (256, 256, 256), (9, 32, 64), (13, 23, 75), (1, 1, 1),
    (1, 11585, 11585), (1, 12000, 12000), (1, 16384, 16384), (2000, 300, 300), (6, 4096, 4368)]]


@pytest.mark.parametrize("dims,prec", SHAPES)
def test_chosen_mode_reaches_every_population(dims, prec):
    L = lib()
    esi, plane, ts = dims[0], dims[1] * dims[2], prec // 8
    N = esi * plane
    mode = L.slbd_step2_mode(plane, N, prec)
    big = 15 * -(-N // TILE) * TILE
    if mode < 0:
        # neither 31-bit population indices nor whole-tile planes under 4 GB
        assert big > 2 ** 31 - 1 and (plane % TILE or 15 * plane * ts >= 2 ** 32)
        return
    rng = np.random.default_rng(7)
    planes = {0, min(1, esi - 1), esi - 1, int(rng.integers(esi))}
    cols = {0, plane - 1, plane // 2} | {int(t) for t in rng.integers(plane, size=40)}
    for m in range(4):
        if not L.slbd_step2_mode_ok(m, plane, N, prec):
            assert m != mode
            continue
        for p in planes:
            for t in cols:
                for l in (0, 7, 14):
                    assert kernel_byte(m, l, p, t, plane, ts) == pidx(l, p * plane + t) * ts, \
                        (m, p, t, l)


def test_large_planes_keep_their_pairs_where_indices_allow():
    """Planes of 4 GB and more whose population indices fit 31 bits."""
    L = lib()
    for dims in ((1, 8192, 8192), (2, 8192, 8192), (3, 6144, 6144)):
        plane, N = dims[1] * dims[2], dims[0] * dims[1] * dims[2]
        assert L.slbd_step2_mode(plane, N, 64) == 3
    assert L.slbd_step2_mode(512 * 512, 512 ** 3, 32) == 2
    assert L.slbd_step2_mode(420 * 420, 420 ** 3, 32) == 3
    assert L.slbd_step2_mode(16384 * 16384, 16384 * 16384, 64) == -1
