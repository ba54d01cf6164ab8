"""Where runs take two steps per pass, decided on the host without a GPU:
shapes on both sides of each line of the rule, as they were measured."""
import ctypes as C
import os

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "sunlightlb_amd", "libsunlightlb.so")


class Plan(C.Structure):
    _fields_ = [(n, C.c_int) for n in ("jt", "kt", "ci", "njt", "nkt", "nch")]


STEP = [  # esi, esj, esk, precision, two steps per pass are the faster way
    (256, 256, 256, 32, 1), (512, 512, 512, 32, 1), (131, 97, 75, 64, 1), (32, 32, 32, 64, 1),
    (4, 4, 4, 32, 1), (1, 64, 64, 64, 1), (1, 256, 256, 32, 1), (2, 1024, 1024, 32, 1),
    (1236, 1, 2635, 32, 1), (1024, 1024, 1, 64, 1), (1000, 10, 10, 32, 1), (12000, 10, 10, 64, 1),
    (20, 109, 665, 32, 1), (1, 1, 4096, 32, 1), (3, 6144, 6144, 64, 1),
    (1, 1024, 1024, 32, 0), (1, 1024, 1024, 64, 0), (1, 2923, 899, 32, 0), (1, 759, 2191, 64, 0),
    (1, 1, 65536, 32, 0), (65536, 1, 1, 64, 0), (4096, 1, 1, 32, 0), (5000, 8, 8, 32, 0),
    (5000, 8, 8, 64, 0), (12000, 10, 10, 32, 0), (1671, 12, 2, 32, 0), (3, 8, 2034, 32, 0),
]


@pytest.mark.parametrize("esi,esj,esk,prec,pays", STEP)
def test_two_steps_per_pass_where_they_are_faster(esi, esj, esk, prec, pays):
    L, p = C.CDLL(LIB), Plan()
    assert L.slbd_step2_plan(esi, esj, esk, prec, C.byref(p)) == 1
    assert (p.jt + 2) * (p.kt + 2) <= (1024 if prec == 32 else 768)
    assert p.njt * p.jt >= esj and p.nkt * p.kt >= esk and p.nch * p.ci >= esi
    assert L.slbd_step2_pays(esi, esj, esk, prec, C.byref(p)) == pays


def test_ragged_rows_do_not_take_the_narrowest_tiles():
    """No tile width puts rows of 665 values on the 128-byte lines."""
    L, p = C.CDLL(LIB), Plan()
    L.slbd_step2_plan(20, 109, 665, 32, C.byref(p))
    assert p.kt >= 64


TRACER = [  # esi, esj, esk, precision, moments tracked (values per node), as above
    (128, 128, 128, 32, 3, 1), (256, 256, 256, 32, 3, 1), (128, 128, 128, 64, 1, 1),
    (1236, 1, 2635, 32, 3, 1), (1024, 1024, 1, 32, 1, 1), (2236, 2, 70, 64, 3, 1),
    (2, 1024, 1024, 32, 1, 1), (100, 90, 70, 32, 3, 1),
    (1, 1024, 1024, 32, 3, 0), (1, 1024, 1024, 32, 1, 0), (1, 2907, 2023, 64, 3, 0),
    (1024, 1024, 1, 32, 3, 0), (2, 1024, 1024, 32, 3, 0), (12000, 10, 10, 32, 3, 0),
    (12000, 10, 10, 64, 1, 0), (1200000, 1, 1, 32, 3, 0), (1, 1, 1200000, 32, 1, 0),
    (663, 3, 334, 32, 3, 0),
]


@pytest.mark.parametrize("esi,esj,esk,prec,nmom,pays", TRACER)
def test_two_tracer_steps_per_pass_where_they_are_faster(esi, esj, esk, prec, nmom, pays):
    L, p = C.CDLL(LIB), Plan()
    ok = L.slbd_mp2_plan(esi, esj, esk, prec, nmom, C.byref(p))
    assert (ok and L.slbd_mp2_pays(esj, esk, nmom, C.byref(p))) == pays


BATCH = [  # boxes (esi, esj, esk, right-hand sides, moving), precision, pairs, least blocks
    ([(64, 64, 64, 1, 0)], 32, 1, 128), ([(64, 64, 64, 1, 1)], 64, 1, 128),
    ([(48, 48, 48, 1, 1)], 32, 1, 100), ([(128, 128, 128, 1, 0)], 32, 1, 200),
    ([(64, 64, 64, 6, 1)], 32, 1, 200), ([(256, 256, 4, 2, 0)] * 2, 32, 1, 200),
    ([(112, 7, 15, 1, 1)] * 2, 64, 1, 60), ([(94, 49, 5, 1, 0)] * 5, 64, 1, 120),
    ([(48, 54, 33, 6, 1), (40, 61, 62, 6, 1), (33, 35, 64, 6, 1)] * 10, 32, 1, 200),
    ([(6, 6, 6, 6, 0)] * 256, 32, 0, 0), ([(8, 8, 8, 6, 1)] * 64, 64, 0, 0),
    ([(64, 64, 1, 6, 0)] * 64, 32, 0, 0), ([(96, 5, 5, 3, 0)] * 40, 64, 0, 0),
    ([(5, 3, 701, 1, 1)], 64, None, 0), ([(1, 1, 1, 1, 0)], 32, None, 0), ([(2, 300, 1, 1, 1)], 64, None, 0),
]


@pytest.mark.parametrize("boxes,prec,pays,least", BATCH)
def test_batch_plan(boxes, prec, pays, least):
    """Tiles that fit a block and cover their box, enough of them to use the
    CUs where the problems are few, and single steps where those are faster."""
    L, n = C.CDLL(LIB), len(boxes)
    box = (C.c_int * (5 * n))(*[v for b in boxes for v in b])
    tile, us = (C.c_int * (3 * n))(), (C.c_double * 2)()
    got = L.slbd_bstep2_plan(n, box, prec, tile, us)
    blocks = 0
    for q, (esi, esj, esk, nrhs, _) in enumerate(boxes):
        jt, kt, ci = tile[3 * q:3 * q + 3]
        assert 1 <= jt <= esj and 1 <= kt <= esk and 1 <= ci <= esi
        assert (jt + 2) * (kt + 2) <= (1024 if prec == 32 else 512)
        blocks += -(-esi // ci) * -(-esj // jt) * -(-esk // kt) * nrhs
    if pays is not None:
        assert got == pays and (us[0] < us[1]) == pays
    if pays:
        assert blocks >= least
