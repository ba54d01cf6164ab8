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
