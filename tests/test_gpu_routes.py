"""Which kernel a run takes (slb_run_kernel, slb_mp_run_kernel,
slb_batch_run_kernel): the two-steps-per-pass kernels where they apply, the
single-step ones where the walls move, the environment says so, or two steps
per pass are the slower way over the lattice."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_pairs import build

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("env,moving,want", [
    ({}, 0, "k_step2"), ({}, 1, "k_step_lds"), ({"SLB_STEP2": "0"}, 0, "k_step_lds"),
    ({"SLB_STEP2": "1"}, 0, "k_step2"), ({"SLB_STEP_LDS": "0"}, 0, "k_step"),
    ({"SLB_INDEX64": "1"}, 0, "k_step_lds"), ({"SLB_STEP_MOM": "1"}, 0, "k_step_mom"),
    ({"SLB_SWEEP": "8"}, 0, "k_step_lds"),
])
def test_kernel_of_a_run(env, moving, want, monkeypatch):
    import sunlightlb_amd as s
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    lat = s.Lattice(40, 32, 64, precision=32)
    lat.s.objects_moving = moving
    assert lat.L.slb_run_kernel(lat.h).decode() == want
    lat.free()


def test_thin_lattices_keep_single_steps(monkeypatch):
    import sunlightlb_amd as s
    for on, want in ((None, "k_step"), ("1", "k_step2")):
        if on:
            monkeypatch.setenv("SLB_STEP2", on)
        lat = s.Lattice(5000, 8, 8, precision=32)
        assert lat.L.slb_run_kernel(lat.h).decode() == want
        lat.free()


@pytest.mark.parametrize("dims,prec,steps,env,want", [
    ((64, 64, 64), 32, 64, {}, "k_mpstep_w"), ((64, 64, 64), 32, 31, {}, "k_mpstep"),
    ((88, 88, 88), 32, 64, {}, "k_mpstep2"), ((88, 88, 88), 64, 64, {}, "k_mpstep2"),
    ((88, 88, 88), 32, 64, {"SLB_MP_STEP2": "0"}, "k_mpstep_w"),
    ((9, 8, 7), 32, 64, {"SLB_MP_STEP2": "1"}, "k_mpstep2"),
    ((1, 800, 800), 32, 64, {}, "k_mpstep_w"), ((1, 800, 800), 32, 64, {"SLB_MP_STEP2": "1"}, "k_mpstep2"),
    ((88, 88, 88), 32, 64, {"SLB_MP_WEIGHTS": "0"}, "k_mpstep"),
    ((88, 88, 88), 32, 64, {"SLB_INDEX64": "1"}, "k_mpstep_w"),
])
def test_kernel_of_a_tracer_run(dims, prec, steps, env, want, monkeypatch):
    import sunlightlb_amd as s
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    lat = s.Lattice(*dims, precision=prec)
    mp = lat.L.newmp(lat.h, b"null")
    assert lat.L.slb_mp_run_kernel(mp, steps).decode() == want
    lat.free()


@pytest.mark.parametrize("dims,boxes,env,want", [
    ((40, 40, 48), 6, {}, "k_bstep2"), ((40, 40, 48), 6, {"SLB_BATCH_STEP2": "0"}, "k_bstep"),
    ((64, 64, 64), 1, {}, "k_bstep2"), ((6, 6, 6), 64, {}, "k_bstep"),
    ((6, 6, 6), 64, {"SLB_BATCH_STEP2": "1"}, "k_bstep2"),
])
def test_kernel_of_a_batch(dims, boxes, env, want, monkeypatch):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    lat = build(dims, 32, 1, 1, 0, 0)
    L, n = lat.L, len(lat.objects())
    b = L.slb_batch_new(32)
    vel = np.zeros((6, n, 6))
    for _ in range(boxes):
        L.slb_batch_add(b, lat.h, 6, vel.ctypes.data_as(C.POINTER(C.c_double)))
    lat.free()
    assert L.slb_batch_commit(b) == 0
    assert L.slb_batch_run_kernel(b).decode() == want
    L.slb_batch_free(b)
