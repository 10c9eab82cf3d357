"""The autotuners time a stage as the steps run it.  In the CPU emulation a
launch lasts one unit of time, so a tile shape's time per stage is its launches
per stage: one where the boundary pass runs inside the stage kernel (shapes 0
and 2 of small work), two where it is a launch of its own.  Tuning at any step
boundary leaves the trajectory as it is."""
import ctypes

import numpy as np
import pytest

import cases
from mcv_sw_amd import capi

FORMS = [("RK4", capi.FP64), ("RK3_TVD", capi.FP64), ("RK4", capi.FP32C), ("RK3_TVD", capi.FP32C)]


def _raw_launches(path):
    return ctypes.c_long.in_dll(ctypes.CDLL(path), "mcv_emu_raw_launches").value


@pytest.mark.parametrize("scheme,precision", FORMS)
@pytest.mark.parametrize("dof,n", [(3, 9), (4, 7)])
def test_emulated_tuner_times_whole_stages(emu_lib, dof, n, scheme, precision):
    m = cases.mesh(dof, n)
    with capi.Solver(dof, n, 200.0, m, cases.case5(m), scheme=scheme, precision=precision,
                     lib=emu_lib) as s:
        raw = _raw_launches(emu_lib)
        tile, ms = s.autotune(reps=2)
        assert list(ms) == [1.0, 2.0, 1.0, 2.0]
        assert tile == 0
        assert _raw_launches(emu_lib) > raw  # shapes 0 and 2 on a raw level


BATCH = [(3, 9, "RK3_TVD", capi.FP32C, 2), (4, 7, "RK4", capi.FP64, 4), (3, 5, "RK4", capi.FP32C, 1)]


def _batch(lib, tune):
    """A batch tuned before its first stage, between steps of all its solves (one
    of them spent by then), and at the end."""
    with capi.Batch(len(BATCH), lib=lib) as b:
        slots = []
        for dof, n, scheme, precision, steps in BATCH:
            m = cases.mesh(dof, n)
            slots.append(b.add(dof, n, 200.0, m, cases.case5(m), steps, scheme=scheme,
                               precision=precision))
        ms = []
        for stages in (12, 4):  # 12: a multiple of 3 and 4
            if tune:
                ms.append(list(b.autotune(reps=1)[1]))
                b.set_tile(0)
            b.run(stages)
        b.run(1)  # finishes every level again, spent solves' too
        return ms, [b.sync(s) for s in slots]


def _check_batch(lib):
    ref = _batch(lib, False)[1]
    ms, out = _batch(lib, True)
    for (dof, n, *_), a, c in zip(BATCH, ref, out):
        ok = cases.masks(dof, n)["defined"]
        for k in capi.STATE_FIELDS:
            assert np.array_equal(a[k][:, ok], c[k][:, ok]), (dof, n, k)
    return ms


def test_emulated_batch_tuner_times_whole_stages(emu_lib):
    ms = _check_batch(emu_lib)
    assert ms == [[1.0, 2.0, 1.0, 2.0]] * 2
    with capi.Batch(1, lib=emu_lib) as b:
        m = cases.mesh(3, 9)
        b.add(3, 9, 200.0, m, cases.case5(m), 5)
        raw = _raw_launches(emu_lib)
        b.autotune(reps=1)
        assert _raw_launches(emu_lib) > raw


@pytest.mark.gpu
def test_gpu_batch_tuning_keeps_the_trajectories(hip_lib):
    print("[tuning] batch", flush=True)
    _check_batch(None)


def _trajectory(lib, dof, n, scheme, precision):
    m = cases.mesh(dof, n)
    st = cases.case5(m)
    ok = cases.masks(dof, n)["defined"]
    outs = []
    for tune in (False, True):
        with capi.Solver(dof, n, 200.0, m, st, scheme=scheme, precision=precision, lib=lib) as s:
            for steps in (1, 2):  # before the first step and between steps
                if tune:
                    s.autotune(reps=1)
                    outs.append(s.sync())
                    s.set_tile(0)
                else:
                    outs.append(s.sync())
                s.step(steps)
            outs.append(s.sync())
    for a, b in zip(outs[:3], outs[3:]):
        for k in capi.STATE_FIELDS:
            assert np.array_equal(a[k][:, ok], b[k][:, ok]), k
        assert a["mass"] == b["mass"] and a["energy"] == b["energy"]


@pytest.mark.parametrize("scheme,precision", FORMS)
def test_emulated_tuning_keeps_the_trajectory(emu_lib, scheme, precision):
    _trajectory(emu_lib, 3, 9, scheme, precision)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,precision", FORMS)
@pytest.mark.parametrize("dof,n", [(3, 21), (4, 13)])
def test_gpu_tuning_keeps_the_trajectory(hip_lib, dof, n, scheme, precision):
    print(f"[tuning] dof={dof} n={n} {scheme} precision={precision}", flush=True)
    _trajectory(None, dof, n, scheme, precision)
