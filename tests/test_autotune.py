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
