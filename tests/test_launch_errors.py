"""A launch that fails in the middle of a call (CPU emulation: the n-th launch of
a call does not run and reports an error): the call says so, the steps (in a
batch, stages) that were completed before it count, what is read back is the
state after them, bit for bit, and the solve goes on from there."""
import ctypes

import numpy as np
import pytest

import cases
from mcv_sw_amd import capi

FORMS = [("RK4", capi.FP64), ("RK3_TVD", capi.FP64), ("RK4", capi.FP32C), ("RK3_TVD", capi.FP32C)]
STEPS, MORE = 3, 2


def _fail_launch(path, n):
    ctypes.c_long.in_dll(ctypes.CDLL(path), "mcv_emu_fail_launch").value = n


def _same(a, b, ok):
    return all(np.array_equal(a[k][:, ok], b[k][:, ok]) for k in capi.STATE_FIELDS)


@pytest.mark.parametrize("tile", [0, 1])  # the boundary pass inside the stages; launches of its own
@pytest.mark.parametrize("scheme,precision", FORMS)
def test_emulated_step_goes_on_after_a_failed_launch(emu_lib, scheme, precision, tile):
    dof, n = 3, 5
    m = cases.mesh(dof, n)
    st = cases.case5(m)
    ok = cases.masks(dof, n)["defined"]

    def solver():
        s = capi.Solver(dof, n, 200.0, m, st, scheme=scheme, precision=precision, lib=emu_lib)
        s.set_tile(tile)
        return s

    with solver() as s:
        ref = [s.sync()]
        for _ in range(STEPS + MORE):
            s.step(1)
            ref.append(s.sync())
    stages = 4 if scheme == "RK4" else 3
    launches = STEPS * stages + 1 if tile == 0 else 2 * STEPS * stages
    for f in range(1, launches + 1):
        with solver() as s:
            _fail_launch(emu_lib, f)
            with pytest.raises(capi.MCVError) as e:
                s.step(STEPS)
            assert e.value.code == capi.MCV_EDEVICE
            done = s.steps_done
            # the step whose last boundary launch fails is complete as well
            whole = (f - 1) // (stages if tile == 0 else 2 * stages)
            assert done in (whole, whole + 1) and done <= STEPS, f
            assert _same(s.sync(), ref[done], ok), f
            s.step(STEPS + MORE - done)
            assert _same(s.sync(), ref[-1], ok), f


@pytest.mark.parametrize("tile", [0, 1])
@pytest.mark.parametrize("timed", [False, True])
def test_emulated_batch_goes_on_after_a_failed_launch(emu_lib, timed, tile):
    specs = [(3, 5, "RK3_TVD", capi.FP32C, 5), (4, 3, "RK4", capi.FP64, 4)]

    def batch():
        b = capi.Batch(3, lib=emu_lib)
        slots = []
        for dof, n, scheme, precision, steps in specs:
            m = cases.mesh(dof, n)
            slots.append(b.add(dof, n, 200.0, m, cases.case5(m), steps, scheme=scheme,
                               precision=precision))
        b.set_tile(tile)
        return b, slots

    def same(b, slots, ref):
        for (dof, n, *_), slot, r in zip(specs, slots, ref):
            assert _same(b.sync(slot), r, cases.masks(dof, n)["defined"])

    b, slots = batch()
    with b:
        b.run(16)
        ref = [b.sync(s) for s in slots]
    stages = 5
    # the launch that fails: a stage or a boundary pass, at either progress table
    for f in range(1, (stages if tile == 0 else 2 * stages) + 1):
        b, slots = batch()
        with b:
            _fail_launch(emu_lib, f)
            with pytest.raises(capi.MCVError) as e:
                b.run_timed(stages) if timed else b.run(stages)
            assert e.value.code == capi.MCV_EDEVICE
            done = f - 1 if tile == 0 else f // 2  # stages launched
            left, steps = b.poll()
            assert list(steps[:2]) == [done // 3, done // 4], f
            # a solve admitted now is not taken from an older table
            extra = b.add(3, 5, 200.0, *_inputs(), 1)
            b.run(12 - done)  # to a step boundary of both
            left, steps = b.poll()
            assert list(steps) == [4, 3, 1] and list(left) == [1, 1, 0], f
            b.run(12)  # a graph where graphs are used
            same(b, slots, ref)
            assert np.isfinite(b.sync(extra)["mass"])


def _inputs():
    m = cases.mesh(3, 5)
    return m, cases.case5(m)
