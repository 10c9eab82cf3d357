"""Large read-backs through the copy threads against the handed-over state, which
a solve holds until its first step: the same bytes, also with two solves read at
once (one of them finds the copy threads busy).  Sizes on both sides of the rule:
six fields of 1.7 MB (four threads) and of 7 MB (eight), none a whole number of
chunks; single fields below the rule (a plain copy) and above it."""
import ctypes
import threading

import numpy as np
import pytest

import cases
from mcv_sw_amd import capi


def _handed_over(m, st):
    return {**{k: st[k] for k in capi.STATE_FIELDS}, "phiG": st["phi"] * m["sqrtG"]}


def _assert_same(out, want):
    for k, x in out.items():
        assert np.array_equal(x, want[k]), k


def _check(lib, dof, n):
    m = cases.mesh(dof, n)
    st = cases.case5(m)
    want = _handed_over(m, st)
    with capi.Solver(dof, n, 50.0, m, st, lib=lib) as a, capi.Solver(dof, n, 50.0, m, st,
                                                                     lib=lib) as b:
        for k in capi.STATE_FIELDS:
            _assert_same(a.sync(fields=(k,), integrals=False), want)
        outs = [None, None]

        def read(i, s):
            outs[i] = [s.sync(integrals=False) for _ in range(3)]

        team = [threading.Thread(target=read, args=x) for x in ((0, a), (1, b))]
        for t in team:
            t.start()
        for t in team:
            t.join()
        for out in outs[0] + outs[1]:
            assert set(out) == set(capi.STATE_FIELDS)
            _assert_same(out, want)


@pytest.mark.parametrize("dof,n", [(4, 60), (3, 190)])
def test_emulated_large_readback(emu_lib, dof, n):
    # one solve at a time here: the shim's launches share their LDS statics
    m = cases.mesh(dof, n)
    st = cases.case5(m)
    want = _handed_over(m, st)
    with capi.Solver(dof, n, 50.0, m, st, lib=emu_lib) as s:
        _assert_same(s.sync(integrals=False), want)
        for k in capi.STATE_FIELDS:
            _assert_same(s.sync(fields=(k,), integrals=False), want)


def test_emulated_pinned_memory_is_kept_by_a_batch(emu_lib):
    """One solve at a time through a resident batch: the pinned memory of the
    read-backs is made once, and given back with the batch."""
    lib = ctypes.CDLL(emu_lib)

    def pinned(name):
        return ctypes.c_long.in_dll(lib, f"mcv_emu_pinned_{name}").value

    m = cases.mesh(4, 60)
    st = cases.case5(m)
    made = pinned("made")
    with capi.Batch(1, lib=emu_lib) as b:
        for _ in range(3):
            slot = b.add(4, 60, 50.0, m, st, 0)
            out = b.sync(slot, integrals=False)
            assert np.array_equal(out["phi"], st["phi"])
            b.remove(slot)
        assert pinned("made") == made + 1 and pinned("live") == 1
    assert pinned("live") == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dof,n", [(4, 60), (3, 190)])
def test_gpu_large_readback(hip_lib, dof, n):
    _check(None, dof, n)
