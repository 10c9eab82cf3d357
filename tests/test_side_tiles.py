"""The boundary pass inside the stage kernel (tile shapes 0 and 2 of a small
solve) against the pass as a launch of its own (shapes 1 and 3): the same
operands in the same order, so every field agrees bit for bit, halo included.

Sizes: one tile over the whole panel (all four sides in one tile), a last tile
of one cell (its neighbour's halo reaches the panel edge), whole tiles only,
and remainders of both small shapes of each order.
"""
import numpy as np
import pytest

import cases
from mcv_sw_amd import capi

SIZES = [(3, 2), (3, 7), (3, 9), (3, 16), (3, 21), (4, 3), (4, 5), (4, 7), (4, 12), (4, 13)]
FORMS = [("RK4", capi.FP64), ("RK3_TVD", capi.FP64), ("RK4", capi.FP32C), ("RK3_TVD", capi.FP32C)]


def _solve(lib, dof, n, scheme, precision, tile, m, st):
    with capi.Solver(dof, n, 200.0, m, st, scheme=scheme, precision=precision, lib=lib) as s:
        s.set_tile(tile)
        s.step(1)
        s.step(3)  # the second call starts from a finished level
        return s.sync()


def _check(lib, dof, n, scheme, precision):
    m = cases.mesh(dof, n)
    st = cases.case5(m)
    ok = cases.masks(dof, n)["defined"]
    ref = _solve(lib, dof, n, scheme, precision, 1, m, st)
    for tile in (0, 2):
        out = _solve(lib, dof, n, scheme, precision, tile, m, st)
        for k in capi.STATE_FIELDS:
            assert np.array_equal(out[k][:, ok], ref[k][:, ok]), (tile, k)
        assert out["mass"] == ref["mass"] and out["energy"] == ref["energy"]


def _check_batch(lib):
    """Two solves of different stage counts, runs that end inside a step."""
    specs = [(3, 9, "RK3_TVD", capi.FP32C, 5), (4, 7, "RK4", capi.FP64, 4)]
    outs = []
    for tile in (2, 1):
        with capi.Batch(2, lib=lib) as b:
            slots = []
            for dof, n, scheme, precision, steps in specs:
                m = cases.mesh(dof, n)
                slots.append(b.add(dof, n, 200.0, m, cases.case5(m), steps, scheme=scheme,
                                   precision=precision))
            b.set_tile(tile)
            for stages in (1, 4, 13, 2):  # spent solves stay as they are
                b.run(stages)
            left, done = b.poll()
            assert list(left) == [0, 0] and list(done) == [5, 4]
            outs.append([b.sync(s) for s in slots])
    for (dof, n, *_), a, c in zip(specs, *outs):
        ok = cases.masks(dof, n)["defined"]
        for k in capi.STATE_FIELDS:
            assert np.array_equal(a[k][:, ok], c[k][:, ok]), (dof, k)


@pytest.mark.parametrize("scheme,precision", FORMS)
@pytest.mark.parametrize("dof,n", SIZES)
def test_emulated_side_tiles(emu_lib, dof, n, scheme, precision):
    _check(emu_lib, dof, n, scheme, precision)


def test_emulated_side_tiles_in_a_batch(emu_lib):
    _check_batch(emu_lib)


@pytest.mark.gpu
@pytest.mark.parametrize("scheme,precision", FORMS)
@pytest.mark.parametrize("dof,n", SIZES + [(3, 64), (4, 45)])
def test_gpu_side_tiles(hip_lib, dof, n, scheme, precision):
    print(f"[side tiles] dof={dof} n={n} {scheme} precision={precision}", flush=True)
    _check(None, dof, n, scheme, precision)


@pytest.mark.gpu
def test_gpu_side_tiles_in_a_batch(hip_lib):
    _check_batch(None)
