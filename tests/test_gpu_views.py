"""Host views of every extent against slices of the whole array: the part of a view inside the
block is moved, the rest of the view and of the block keeps its values.  Boxes of one cell, of the
interior, of a single row and plane, beyond the block on all sides, apart from the block; arrays of
one, seven and eighteen components (the last in more than one slab for a context of one block)."""
import ctypes as C

import numpy as np
import pytest

from trans_amd import capi, cases, solver
from trans_amd.solver import Solver

pytestmark = pytest.mark.gpu

NI, NJ, NK = 12, 7, 5
BOXES = [((-2, -2, -2), (NI + 2, NJ + 2, NK + 2)), ((1, 1, 1), (NI - 1, NJ - 1, NK - 1)), ((3, 2, 1), (3, 2, 1)),
         ((-2, 4, 2), (NI + 2, 4, 2)), ((-5, -4, -3), (NI + 6, NJ + 3, NK + 4)), ((2, -2, 0), (5, NJ + 2, 3)),
         ((NI + 3, 1, 1), (NI + 4, 2, 2))]


def _box(nc, lo, hi, fill):
    shp = tuple(h - l + 1 for l, h in zip(lo, hi))
    return np.asfortranarray(np.full(shp if nc == 1 else (nc,) + shp, fill))


def _cut(a, lo, hi, lo0=(-2, -2, -2)):
    return a[(Ellipsis,) + tuple(slice(l - z, h - z + 1) for l, h, z in zip(lo, hi, lo0))]


@pytest.mark.parametrize("lo,hi", BOXES)
def test_view_boxes(lo, hi):
    blocks, org, glob = cases.bump_channel(NI, NJ, NK)
    prm = solver.prepare_case(blocks, org, glob)
    sv = Solver(blocks, prm, ki=1)
    ilo = tuple(max(l, -2) for l in lo)
    ihi = tuple(min(h, n + 2) for h, n in zip(hi, (NI, NJ, NK)))
    inside = all(a <= b for a, b in zip(ilo, ihi))
    # eighteen components: a box against the whole array
    sv.iterate(1)
    whole = _box(18, (-2, -2, -2), (NI + 2, NJ + 2, NK + 2), 0.0)
    part = _box(18, lo, hi, -9.0)
    for a, at in ((whole, (-2, -2, -2)), (part, lo)):
        assert sv.lib.trans_hip_get_field(sv.ctx, 0, capi.FIELD_DQDXYZ, C.byref(capi.fview(a, at))) == 0
    want = np.full_like(part, -9.0)
    if inside:
        _cut(want, ilo, ihi, lo)[...] = _cut(whole, ilo, ihi)
    assert np.array_equal(part, want)
    rng = np.random.Generator(np.random.PCG64(3))
    full = {nm: np.asfortranarray(rng.random(blocks[0][nm].shape)) for nm in ("v", "pp", "wt0")}

    def state(arrays, at, call):
        s = capi.TransStateView()
        for nm, a in arrays.items():
            setattr(s, nm, capi.fview(a, at))
        assert call(sv.ctx, 0, C.byref(s)) == 0

    state(full, (-2, -2, -2), sv.lib.trans_hip_set_state)
    # read: the part inside the block, the view's other cells untouched
    got = {nm: _box(7 if a.ndim == 4 else 1, lo, hi, -9.0) for nm, a in full.items()}
    state(got, lo, sv.lib.trans_hip_get_state)
    for nm, a in got.items():
        want = np.full_like(a, -9.0)
        if inside:
            _cut(want, ilo, ihi, lo)[...] = _cut(full[nm], ilo, ihi)
        assert np.array_equal(a, want), nm
    # write: the block's cells inside the view, the others kept
    new = {nm: np.asfortranarray(rng.random(a.shape)) for nm, a in got.items()}
    state(new, lo, sv.lib.trans_hip_set_state)
    back = {nm: np.asfortranarray(np.zeros_like(a)) for nm, a in full.items()}
    state(back, (-2, -2, -2), sv.lib.trans_hip_get_state)
    for nm, a in back.items():
        want = full[nm].copy(order="F")
        if inside:
            _cut(want, ilo, ihi)[...] = _cut(new[nm], ilo, ihi, lo)
        assert np.array_equal(a, want), nm
    sv.close()


@pytest.mark.parametrize("size", [(33, 17, 9), (97, 81, 33)])
def test_state_through_pinned_pieces(size):
    """A whole state there and back: one piece of the pinned buffers, and many over several host
    threads with arrays that begin inside a piece."""
    blocks, org, glob = cases.bump_channel(*size)
    prm = solver.prepare_case(blocks, org, glob)
    sv = Solver(blocks, prm, ki=1)
    rng = np.random.Generator(np.random.PCG64(5))
    names = ("v", "pp", "t", "rmiu", "wt0", "wt1", "wt2")
    put = {nm: np.asfortranarray(rng.random(blocks[0][nm].shape)) for nm in names}
    got = {nm: np.asfortranarray(np.zeros_like(a)) for nm, a in put.items()}
    for arrays, call in ((put, sv.lib.trans_hip_set_state), (got, sv.lib.trans_hip_get_state)):
        s = capi.TransStateView()
        for nm, a in arrays.items():
            setattr(s, nm, capi.fview(a))
        assert call(sv.ctx, 0, C.byref(s)) == 0
    for nm in names:
        assert np.array_equal(put[nm], got[nm]), nm
    sv.close()
