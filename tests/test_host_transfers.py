"""Host transfers: what several host threads write, and what happens without host memory."""
import ctypes as C

import numpy as np
import pytest

from trans_amd import capi, cases, solver
from trans_amd.solver import Solver

from stub_lib import events, stub  # noqa: F401


def _solver(n=9):
    blocks, org, glob = cases.bump_channel(n, n, n)
    return Solver(blocks, solver.prepare_case(blocks, org, glob), ki=1)


def _views(lib):
    return sum(what == "launch" and "k_view" in nm for what, nm, _ in events(lib))


def test_views_of_one_array_are_filled_in_order(stub):
    """Two arrays of a read-back into the same host array: the later one stays, however long the
    copies of the earlier one take (a host that does not want the history may aim it anywhere)."""
    sv = _solver(45)  # several pieces per array, so that several threads take part
    b = sv.blocks[0]
    one = np.zeros((7,) + b.shape(), order="F")

    def read(**views):
        s = capi.TransStateView()
        for nm, a in views.items():
            setattr(s, nm, capi.fview(a))
        assert sv.lib.trans_hip_get_state(sv.ctx, 0, C.byref(s)) == 0

    # (the stand-in fills the boxes of a read-back with their numbers)
    stub.stub_reset()
    read(v=one)
    first = _views(stub)
    stub.stub_reset()
    read(v=one, wt0=one)
    second = _views(stub)
    stub.stub_reset()
    stub.stub_slow_value(1)  # the copies of the first box are late
    read(v=one, wt0=one, wt1=one)
    assert one.min() > second
    # arrays that overlap in part
    long = np.zeros(2 * one.size)
    half, shift = one.size, one.size // 3

    def at(o):
        return long[o:o + half].reshape(one.shape, order="F")
    stub.stub_reset()
    stub.stub_slow_value(1)
    read(v=at(0), wt0=at(shift))
    assert long[:shift].max() <= first and long[shift:shift + half].min() > first
    # and side by side in one allocation
    stub.stub_reset()
    stub.stub_slow_value(1)
    read(v=at(0), wt0=at(half))
    assert 0 < long[:half].min() and long[:half].max() <= first and long[half:].min() > first
    sv.close()
