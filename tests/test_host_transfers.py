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


@pytest.mark.parametrize("call", ["get_state", "set_state", "get_field"])
def test_no_host_memory_is_an_error_code(stub, call):
    """Wherever host memory runs out in a transfer (lists, gather buffers, threads), the call
    returns TRANS_ENOMEM, every thread has ended and the pinned buffers are back."""
    sv = _solver(45)
    b = sv.blocks[0]
    # views of wider arrays, so that rows are gathered and scattered on the host
    wide = tuple(n + 2 for n in b.shape())
    host = {nm: np.zeros((nc,) + wide if nc > 1 else wide, order="F") for nm, nc in (("v", 7), ("pp", 1), ("wt0", 7))}
    s = capi.TransStateView()
    for nm, a in host.items():
        setattr(s, nm, capi.fview(a, lo=(-3, -3, -3)))

    def go():
        if call == "get_field":
            return sv.lib.trans_hip_get_field(sv.ctx, 0, capi.FIELD_D, C.byref(s.v))
        return getattr(sv.lib, "trans_hip_" + call)(sv.ctx, 0, C.byref(s))
    assert go() == 0
    pinned = stub.stub_mapped()
    n = 0
    while True:
        stub.stub_fail_new(n)
        rc = go()
        left = stub.stub_new_left()
        stub.stub_fail_new(-1)
        assert rc in (0, capi.TRANS_ENOMEM), (n, rc)
        if left > 0:  # more than the call needs
            assert rc == 0
            break
        n += 1
    assert n > 5  # (the first attempts had failed)
    assert go() == 0
    assert stub.stub_mapped() == pinned
    sv.close()
