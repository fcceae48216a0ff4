"""Work on the helper stream is waited for, whatever a call returns: with a launch that fails
anywhere in an iteration, the context's stream still waits for everything queued on the helper
stream before the call comes back."""
import pytest

from trans_amd import cases, solver
from trans_amd.solver import Solver, TransError

from stub_lib import events, stub  # noqa: F401


def _unjoined(ev, main):
    """Launches on streams other than `main` that `main` has not waited for."""
    open_, recorded = {}, {}
    for n, (what, name, s) in enumerate(ev):
        if what == "launch" and s != main:
            open_[n] = s
        elif what == "record":
            recorded[name] = [q for q, st in open_.items() if st == s]
        elif what == "wait" and s == main:
            for q in recorded.get(name, ()):
                open_.pop(q, None)
    return [ev[q][1] for q in open_]


def _case(kind):
    if kind == "sector":  # inlet and outlet: the outlet march runs on the helper stream
        blocks, org, glob = cases.compressor_sector(scale=1 / 16)
    else:
        blocks, org, glob = cases.flat_plate(nblk=2, ni_total=33, nj=17, nk=4, lo=9, hi=25)
    return blocks, solver.prepare_case(blocks, org, glob)


@pytest.mark.parametrize("kind", ["sector", "plate"])
@pytest.mark.parametrize("call", ["residual", "space", "iterate"])
def test_failed_launch_leaves_nothing_unordered(stub, kind, call):
    blocks, prm = _case(kind)
    sv = Solver(blocks, prm, ki=1)
    go = (lambda: sv.iterate(1, want_resid=False)) if call == "iterate" else getattr(sv, call)
    stub.stub_reset()
    go()
    launches = [(name, s) for what, name, s in events(stub) if what == "launch"]
    main = next(s for name, s in launches if "k_prim_ghost" in name)
    assert any(s != main for _, s in launches)
    assert not _unjoined(events(stub), main)
    for q in range(len(launches)):
        stub.stub_reset()
        stub.stub_fail_launch(q)
        with pytest.raises(TransError):
            go()
        assert not _unjoined(events(stub), main), q
    stub.stub_reset()
    sv.close()
