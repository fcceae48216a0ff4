"""A sweep whose buffers cannot be allocated leaves a context that can go on."""
import pytest

from trans_amd import capi, cases, solver
from trans_amd.solver import Solver, TransError

from stub_lib import events, stub  # noqa: F401


def _solver():
    blocks, org, glob = cases.flat_plate(nblk=2, ni_total=33, nj=17, nk=4, lo=9, hi=25)
    return Solver(blocks, solver.prepare_case(blocks, org, glob), ki=1)


@pytest.mark.parametrize("sweep,allocations", [(3, 4), (0, 1), (2, 1), (-2, 1), (-3, 1)])
def test_failed_allocation_leaves_the_hyperplane_sweep(stub, sweep, allocations):
    """Whichever allocation of a sweep fails, the call says so and the context falls back to the
    sweep that needs no buffer, instead of launching on buffers that are not there."""
    for n in range(allocations):
        sv = _solver()
        if sweep == 3:  # from the other state of the plain schedule
            sv.set_tuning(-3, 1, 0)
        stub.stub_reset()
        stub.stub_fail_malloc(n)
        with pytest.raises(TransError) as e:
            sv.set_tuning(sweep, 1, 0)
        assert e.value.rc == capi.TRANS_ENOMEM, n
        assert sv.tuning()["sweep"] == -1, n
        stub.stub_fail_malloc(-1)
        done = len(events(stub))
        sv.iterate(2)
        names = {nm for what, nm, _ in events(stub)[done:] if what == "launch"}
        assert any("k_lusgs_sweep" in nm for nm in names), n
        assert not any(k in nm for nm in names for k in ("_wave", "_wplane", "_line", "_rhs_w", "unskew")), names
        sv.set_tuning(sweep, 1, 0)  # with memory, the sweep asked for
        assert sv.tuning()["sweep"] == sweep
        stub.stub_reset()
        sv.iterate(1)
        assert not any("k_lusgs_sweep" in nm for what, nm, _ in events(stub) if what == "launch")
        sv.close()


def test_failed_allocations_free_what_they_took(stub):
    sv = _solver()
    sv.set_tuning(-1, 1, 0)
    before = stub.stub_mapped()
    for n in range(4):
        stub.stub_fail_malloc(n)
        with pytest.raises(TransError):
            sv.set_tuning(3, 1, 0)
        assert stub.stub_mapped() == before
    sv.close()


def test_refused_configuration_changes_nothing(stub):
    blocks, org, glob = cases.flat_plate(nblk=1, ni_total=70, nj=35, nk=34, lo=9, hi=70)  # no axis fits a line march
    sv = Solver(blocks, solver.prepare_case(blocks, org, glob), ki=1)
    for keep in ((-3, 1, 0), (3, 4, 1), (-2, 1, 0)):
        sv.set_tuning(*keep)
        stub.stub_reset()
        sv.iterate(1)
        was = sv.tuning()
        launches = events(stub)
        for bad in ((3, 2, 0), (5, 1, 0), (0, 1, 0), (1, 4, 0), (3, 4, 0, 0, 1, 8)):
            with pytest.raises(TransError) as e:
                sv.set_tuning(*bad)
            assert e.value.rc == capi.TRANS_EINVAL
            assert sv.tuning() == was, (keep, bad)
            stub.stub_reset()
            sv.iterate(1)
            assert [x[:2] for x in events(stub) if x[0] == "launch"] == [x[:2] for x in launches if x[0] == "launch"]
    sv.close()
