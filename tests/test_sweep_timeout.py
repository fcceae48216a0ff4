"""A sweep whose bounded wait expired is reported by the call that hands its results out."""
import pytest

from trans_amd import capi, cases, serving, solver
from trans_amd.solver import Solver, TransError

from stub_lib import events, stub  # noqa: F401


def _case():
    blocks, org, glob = cases.flat_plate(nblk=2, ni_total=33, nj=17, nk=4, lo=9, hi=25)
    org.CFL_Sub_start = org.CFL_Sub_end = 2.0
    org.CFL_Sub_step = 1
    return blocks, solver.prepare_case(blocks, org, glob)


CALLS = {
    "get_state": lambda sv, tmp: sv.get_state(1),
    "get_field": lambda sv, tmp: sv.get_field(0, capi.FIELD_D),
    "get_stats": lambda sv, tmp: sv.get_stats(0),
    "plane_integrals": lambda sv, tmp: sv.plane_integrals(0, 1, 1),
    "write_restart": lambda sv, tmp: sv.write_restart(0, 1, tmp / "r"),
    "write_stats": lambda sv, tmp: sv.write_stats(0, *[sv.blocks[0].arrays[n] for n in ("xc", "yc", "zc")], tmp / "s"),
    "write_tecplot": lambda sv, tmp: sv.write_tecplot(0, tmp / "t"),
    "sync": lambda sv, tmp: sv.sync(),
    "iterate": lambda sv, tmp: sv.iterate(1),
}


@pytest.mark.parametrize("how", ["eager", "replayed", "lusgs", "rk"])
@pytest.mark.parametrize("call", CALLS)
def test_expired_wait_is_reported_once(stub, tmp_path, call, how):
    blocks, prm = _case()
    sv = Solver(blocks, prm, ki=1)
    sv.stats_enable(1, 1)
    if how == "replayed":
        stub.stub_graphs(1)
        sv.set_iteration(100)  # past the ramps: captured
        sv.iterate(1, want_resid=False)
    stub.stub_expire(1)
    if how == "lusgs":
        assert sv.lib.trans_hip_lusgs_update(sv.ctx, None) == 0
    elif how == "rk":
        assert sv.lib.trans_hip_rk_update(sv.ctx, 1, None) == 0
    else:
        done = len(events(stub))
        sv.iterate(2, want_resid=False)
        assert any(nm == "graph" for _, nm, _ in events(stub)[done:]) == (how == "replayed")
    stub.stub_expire(0)
    with pytest.raises(TransError) as e:
        CALLS[call](sv, tmp_path)
    assert e.value.rc == capi.TRANS_ETIMEOUT
    assert not list(tmp_path.iterdir())  # no file of invalid results
    CALLS[call](sv, tmp_path)
    sv.close()


@pytest.mark.parametrize("norms", ["finite", "nan"])
@pytest.mark.parametrize("end", ["target", "limit", "cancel"])
def test_served_request_with_an_expired_wait_fails(stub, norms, end):
    blocks, prm = _case()
    srv = serving.Server(hbm_budget=1 << 36, max_active=2, chunk=5)
    stub.stub_expire(2 if norms == "nan" else 1)
    rid = srv.submit(blocks, prm, target_drop=1e-30 if end != "target" else 0.5, max_iter=5 if end != "cancel" else 50)
    if end == "cancel":
        srv.progress(wait=False)
        srv.cancel(rid)
    else:
        srv.run()
    st = srv.poll(rid)
    assert (st["state_name"], st["error"]) == ("failed", capi.TRANS_ETIMEOUT)
    srv.close()
