"""Which grids the sweeps take, through the sizing call (trans_hip_footprint), which runs
trans_hip_create's own checks without a device."""
import ctypes as C

import pytest

from trans_amd import capi, cases, serving, solver

from stub_lib import events, stub  # noqa: F401


def _footprint(size, fp32):
    blocks, org, glob = cases.flat_plate(nblk=1, ni_total=33, nj=17, nk=4, lo=9, hi=33)
    prm = solver.prepare_case(blocks, org, glob, implicit_fp32=fp32)
    descs, keep = serving._descs(blocks)
    descs[0].ni, descs[0].nj, descs[0].nk = size
    descs[0].npatch = 0
    out = C.c_size_t()
    rc = capi.load_library().trans_hip_footprint(C.byref(prm), 1, descs, C.byref(out))
    return rc, out.value


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("size", [(33, 33, 4097), (25, 25, 6000), (4097, 33, 33), (700, 9, 700)])
def test_long_blocks_are_taken(size, fp32):
    """The wave sweeps hold packets of the lines along j, whose size follows the cells: a block
    that is long along k or i is no larger than any other, however many slots the hyperplanes of a
    march along j would have (beyond 2^29 of them the sweeps on those refuse it)."""
    n = [m - 1 for m in size]
    assert (sum(n) - 2) * n[0] * n[2] * 8 + 2 * 1024 * 8 >= 1 << 32
    rc, nbytes = _footprint(size, fp32)
    assert rc == 0
    cells = n[0] * n[1] * n[2]
    assert nbytes < 4000 * cells


def test_tuning_reports_the_sweep_that_runs(stub):
    """A wave addresses its tile's rows with 31-bit offsets: beyond about 144 000 points along j
    the sweeps run one launch per hyperplane, and the tuning says so."""
    blocks, org, glob = cases.flat_plate(nblk=1, ni_total=33, nj=17, nk=4, lo=9, hi=33)
    prm = solver.prepare_case(blocks, org, glob)
    descs, keep = serving._descs(blocks)
    descs[0].npatch = 0
    lib = capi.load_library()
    for nj, want in ((17, 1), (140_000, 1), (150_000, -2)):
        descs[0].ni, descs[0].nj, descs[0].nk = 4, nj, 4
        ctx, t = C.c_void_p(), capi.TransTuneEntry()
        assert lib.trans_hip_create(C.byref(prm), 1, descs, C.byref(ctx)) == 0
        for sweep in (None, 3, 1):
            if sweep:
                t = capi.TransTuneEntry(sweep, 1, 0, 0.0, 16, 16, 8)
                assert lib.trans_hip_set_tuning(ctx, C.byref(t)) == 0
            assert lib.trans_hip_get_tuning(ctx, C.byref(t)) == 0
            assert t.sweep == (want if want < 0 else sweep or want), (nj, sweep)
        lib.stub_reset()
        assert lib.trans_hip_lusgs_update(ctx, None) == 0
        names = [nm for what, nm, _ in events(lib) if what == "launch"]
        assert any("k_lusgs_wave" in nm for nm in names) == (want == 1)
        assert any("k_lusgs_wplane" in nm for nm in names) == (want == -2)
        lib.trans_hip_destroy(ctx)
