"""The wave LU-SGS sweeps in every form against the oracle and against the device's sweep with one
launch per hyperplane (mode -2), which shares no code with them.

Forms: the mean flow with k-omega (SST), the mean flow alone (Euler) and k-omega alone (a
Runge-Kutta stage); the FP64 and the FP32 operator; blocks whose cross sections fit a line march
and blocks where none does (the contraction of the multiply-adds alternates in the first); fewer
than 1024 tiles and 1024 of them (from which the FP32 sweeps keep more rows in flight).  Sizes: one
lane short of a tile, one tile, one lane more, two tiles and one lane, the shortest lines.

Bars as for the other sweeps: one update from identical inputs within 1e-12 with the norms' argmax
locations exact (FP64 operator), the FP32 operator's increment within 1e-5 of the FP64 one.  The
order of every sum is fixed, so that a repeated update gives the same bits.
"""
import numpy as np
import pytest

from oracle.oracle import OracleCase
from trans_amd import capi, cases, solver
from trans_amd.solver import Solver

from helpers import interior, perturb, relerr

pytestmark = pytest.mark.gpu

FORMS = ["sst", "euler", "rk"]
FITS = [(16, 12, 4), (17, 4, 5), (18, 13, 6), (34, 4, 9), (257, 4, 257)]
WIDE = [(34, 34, 34), (257, 12, 257)]  # no cross section of at most 1024 lines
SIZES = FITS + WIDE


def _case(form, size, seed=29):
    ni, nj, nk = size
    if form == "euler":
        blocks, org, glob = cases.bump_channel(ni, nj, nk)
    else:
        blocks, org, glob = cases.flat_plate(nblk=1, ni_total=ni, nj=nj, nk=nk, lo=9, hi=ni)
    if form == "rk":
        org.IF_RK = 1
        org.CFL_Sub_start = org.CFL_Sub_end = 0.8
    prm = solver.prepare_case(blocks, org, glob, device_geometry=True)
    perturb(blocks, prm, seed=seed, turb=form != "euler")
    # device and oracle start from the oracle's boundary values, bit for bit
    oc = OracleCase(blocks, prm)
    oc.spectral_radius(1)
    oc.bc(1, -1)
    for n, b in enumerate(blocks):
        for nm in ("v", "pp", "t", "rmiu"):
            b[nm][...] = oc[n][nm]
    return blocks, prm, oc


def _solver(blocks, prm, fp32, sweep):
    p = capi.TransParams.from_buffer_copy(prm)
    p.implicit_fp32 = fp32
    sv = Solver(blocks, p, ki=1)
    sv.set_tuning(sweep, 4, 0)
    assert sv.tuning()["sweep"] == sweep
    return sv


def _update(sv, form):
    sv.spectral_radius()
    sv.space()
    return sv.rk_update(1) if form == "rk" else sv.lusgs_update()


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("form", FORMS)
def test_one_update(form, size, fp32):
    print(f"case: {form} {size}, wave sweeps, fp32 operator {fp32}", flush=True)
    blocks, prm, oc = _case(form, size)
    v0 = [b["v"].copy() for b in blocks]
    sv = _solver(blocks, prm, fp32, 3)
    oc.residual(1)
    ores = oc.rk_update(1, 1) if form == "rk" else oc.lusgs_update(1)
    gres = _update(sv, form)
    comps = slice(0, 5) if form == "euler" else slice(0, 7)
    for n, b in enumerate(blocks):
        got, want = interior(sv.get_state(n)["v"], b)[comps], interior(oc[n]["v"], b)[comps]
        if fp32:
            o = interior(v0[n], b)[comps]
            assert np.all(relerr(got - o, want - o) < 1e-5), n
            continue
        assert np.all(relerr(got, want) < 1e-12), n
        for key in ("ima", "jma", "kma") + (() if form == "euler" else ("imk", "jmk", "kmk", "imo", "jmo", "kmo")):
            assert gres[n][key] == ores[n][key], (n, key)
    if not fp32:
        pl = _solver(blocks, prm, fp32, -2)
        pres = _update(pl, form)
        for n, b in enumerate(blocks):
            got, want = interior(sv.get_state(n)["v"], b)[comps], interior(pl.get_state(n)["v"], b)[comps]
            assert np.all(relerr(got, want) < 1e-12), (n, "hyperplanes")
            assert abs(gres[n]["drsa"] - pres[n]["drsa"]) <= 1e-12 * pres[n]["drsa"]
        pl.close()
    sv.close()


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("size", [(58, 21, 30), (257, 4, 257)] + WIDE)
@pytest.mark.parametrize("form", FORMS)
def test_updates_repeat_bit_for_bit(form, size, fp32):
    """However the tiles follow each other, and whichever edge values a tile has to wait for."""
    print(f"case: {form} {size}, repeated update, fp32 operator {fp32}", flush=True)
    blocks, prm, _ = _case(form, size, seed=31)
    sv = _solver(blocks, prm, fp32, 3)
    start = [sv.get_state(n) for n in range(len(blocks))]
    first = None
    for q in range(6):
        for n in range(len(blocks)):
            sv.set_state(n, start[n])
        norms = _update(sv, form)
        got = [(sv.get_state(n)["v"], sv.get_field(n, capi.FIELD_D)) for n in range(len(blocks))]
        if first is None:
            first = got, norms
            continue
        for n, b in enumerate(blocks):
            for x, y in zip(got[n], first[0][n]):
                assert np.array_equal(interior(x, b), interior(y, b)), (q, n)
        assert norms == first[1], q
    sv.close()


def test_long_blocks():
    """A block for which only the wave sweeps have a buffer: the same update as the line march
    along k, which holds a smaller one."""
    size = (25, 25, 6000)
    print(f"case: {size}, wave sweeps and line march along k", flush=True)
    ni, nj, nk = size
    blocks, org, glob = cases.bump_channel(ni, nj, nk)
    prm = solver.prepare_case(blocks, org, glob, device_geometry=True)
    perturb(blocks, prm, seed=37)
    out = []
    for sweep in (3, 2):
        sv = Solver(blocks, prm, ki=1)
        assert sv.tuning()["sweep"] == 3
        sv.set_tuning(sweep, 4, 0)
        sv.spectral_radius()
        sv.space()
        res = sv.lusgs_update()
        out.append((sv.get_state(0)["v"], res[0]["drsa"]))
        sv.close()
    b = blocks[0]
    assert np.all(relerr(interior(out[0][0], b)[:5], interior(out[1][0], b)[:5]) < 1e-12)
    assert abs(out[0][1] - out[1][1]) <= 1e-12 * out[1][1]
