"""GPU parity of the wave LU-SGS sweeps (tiles of 16 x 4 lines, one wave each) against the oracle
at the sizes where a tile can go wrong.

Cells along i of 15, 16, 17 and 33 (one lane short of a tile, one tile, one lane more, two tiles
and one lane), along k of 3, 4, 5 and 8, lines of 3 cells (the shortest, where no row has all its
lanes) and longer ones of odd and even length, blocks of different sizes in one launch; both
operator precisions; and 1024 tiles, from which the FP32 sweeps keep more rows in flight.  Bars,
as for the other sweeps: one update within 1e-12 with the norms' argmax locations exact (FP64
operator), the FP32 operator's increment within 1e-5 of the FP64 one.
"""
import numpy as np
import pytest

from oracle.oracle import OracleCase
from trans_amd import capi, cases, solver
from trans_amd.solver import Solver

from helpers import interior, perturb, relerr

pytestmark = pytest.mark.gpu

SIZES = [  # blocks, points along i (all blocks), j, k
    (1, 16, 12, 4), (1, 17, 4, 5), (1, 18, 13, 6), (1, 34, 4, 9), (3, 58, 21, 6), (1, 257, 4, 257)]


@pytest.mark.parametrize("fp32", [0, 1])
@pytest.mark.parametrize("size", SIZES)
def test_wave_sweep_edges(size, fp32):
    nblk, ni, nj, nk = size
    print(f"case: plate {size}, wave sweeps, fp32 operator {fp32}", flush=True)
    blocks, org, glob = cases.flat_plate(nblk=nblk, ni_total=ni, nj=nj, nk=nk, lo=9, hi=30 if nblk > 1 else ni)
    prm = solver.prepare_case(blocks, org, glob, device_geometry=True)
    perturb(blocks, prm, seed=23, turb=True)
    oc = OracleCase(blocks, prm)
    # device and oracle start from the oracle's boundary values, bit for bit
    oc.spectral_radius(1)
    oc.bc(1, -1)
    for n, b in enumerate(blocks):
        for nm in ("v", "pp", "t", "rmiu"):
            b[nm][...] = oc[n][nm]
    v0 = [b["v"].copy() for b in blocks]
    p = capi.TransParams.from_buffer_copy(prm)
    p.implicit_fp32 = fp32
    sv = Solver(blocks, p, ki=1)
    sv.set_tuning(3, 4, 0)
    oc.residual(1)
    sv.spectral_radius()
    sv.space()
    ores = oc.lusgs_update(1)
    gres = sv.lusgs_update()
    for n, b in enumerate(blocks):
        got, want = interior(sv.get_state(n)["v"], b), interior(oc[n]["v"], b)
        if fp32:
            o = interior(v0[n], b)
            assert np.all(relerr(got - o, want - o) < 1e-5), n
            continue
        assert np.all(relerr(got, want) < 1e-12), n
        for key in ("ima", "jma", "kma", "imk", "jmk", "kmk", "imo", "jmo", "kmo"):
            assert gres[n][key] == ores[n][key], (n, key)
    sv.close()
