"""The gradients and the face fluxes over bricks of rows (256 elements per workgroup, three
directions per launch) against the oracle at the sizes where the schedule can go wrong: planes
of exactly one workgroup, below and above the size from which a block is cut into bricks (2048
elements; of points first, then of cells), bricks of unequal height, the smallest block, several
blocks in one launch.  Flat plate, SST, MDCD + AUSMPW+, perturbed; bar as for the other residual
tests: 1e-12 (the operations are the oracle's, but for the device's pow and tanh)."""
import numpy as np
import pytest

from oracle.oracle import OracleCase
from trans_amd import capi, cases, solver
from trans_amd.solver import Solver

from helpers import interior, perturb, relerr

pytestmark = pytest.mark.gpu

SIZES = [(1, 6, 5, 4), (1, 17, 17, 5), (1, 50, 42, 4), (1, 50, 44, 5), (3, 140, 61, 4)]


@pytest.mark.parametrize("size", SIZES)
def test_residual_over_bricks(size):
    nblk, ni, nj, nk = size
    print(f"case: plate {size}, residual", flush=True)
    blocks, org, glob = cases.flat_plate(nblk=nblk, ni_total=ni, nj=nj, nk=nk, lo=4, hi=60 if nblk > 1 else ni)
    org.Kind_Spatial, org.Kind_Roe = 3, 3
    prm = solver.prepare_case(blocks, org, glob)
    perturb(blocks, prm, seed=29, turb=True)
    oc = OracleCase(blocks, prm)
    # device and oracle start from the oracle's boundary values, bit for bit
    oc.spectral_radius(1)
    oc.bc(1, -1)
    for n, b in enumerate(blocks):
        for nm in ("v", "pp", "t", "rmiu"):
            b[nm][...] = oc[n][nm]
    sv = Solver(blocks, prm, ki=1)
    oc.residual(1)
    sv.spectral_radius()
    sv.space()
    for n, b in enumerate(blocks):
        for field, key in ((capi.FIELD_DQDXYZ, "DQdxyz"), (capi.FIELD_D, "D")):
            e = relerr(interior(sv.get_field(n, field), b), interior(oc[n][key], b))
            assert np.all(e < 1e-12), (n, key, e)
    sv.close()
