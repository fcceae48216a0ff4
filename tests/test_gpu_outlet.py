"""The outlet's pressure march against the oracle: with reciprocals known beforehand, and with
divisions where a quotient could underflow (a hub pressure of 1e-120).  Bar: 1e-12 relative in
every outlet ghost; a step rounds about ten times, the lines have fewer than 200 steps, and the
device's sine and cosine enter through the small radial increments only."""
import numpy as np
import pytest

from oracle.oracle import OracleCase
from trans_amd import cases, solver
from trans_amd.solver import Solver

from helpers import perturb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pouthub", [None, 1e-120])
@pytest.mark.parametrize("case", ["sector", "plate"])
def test_outlet_march(case, pouthub):
    print(f"case: {case}, outlet march from {pouthub}", flush=True)
    if case == "sector":
        blocks, org, glob = cases.compressor_sector(scale=1 / 8)
    else:
        blocks, org, glob = cases.flat_plate(nblk=1, ni_total=20, nj=161, nk=4, lo=9, hi=20)
    prm = solver.prepare_case(blocks, org, glob)
    if pouthub is not None:
        prm.pouthub = pouthub
    perturb(blocks, prm, seed=31, turb=True)
    oc = OracleCase(blocks, prm)
    sv = Solver(blocks, prm, ki=1)
    oc.spectral_radius(1)
    oc.bc(1, -1)
    sv.spectral_radius()
    sv.bc(-1)
    seen = 0
    for n, b in enumerate(blocks):
        st = sv.get_state(n)
        for q in b.patches:
            if q["bctype"] != 7:
                continue
            lo = [q["point_start"][d] + q["ceijkadd"][d] for d in range(3)]
            hi = [q["point_end"][d] + q["ceijkadd"][d] for d in range(3)]
            cut = tuple(slice(l + 2, h + 3) for l, h in zip(lo, hi))
            for a, o in ((st["pp"], oc[n]["pp"]), (st["t"], oc[n]["t"]), (st["v"][0], oc[n]["v"][0])):
                assert np.all(np.abs(a[cut] - o[cut]) <= 1e-12 * np.abs(o[cut])), (n, np.max(np.abs(a[cut] / o[cut] - 1)))
                seen += a[cut].size
    assert seen
    sv.close()
