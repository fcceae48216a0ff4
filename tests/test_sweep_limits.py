"""Which grids the sweeps take, through the sizing call (trans_hip_footprint), which runs
trans_hip_create's own checks without a device."""
import ctypes as C

import pytest

from trans_amd import capi, cases, serving, solver


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
