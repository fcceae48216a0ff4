"""The wall distance over sorted cells and panels against every cell against every panel on the
host, bit for bit: sizes around the line from which it is used and around whole waves and tiles,
panels in one plane, on one line and in one point, clustered and far-away cells, cells on panels,
coordinates that are not finite."""
import numpy as np
import pytest

from trans_amd import mesh

pytestmark = pytest.mark.gpu


def _host(cells, panels):
    out = np.empty(len(cells))
    for a in range(0, len(cells), 512):
        c = cells[a:a + 512]
        with np.errstate(all="ignore"):
            dx, dy, dz = (c[:, None, d] - panels[None, :, d] for d in range(3))
            q = dx * dx + dy * dy + dz * dz
        q = np.where(np.isnan(q), np.inf, q).min(axis=1)
        out[a:a + 512] = np.sqrt(np.maximum(np.minimum(q, 1e20), 1e-20))
    return out


@pytest.mark.parametrize("kind", ["cloud", "plane", "line", "point", "clusters", "nonfinite"])
@pytest.mark.parametrize("ncell,npanel", [(4095, 2048), (4096, 2047), (4096, 2048), (4097, 2111), (5003, 2049)])
def test_sorted_wall_distance(ncell, npanel, kind):
    rng = np.random.Generator(np.random.PCG64(41))
    cells = rng.random((ncell, 3)) * np.array([3.0, 1.0, 0.5])
    panels = rng.random((npanel, 3)) * np.array([3.0, 1.0, 0.5])
    if kind == "plane":
        panels[:, 1] = 0.25
    elif kind == "line":
        panels[:, 1:] = 0.0
    elif kind == "point":
        panels[:] = panels[0]
    elif kind == "clusters":
        panels[: npanel // 2] = panels[: npanel // 2] * 1e-3 + 7.0
        cells[::5] = cells[::5] * 1e-4 + 7.0
        cells[1::7] *= 1e12
        cells[3::11] = panels[rng.integers(0, npanel, len(cells[3::11]))]
    elif kind == "nonfinite":
        panels[7, 1] = np.inf
        panels[9] = np.nan
        cells[11, 0] = np.nan
        cells[13, 2] = -np.inf
    assert np.array_equal(mesh.wall_distance_device(cells, panels), _host(cells, panels))
