"""The wall distance keeps its speed however the points are spread.

With 485 000 cells and 30 000 panels, far-away points must not cost more than five times what the
evenly spread ones do (measured: the same; boxes of equal size made it nine to ten times).
"""
import time

import numpy as np
import pytest

from trans_amd import mesh

pytestmark = pytest.mark.gpu


def _best(cells, panels):
    best = np.inf
    for _ in range(10):
        t0 = time.perf_counter()
        mesh.wall_distance_device(cells, panels)
        best = min(best, time.perf_counter() - t0)
    return best


def test_far_points_do_not_slow_the_wall_distance():
    rng = np.random.Generator(np.random.PCG64(43))
    cells = rng.random((485_000, 3)) * np.array([3.0, 1.0, 0.5])
    panels = rng.random((30_000, 3)) * np.array([3.0, 0.0, 0.5])
    even = _best(cells, panels)
    for kind in ("cell", "cell and panel", "every 64th cell"):
        print(f"case: far {kind}", flush=True)
        c, p = cells.copy(), panels.copy()
        if kind == "every 64th cell":
            c[::64] *= 1e4
        else:
            c[77] = 1e4
            if "panel" in kind:
                p[77] = 1e4
        assert _best(c, p) < 5 * even, kind
