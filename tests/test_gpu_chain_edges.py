"""Chain kernels where a strip's or a segment's edge meets the grid's: every
field equals the tile kernel's bit for bit (no tolerance), plastic and elastic
(interior segments have code of their own for each), with a NaN and an infinity
beside the boundary too."""
import numpy as np
import pytest
# torch before the library: one HIP runtime in the process
import torch  # noqa: F401

from effplast2d_amd import EffPlast2D
from tests.pairs import PLASTIC_FIELDS, STATE_FIELDS, STRESS_FIELDS, make_pa, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp64", "split"])
@pytest.mark.parametrize("nX", [108, 109, 167, 216, 217])
def test_chain_edges_equal_tiles(mode, nX):
    pa = make_pa(nX, nPores=2, porosity=0.02)
    init = random_state(nX, 40 + nX, pa=pa, boundary_v=True)
    if mode == "split":
        for k in ("Vx", "Vy"):
            init[k] = init[k].astype(np.float32).astype(np.float64)

    def run(nl, state, **kw):
        with EffPlast2D(pa, nX, nTasks=nl, mode=mode, **kw) as g:
            for k in STATE_FIELDS:
                g.set(k, state[k])
            g.iterate(9)
            return {k: g.get(k) for k in STATE_FIELDS + STRESS_FIELDS +
                    (PLASTIC_FIELDS if nl > 1 else [])}

    odd = {k: v.copy() for k, v in init.items()}
    odd["Ux"][2 * (nX + 1) + 1] = np.nan
    odd["Uy"][(nX - 2) * nX + nX - 2] = np.inf
    for nl, state in ((3, init), (1, init), (3, odd)):
        ref = run(nl, state, tileRows=8)
        for kw in ({"itersPerLaunch": 4, "stageWaves": 2}, {"itersPerLaunch": 3, "stageWaves": 2},
                   {"itersPerLaunch": 4, "stageWaves": 1}, {"itersPerLaunch": 2}):
            for rows in (1, 7, 30):
                print(f"chain edges {mode} nX={nX} nl={nl} {kw} rows={rows}", flush=True)
                a = run(nl, state, marchRows=rows, **kw)
                for k in ref:
                    assert np.array_equal(a[k], ref[k], equal_nan=True), (nl, kw, rows, k)
