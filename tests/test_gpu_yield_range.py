"""FP64 return mapping over the range of its arguments: the chain and resident
kernels' root and quotient (used where the yield radius lies in 2^-300 .. 2^300)
against the tile kernel's library ones, bit for bit.  State and radius are scaled
together, up to squared invariants that overflow."""
import numpy as np
import pytest
# torch before the library: one HIP runtime in the process
import torch  # noqa: F401

from effplast2d_amd import EffPlast2D
from tests.pairs import PLASTIC_FIELDS, STATE_FIELDS, STRESS_FIELDS, make_pa, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("exponent", [-330, -290, -100, 0, 100, 290, 310, 500, 520])
def test_yield_factor_over_the_range(exponent):
    nX = 125
    print(f"yield range 2^{exponent}", flush=True)
    pa = make_pa(nX, nPores=2, porosity=0.03)
    init = random_state(nX, 11, pa=pa, boundary_v=True)
    f = 2.0 ** exponent
    pa = pa.copy()
    pa[8] *= f
    for k in STATE_FIELDS:
        init[k] = init[k] * f

    def run(**kw):
        with EffPlast2D(pa, nX, nTasks=3, mode="fp64", **kw) as g:
            for k in STATE_FIELDS:
                g.set(k, init[k])
            g.iterate(17)
            return {k: g.get(k) for k in STATE_FIELDS + STRESS_FIELDS + PLASTIC_FIELDS}

    ref = run(tileRows=8)
    for kw in ({}, {"marchRows": 20, "itersPerLaunch": 4, "stageWaves": 2},
               {"marchRows": 20, "itersPerLaunch": 3, "stageWaves": 1},
               {"marchRows": 20, "itersPerLaunch": 2}):
        a = run(**kw)
        for k in ref:
            assert np.array_equal(a[k], ref[k], equal_nan=True), (kw, k)
