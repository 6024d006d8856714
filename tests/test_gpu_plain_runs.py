"""Plain scheme: long runs replay captured iterations, short ones are launched;
any mix of lengths gives the bits of single iterations."""
import numpy as np
import pytest
# torch before the library: one HIP runtime in the process
import torch  # noqa: F401

from effplast2d_amd import EffPlast2D
from tests.pairs import PLASTIC_FIELDS, STATE_FIELDS, STRESS_FIELDS, make_pa, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nX,nl", [(8, 1), (33, 3), (64, 1), (65, 3)])
def test_plain_runs_equal_single_iterations(nX, nl):
    print(f"plain runs nX={nX} nl={nl}", flush=True)
    pa = make_pa(nX, nPores=1, porosity=0.02)
    init = random_state(nX, 7 + nX, pa=pa, boundary_v=True)

    def run(steps):
        with EffPlast2D(pa, nX, nTasks=nl, mode="plain") as g:
            for k in STATE_FIELDS:
                g.set(k, init[k])
            for n in steps:
                g.iterate(n)
            return {k: g.get(k) for k in STATE_FIELDS + STRESS_FIELDS +
                    (PLASTIC_FIELDS if nl > 1 else [])}

    a = run((199, 49, 50, 1, 101, 250))
    b = run((25,) * 26)     # never as long as a captured run
    for k in a:
        assert np.array_equal(a[k], b[k], equal_nan=True), k
