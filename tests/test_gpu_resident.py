"""Resident runs: 16 iterations and more of a handle on the automatic shape, on
a grid whose tiles fit the GPU together, run in one launch with the state in
registers.  They evaluate the tile kernel's expressions in the same order, so
every field equals the tile kernel's bit for bit (no tolerance), in FP64 and in
the split scheme."""
import sys

import numpy as np
import pytest
# torch before the library: one HIP runtime in the process
import torch

from effplast2d_amd import EffPlast2D
from tests.pairs import PLASTIC_FIELDS, STATE_FIELDS, STRESS_FIELDS, make_pa, random_state

pytestmark = pytest.mark.gpu


def _note(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def _init(nX, mode, pa, seed):
    init = random_state(nX, seed, pa=pa, boundary_v=True)
    if mode == "split":
        for k in ("Vx", "Vy"):
            init[k] = init[k].astype(np.float32).astype(np.float64)
    return init


def _run(nX, mode, nl, pa, init, steps, **kw):
    with EffPlast2D(pa, nX, nTasks=nl, mode=mode, **kw) as g:
        for k in STATE_FIELDS:
            g.set(k, init[k])
        for n in steps:
            g.iterate(n)
        name = g.timing()[2]
        return {k: g.get(k) for k in STATE_FIELDS + STRESS_FIELDS +
                (PLASTIC_FIELDS if nl > 1 else [])}, name


def _same(a, b):
    for k in a:
        assert np.array_equal(a[k], b[k], equal_nan=True), \
            f"{k}: {np.count_nonzero(a[k] != b[k])} differ"


# one tile; strips and bands one node short of, at and past a tile's width (60
# or 56 columns and 8, 24 or 44 rows, the first and last tiles a few more); the
# largest grids of each tile shape, and the smallest grid of the next
@pytest.mark.parametrize("mode,nX", [(m, n) for m in ("fp64", "split")
                                     for n in (16, 17, 31, 62, 63, 64, 115, 116, 125, 333)] +
                         [("fp64", n) for n in (448, 560, 672, 768)] +
                         [("split", n) for n in (448, 449, 560)])
def test_resident_equals_tiles(mode, nX):
    _note(f"resident {mode} nX={nX}")
    pa = make_pa(nX, nPores=1 + nX % 3, porosity=0.03)
    init = _init(nX, mode, pa, 900 + nX)
    for nl, steps in ((3, (17, 16)), (1, (24,))):
        a, name = _run(nX, mode, nl, pa, init, steps)
        assert "k_resident" in name, name
        b, _ = _run(nX, mode, nl, pa, init, steps, tileRows=8)
        _same(a, b)


@pytest.mark.parametrize("mode", ["fp64", "split"])
def test_short_and_long_runs_mix(mode):
    """Runs below the resident length take the chains, closed by the tile
    kernel; any mix of lengths gives the bits of single iterations."""
    nX = 130
    _note(f"resident mix {mode}")
    pa = make_pa(nX, nPores=2, porosity=0.02)
    init = _init(nX, mode, pa, 31)
    steps = (1, 16, 2, 3, 4, 5, 15, 33, 1, 20)
    a, _ = _run(nX, mode, 3, pa, init, steps)
    b, _ = _run(nX, mode, 3, pa, init, (sum(steps),), tileRows=8)
    _same(a, b)


def test_pore_moduli_nan_and_infinity():
    """A NaN and an infinity in U spread as in the tile kernel (the edge tiles
    read no node outside the grid into it)."""
    nX = 125
    _note("resident nan")
    pa = make_pa(nX, nPores=2, porosity=0.03)
    for mode in ("fp64", "split"):
        init = _init(nX, mode, pa, 77)
        init["Ux"][40 * (nX + 1) + 59] = np.nan
        init["Uy"][90 * nX + 60] = np.inf
        a, _ = _run(nX, mode, 3, pa, init, (16,))
        b, _ = _run(nX, mode, 3, pa, init, (16,), tileRows=8)
        _same(a, b)


@pytest.mark.parametrize("mode,nX", [("fp64", 512), ("split", 333)])
def test_two_handles_at_once(mode, nX):
    """Two handles whose tiles do not find room together: a run that is turned
    away leaves the state alone and its iterations take the other kernels, so
    both handles end with the bits of a handle alone."""
    _note(f"resident two handles {mode}")
    pa = make_pa(nX, nPores=2, porosity=0.03)
    inits = [_init(nX, mode, pa, 5 + k) for k in range(3)]
    alone = [_run(nX, mode, 3, pa, i, (200, 100), tileRows=8)[0] for i in inits]
    hs = [EffPlast2D(pa, nX, nTasks=3, mode=mode) for _ in inits]
    try:
        for h, i in zip(hs, inits):
            for k in STATE_FIELDS:
                h.set(k, i[k])
        for n in (200, 100):
            for h in hs:       # launched side by side, on three streams
                h.iterate(n)
        for h, ref in zip(hs, alone):
            _same({k: h.get(k) for k in ref}, ref)
    finally:
        for h in hs:
            h.close()


def test_callers_stream_and_capture():
    """On a caller's stream the iterations stay on the tile kernel: a captured
    run of an even number of them replays on the buffers that eager runs
    between the replays leave current."""
    nX, n = 96, 32
    _note("captured run on a caller's stream")
    pa = make_pa(nX, nPores=1, porosity=0.02)
    init = _init(nX, "fp64", pa, 3)
    ref, _ = _run(nX, "fp64", 3, pa, init, (n, n, n, n), tileRows=8)
    st = torch.cuda.Stream()
    with EffPlast2D(pa, nX, nTasks=3, mode="fp64", stream=st.cuda_stream) as g:
        for k in STATE_FIELDS:
            g.set(k, init[k])
        g.iterate(n)
        g.sync()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st):
            g.iterate(n)
        graph.replay()
        torch.cuda.synchronize()
        g.iterate(n)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _same({k: g.get(k) for k in ref}, ref)
