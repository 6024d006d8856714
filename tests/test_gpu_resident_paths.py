"""Which path the iterations of a handle on the automatic shape took: resident
runs are counted by their outcome, so a run that was meant to be resident is
seen to be one, and the paths a busy device takes are forced from the host (a
launch that may not wait for its workgroups).  Every path gives the tile
kernel's bits (no tolerance)."""
import threading
import time

import numpy as np
import pytest
# torch before the library: one HIP runtime in the process
import torch  # noqa: F401

from effplast2d_amd import Batch, EffPlast2D, Ep2dError
from tests.pairs import PLASTIC_FIELDS, STATE_FIELDS, STRESS_FIELDS, make_pa, random_state

pytestmark = pytest.mark.gpu

FIELDS = STATE_FIELDS + STRESS_FIELDS + PLASTIC_FIELDS


def _case(nX, mode, seed):
    pa = make_pa(nX, nPores=1 + nX % 3, porosity=0.03)
    init = random_state(nX, seed, pa=pa, boundary_v=True)
    if mode == "split":
        for k in ("Vx", "Vy"):
            init[k] = init[k].astype(np.float32).astype(np.float64)
    return pa, init


def _start(g, init):
    for k in STATE_FIELDS:
        g.set(k, init[k])


def _same(a, b):
    for k in a:
        assert np.array_equal(a[k], b[k], equal_nan=True), \
            f"{k}: {np.count_nonzero(a[k] != b[k])} differ"


def _tiles(nX, mode, pa, init, n):
    with EffPlast2D(pa, nX, nTasks=3, mode=mode, tileRows=8) as g:
        _start(g, init)
        g.iterate(n)
        return {k: g.get(k) for k in FIELDS}


# the smallest and largest grid of each tile shape, on 256 CUs
@pytest.mark.parametrize("mode,nX", [("fp64", 16), ("fp64", 336), ("fp64", 448), ("fp64", 560),
                                     ("fp64", 672), ("fp64", 792), ("split", 16), ("split", 392),
                                     ("split", 448), ("split", 560)])
def test_long_runs_are_resident(mode, nX):
    print(f"resident {mode} nX={nX}", flush=True)
    pa, init = _case(nX, mode, 50 + nX)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        for n in (16, 15, 40):      # the second takes the chains
            g.iterate(n)
        assert g.diag_resident() == (2, 0, 0)


@pytest.mark.parametrize("mode,nX", [("fp64", 64), ("split", 333), ("fp64", 500)])
def test_runs_that_may_not_start(mode, nX):
    """A launch that finds no time for its workgroups leaves the state alone; its
    iterations take the chains, and so do the runs after it."""
    print(f"late start {mode} nX={nX}", flush=True)
    pa, init = _case(nX, mode, 7 + nX)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        g.diag_resident(arrive_ticks=0)
        for n in (33, 16, 18):
            g.iterate(n)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (0, 1, 0)
    _same(a, _tiles(nX, mode, pa, init, 67))


@pytest.mark.parametrize("mode", ["fp64", "split"])
def test_runs_of_several_launches(mode):
    """One call of more than 65536 iterations is several launches."""
    nX, n = 17, 2 * 65536 + 21
    print(f"long run {mode}", flush=True)
    pa, init = _case(nX, mode, 3)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        g.iterate(n)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (3, 0, 0)
    _same(a, _tiles(nX, mode, pa, init, n))


@pytest.mark.parametrize("mode", ["fp64", "split"])
def test_exchange_numbers_start_again(mode):
    """The 32 bits that count the exchanges run out: the buffer is cleared and
    the count starts again."""
    nX = 125
    print(f"exchange numbers {mode}", flush=True)
    pa, init = _case(nX, mode, 9)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        g.diag_resident(tag=2 ** 32 - 1 - 150)
        for n in (64, 64, 64, 64):
            g.iterate(n)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (4, 0, 0)
    _same(a, _tiles(nX, mode, pa, init, 256))


# grids below 16, between and beyond the resident shapes' ranges, up to the
# largest that takes the shortest segments of one round
@pytest.mark.parametrize("mode,nX", [(m, n) for m in ("fp64", "split") for n in (8, 9, 15)] +
                         [("fp64", n) for n in (337, 447, 561, 671, 793, 900, 1023, 1024)] +
                         [("split", n) for n in (393, 447, 561, 700, 900, 1023, 1024)])
def test_automatic_chains_equal_tiles(mode, nX):
    """Without a resident shape the automatic shape is a chain on segments of a
    computed height, with closing launches of as few rows."""
    print(f"automatic chains {mode} nX={nX}", flush=True)
    pa, init = _case(nX, mode, 11 + nX)
    steps = (21, 4, 3, 2, 1, 16)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        for n in steps:
            g.iterate(n)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (0, 0, 0)
    _same(a, _tiles(nX, mode, pa, init, sum(steps)))


@pytest.mark.parametrize("mode,nX", [("fp64", 500), ("split", 500)])
def test_a_run_that_did_not_start_is_no_sample(mode, nX):
    """Its iterations are timed where they ran, on the chains: as many samples
    as a run on the chains gives, and their name."""
    print(f"timing of a late start {mode}", flush=True)
    pa, init = _case(nX, mode, 21)

    def run(n, calls, late):
        with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
            _start(g, init)
            if late:
                g.diag_resident(arrive_ticks=0)
            g.set_timing(1)
            for _ in range(calls):
                g.iterate(n)
            return g.timing()

    # 401 iterations: 100 four-iteration launches and one on its own
    ms, n, name = run(401, 1, True)
    assert n == 401 and "k_chain" in name, (ms, n, name)
    ms, n, name = run(401, 3, False)
    assert n == 3 * 401 and "k_resident" in name, (ms, n, name)
    # short runs: 3 four-iteration launches, a closing one of two (not
    # sampled) and one on its own
    ms, n, name = run(15, 2, False)
    assert n == 2 * 13 and "k_chain" in name, (ms, n, name)
    ms, n, name = run(1, 3, False)
    assert n == 3 and "k_fused" in name, (ms, n, name)


@pytest.mark.parametrize("mode", ["fp64", "split"])
def test_a_lost_run_leaves_no_state(mode):
    """A run that lost a wait (here: one that may not wait for its neighbours'
    words) is reported, and nothing reads its torn fields: every call that uses
    the state fails until U and V are set, then the handle goes on."""
    nX = 200
    print(f"lost run {mode}", flush=True)
    pa, init = _case(nX, mode, 13)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        g.diag_resident(polls=0)
        g.iterate(2000)
        with pytest.raises(Ep2dError) as e:
            g.get("Ux")
        assert e.value.status == -2         # EP2D_ERR_HIP
        assert g.diag_resident(polls=1 << 20) == (0, 0, 1)
        calls = [lambda: g.get("Ux"), lambda: g.get("tauXX"), lambda: g.iterate(1),
                 lambda: g.iterate(100), lambda: g.residual([1e-3, 0.0, 0.0]),
                 lambda: g.apply_affine(1e-3, 0.0, 0.0, 0.0), g.averages, g.boundary,
                 g.hole_area, lambda: g.device_ptr("Vx"),
                 lambda: g.ComputeEffModuli(-1e-3, [1.0, 1.0, 0.0])]
        for k in STATE_FIELDS:
            for c in calls:
                with pytest.raises(Ep2dError) as e:
                    c()
                assert e.value.status == -7     # EP2D_ERR_STATE
            g.set(k, init[k])
        g.iterate(41)
        a = {k: g.get(k) for k in FIELDS}
    _same(a, _tiles(nX, mode, pa, init, 41))


def test_one_late_start_a_call():
    """The later launches of a call do not wait where the first one did in vain."""
    nX, n = 40, 3 * 65536 + 20
    print("late start of a long call", flush=True)
    pa, init = _case(nX, "split", 5)
    with EffPlast2D(pa, nX, nTasks=3, mode="split") as g:
        _start(g, init)
        g.diag_resident(arrive_ticks=0)
        g.iterate(n)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (0, 1, 0)
    _same(a, _tiles(nX, "split", pa, init, n))


def test_room_beside_another_run():
    """Tiles of half a CU each may lie one to a CU: beside a run of 252 of them 16
    more half tiles run resident, a grid of 48 whole-CU tiles (on 256 CUs) takes
    the chains at once and does not wait for that run."""
    print("room", flush=True)
    cases = [("split", 333, 60000), ("split", 64, 500), ("fp64", 128, 500)]
    hs, inits = [], []
    try:
        for mode, nX, _ in cases:
            pa, init = _case(nX, mode, 2 + nX)
            hs.append(EffPlast2D(pa, nX, nTasks=3, mode=mode))
            inits.append((pa, init))
            _start(hs[-1], init)
        for h in hs:        # (the first launches of the kernels load them)
            h.iterate(20)
            h.sync()
        t0 = time.perf_counter()
        ends = []
        for h, (_, _, n) in zip(hs, cases):
            h.iterate(n)
        for h in hs[1:] + hs[:1]:
            h.sync()
            ends.append(time.perf_counter() - t0)
        print("ends", ends, flush=True)
        assert [h.diag_resident() for h in hs] == [(2, 0, 0), (2, 0, 0), (1, 0, 0)]
        assert max(ends[:2]) < 0.5 * ends[2]
        for h, (mode, nX, n), (pa, init) in zip(hs, cases, inits):
            if n < 1000:
                _same({k: h.get(k) for k in FIELDS}, _tiles(nX, mode, pa, init, n + 20))
    finally:
        for h in hs:
            h.close()


def test_plain_capture_beside_other_handles():
    """Plain handles capture their runs on one thread while another thread's handle
    asks which handles are at work."""
    print("plain capture beside another thread", flush=True)
    nX, n = 33, 250
    pa, init = _case(nX, "plain", 1)
    errors = []

    def plain():
        try:
            with EffPlast2D(pa, nX, nTasks=3, mode="plain", tileRows=0) as g:
                _start(g, init)
                for _ in range(10):
                    g.iterate(25)
                ref = {k: g.get(k) for k in FIELDS}
            for _ in range(20):
                with EffPlast2D(pa, nX, nTasks=3, mode="plain") as g:
                    _start(g, init)
                    g.iterate(n)
                    _same({k: g.get(k) for k in FIELDS}, ref)
        except Exception as e:      # noqa: BLE001
            errors.append(e)

    th = threading.Thread(target=plain)
    with EffPlast2D(pa, nX, nTasks=3, mode="fp64") as g:
        _start(g, init)
        th.start()
        while th.is_alive():
            g.iterate(16)
            g.sync()
        th.join()
    assert not errors, errors


@pytest.mark.parametrize("mode", ["fp64", "split"])
def test_runs_queue_up(mode):
    """Resident runs are queued behind each other: the calls return at once, and
    a launch that did not start keeps those behind it from running."""
    nX = 125
    print(f"queued runs {mode}", flush=True)
    pa, init = _case(nX, mode, 31)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        g.iterate(16)
        g.sync()
        t0 = time.perf_counter()
        for n in (20001, 30, 16, 20000):
            g.iterate(n)
        t1 = time.perf_counter()
        g.sync()
        t2 = time.perf_counter()
        assert t1 - t0 < 0.25 * (t2 - t0)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (5, 0, 0)
        _same(a, _tiles(nX, mode, pa, init, 40063))
        # two run, the third does not start, nor the two queued behind it
        _start(g, init)
        g.iterate(3000)
        g.iterate(17)
        g.diag_resident(arrive_ticks=0)
        g.set_timing(1)
        for n in (18, 16, 19):
            g.iterate(n)
        ms, samples, name = g.timing()
        a = {k: g.get(k) for k in FIELDS}
        done, late, lost = g.diag_resident()
        assert (done, lost) == (7, 0) and late >= 1
        # (16-step launches of four, one on its own: closing ones are no samples)
        assert "k_chain" in name and samples <= 53
        _same(a, _tiles(nX, mode, pa, init, 3000 + 17 + 53))


@pytest.mark.parametrize("mode,nX", [("fp64", 256), ("split", 400), ("fp64", 700)])
def test_many_handles_at_once(mode, nX):
    """With several handles at work the chains take taller segments: one height
    for two handles, one for more."""
    print(f"many handles {mode} nX={nX}", flush=True)
    cases = [_case(nX, mode, 60 + k) for k in range(6)]
    hs = [EffPlast2D(pa, nX, nTasks=3, mode=mode) for pa, _ in cases]
    steps = (40, 11, 4, 3, 18)
    try:
        for h, (_, init) in zip(hs, cases):
            _start(h, init)
        hs[0].iterate(5000)      # the others find it at work
        for n in steps:
            for h in hs[1:]:
                h.iterate(n)
        for h in hs[1:]:
            h.sync()
        for h, (pa, init) in zip(hs[1:], cases[1:]):
            _same({k: h.get(k) for k in FIELDS}, _tiles(nX, mode, pa, init, sum(steps)))
    finally:
        for h in hs:
            h.close()


def test_many_handles_are_no_slower_than_tiles():
    """Eight FP64 handles of 256^2 side by side: the chains of one handle alone
    would take 1.5 times the tile kernel's time (measured 3.7 us per handle
    iteration against 2.5), those for several take less than it (2.2)."""
    nX, n, reps = 256, 500, 4
    print("many handles, time", flush=True)
    pa, init = _case(nX, "fp64", 4)

    def run(**kw):
        hs = [EffPlast2D(pa, nX, nTasks=3, mode="fp64", **kw) for _ in range(8)]
        try:
            for h in hs:
                _start(h, init)
                h.iterate(20)
                h.sync()
            best = 1e9
            for _ in range(3):
                t0 = time.perf_counter()
                for _ in range(reps):
                    for h in hs:
                        h.iterate(n)
                for h in hs:
                    h.sync()
                best = min(best, time.perf_counter() - t0)
            return best
        finally:
            for h in hs:
                h.close()

    mine, tiles = run(), run(tileRows=8)
    print(f"{mine * 1e3:.1f} ms, tiles {tiles * 1e3:.1f} ms", flush=True)
    assert mine < 1.1 * tiles


@pytest.mark.parametrize("mode,nX", [("fp64", 125), ("split", 200)])
def test_runs_that_find_no_room(mode, nX):
    """A launch that finds other tiles in its room ends at once; the next run is
    tried again."""
    print(f"no room {mode} nX={nX}", flush=True)
    pa, init = _case(nX, mode, 17 + nX)
    steps = (33, 16, 18)
    with EffPlast2D(pa, nX, nTasks=3, mode=mode) as g:
        _start(g, init)
        g.diag_resident(cus=1)
        for n in steps:
            g.iterate(n)
            g.sync()
        assert g.diag_resident(cus=256) == (0, 3, 0)
        g.iterate(20)
        a = {k: g.get(k) for k in FIELDS}
        assert g.diag_resident() == (1, 3, 0)
    _same(a, _tiles(nX, mode, pa, init, sum(steps) + 20))


@pytest.mark.parametrize("mode,nX,k", [("fp64", 128, 8), ("split", 128, 16)])
def test_small_handles_share_the_device(mode, nX, k):
    """Handles whose tiles fit the device as far as they can run at once stay
    resident side by side, however many are queued."""
    print(f"{k} handles {mode} nX={nX}", flush=True)
    cases = [_case(nX, mode, 80 + q) for q in range(k)]
    hs = [EffPlast2D(pa, nX, nTasks=3, mode=mode) for pa, _ in cases]
    try:
        for h, (_, init) in zip(hs, cases):
            _start(h, init)
        for n in (700, 33):
            for h in hs:
                h.iterate(n)
        for h in hs:
            assert h.diag_resident() == (2, 0, 0)
        for h, (pa, init) in list(zip(hs, cases))[::5]:
            _same({f: h.get(f) for f in FIELDS}, _tiles(nX, mode, pa, init, 733))
    finally:
        for h in hs:
            h.close()


@pytest.mark.parametrize("nX,resident", [(512, 0), (128, 4)])
def test_a_batch_keeps_its_share(nX, resident):
    """Beside a batch in a step a handle runs resident if its tiles take a quarter
    of the device at most (240 and 48 CUs here), else its iterations take the
    chains; both end with their results."""
    print(f"batch beside a handle {nX}", flush=True)
    pa, init = _case(nX, "fp64", 6)
    bpa = make_pa(1024, nPores=1, porosity=0.02)
    state = {}

    def batch():
        with Batch(mode="split", checkInterval=500) as eng:
            for tag in range(8):
                eng.submit(bpa, nX=1024, nTasks=1, nIter=6000, eIter=1e-30, initLoad=-1e-3,
                           loadType=[1.0, 1.0, 0.0], tag=tag)
            state["started"] = True
            eng.run()
            state["out"] = eng.poll()

    th = threading.Thread(target=batch)
    with EffPlast2D(pa, nX, nTasks=3, mode="fp64") as g:
        _start(g, init)
        th.start()
        while "started" not in state:
            time.sleep(0.001)
        time.sleep(0.05)
        for _ in range(4):
            g.iterate(25)
            g.sync()
        busy = th.is_alive()
        a = {k: g.get(k) for k in FIELDS}
        runs = g.diag_resident()
        th.join()
    assert busy and runs == (resident, 0, 0)
    assert [r["status"] for r in state["out"]] == [0] * 8
    _same(a, _tiles(nX, "fp64", pa, init, 100))


def test_handles_beside_a_capture():
    """While a caller's stream is captured (in the mode that watches every thread),
    handles on streams of their own go on, and ask which of them are at work."""
    nX = 96
    print("handles beside a capture", flush=True)
    pa, init = _case(nX, "fp64", 8)
    st = torch.cuda.Stream()
    with EffPlast2D(pa, nX, nTasks=3, mode="fp64", stream=st.cuda_stream) as c, \
            EffPlast2D(pa, nX, nTasks=3, mode="fp64") as a, \
            EffPlast2D(pa, nX, nTasks=3, mode="split") as b, \
            EffPlast2D(pa, nX, nTasks=3, mode="fp64", marchRows=16) as d:
        for h in (a, c, d):
            _start(h, init)
        for h in (a, b, c, d):
            h.iterate(32)       # (the first launches of the kernels load them)
            h.sync()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=st, capture_error_mode="global"):
            for n in (32, 5, 3, 200):   # the second waits for the first
                for h in (d, a, b):
                    h.iterate(n)
            a.apply_affine(0.0, 0.0, 0.0, 0.0)
            c.iterate(32)
        for _ in range(2):
            graph.replay()
            torch.cuda.synchronize()
        _same({k: c.get(k) for k in FIELDS}, _tiles(nX, "fp64", pa, init, 96))
        for h in (a, d):
            _same({k: h.get(k) for k in FIELDS}, _tiles(nX, "fp64", pa, init, 272))
