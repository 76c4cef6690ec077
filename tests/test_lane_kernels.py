"""The kernels with one lane per search, which take the batches that keep very many lanes busy: every
schedule and occupancy on more than 65,536 lanes with more than two jobs each. Tables and every
counter of the search equal the CPU's. A small batch on the same handle goes to the wave kernel,
with the same TTs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LANES = 65792  # one block of 256 above the line


@pytest.fixture(scope="module")
def batch(ddx):
    hands = ddx.random_deals(91, 6600, 5)
    return hands, ddx.cpu_solve(hands, threads=8, tt_log2=9, jobs_per_deal=20)


def same(got, want):
    (out, st), (tables, cpu) = got, want
    assert np.array_equal(out, tables)
    for f in ("jobs_done", "nodes", "tt_probes", "tt_hits", "tt_entry_reads", "tt_stores"):
        assert getattr(st, f) == getattr(cpu, f), f


@pytest.mark.parametrize("schedule,waves", [(0, 0), (1, 0), (2, 0), (3, 0), (2, 3), (2, 4)])
def test_equal_to_cpu(ddx, batch, schedule, waves):
    hands, want = batch
    few = ddx.random_deals(92, 300, 6)
    want_few = ddx.cpu_solve(few, tt_log2=9, jobs_per_deal=20)
    with ddx.GpuSolver(lanes=LANES, tt_log2=9, jobs_per_deal=20, schedule=schedule, waves_per_simd=waves) as g:
        assert g.waves(len(hands)) == 0 and g.waves(len(few)) == 6000 and g.waves(0) == 0
        for _ in range(2):
            print("schedule", schedule, "waves", waves, flush=True)
            same(g.solve(hands), want)
            same(g.solve(few), want_few)


def test_seeded(ddx, batch):
    hands, _ = batch
    seeds = np.random.default_rng(4).integers(0, 14, (len(hands), 20)).astype(np.uint8)
    want = ddx.cpu_solve(hands, threads=8, tt_log2=9, jobs_per_deal=20, seed_mode=ddx.SEED_CERT, seeds=seeds)
    with ddx.GpuSolver(lanes=LANES, tt_log2=9, jobs_per_deal=20, schedule=ddx.SCHED_SPLIT, waves_per_simd=3,
                       seed_mode=ddx.SEED_CERT, graph=True) as g:
        assert g.waves(len(hands)) == 0
        for _ in range(2):
            same(g.solve(hands, seeds=seeds), want)


@pytest.mark.parametrize("schedule", [0, 1, 2])
def test_team_kernel(ddx, schedule):
    """16-lane teams, which have a kernel of their own for the stage profile only: tables exact, every
    node counted at one exit. (Its node counts vary a little from run to run.)"""
    hands = ddx.random_deals(93, 400, 7)
    want, _ = ddx.cpu_solve(hands, threads=8, tt_log2=9)
    with ddx.GpuSolver(lanes=16384, tt_log2=9, team=16, schedule=schedule, profile=True) as g:
        assert g.waves(len(hands)) == 0
        g.profile(reset=True)
        out, st = g.solve(hands)
        exits = g.profile(reset=True).astype(np.int64)[16:23]
    assert np.array_equal(out, want) and exits.sum() == st.nodes and st.jobs_done == 2000


def test_stop_on_waves(ddx):
    """A stop request to the wave kernel, sent once the first jobs are done: it ends soon, and what is
    finished is exact."""
    import threading
    import time
    g = np.load(__file__.replace("test_lane_kernels.py", "golden/full_2000.npz"))
    with ddx.GpuSolver(lanes=65536, tt_log2=10) as s:
        assert s.waves(2000) == s.waves(10 ** 6) > 0  # 10,000 jobs of up to 5e8 nodes: minutes
        stopped = []

        def stop():
            while s.progress() < 500:
                time.sleep(0.01)
            stopped.append(time.time())
            s.request_stop()

        t = threading.Thread(target=stop, daemon=True)
        t.start()
        out, st = s.solve(g["hands"], allow_stop=True)
        took = time.time() - stopped[0]
        t.join()
        assert took < 2 and 500 <= st.jobs_done < 10000
        done = out != 255
        assert (out[done] == g["tables"][done]).all() and done.sum() >= 4 * 500
        out, st = s.solve(g["hands"][:0])  # and the handle goes on
        assert st.jobs_done == 0
