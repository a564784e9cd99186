"""Stage times of a call, noted by the call's own kernels: for every form of a
batch each stage time is at least 0, the stages that follow each other add up
to no more than the call, and the call to no more than the host's clock around
it. The results stay the oracle's."""
import time

import numpy as np
import pytest

import coincgraph_amd as cg
from tests.helpers import oracle_apply, oracle_graph, oracle_values

pytestmark = pytest.mark.gpu

TICK_MS = 1e-5 * 8  # one tick of the 100 MHz clock a stage, rounding


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


def _check(st, wall_ms, where):
    parts = ["mutate_ms", "repair_ms", "seed_ms", "propagate_ms", "invalidate_ms", "scan_kernel_ms"]
    for p in parts:
        assert st[p] >= 0.0, (where, p, st[p])
    assert 0.0 < st["total_ms"] <= wall_ms + TICK_MS, (where, st["total_ms"], wall_ms)
    assert sum(st[p] for p in parts[:4]) <= st["total_ms"] + TICK_MS, where
    assert max(st["invalidate_ms"], st["scan_kernel_ms"]) <= st["total_ms"] + TICK_MS, where


@pytest.mark.parametrize("algo,kw", [
    ("sssp", {}),
    ("sssp", dict(n_stream=1)),
    ("sssp", dict(flags=cg.CFG_GRAPH_BATCHES)),
    ("sssp", dict(flags=cg.CFG_GRAPH_BATCHES, n_stream=1)),
    ("bfs", dict(flags=cg.CFG_SCAN_REPAIR)),
    ("sssp", dict(flags=cg.CFG_ORDERED_REPAIR)),
    ("cc", {}),
    ("cc", dict(flags=cg.CFG_SYMMETRIC | cg.CFG_CC_UNION_REPAIR)),
    ("sssp", dict(flags=cg.CFG_COOPERATIVE)),
    ("cc", dict(flags=cg.CFG_SYMMETRIC | cg.CFG_CC_UNION_REPAIR)),
    ("sssp", dict(flags=cg.CFG_COOPERATIVE)),
    ("pr", dict(pr_epsilon=1e-6)),
])
def test_stage_times(algo, kw):
    print(f"[gpu-case] stage times {algo} {kw}", flush=True)
    g = cg.rmat_graph(11, 8, seed=3, symmetric=algo == "cc")
    s = cg.rmat_stream(g, 11, 6, 200, 200, seed=4, symmetric=algo == "cc")
    og = oracle_graph(g)
    none = np.zeros(0, dtype=s.batch(0)[0].dtype)
    with cg.Engine(algo, **kw) as e:
        e.load_graph(g)
        e.init_graph(0)
        e.start()
        for b in range(6):
            dels, adds = s.batch(b)
            if b == 3:
                adds = none
            if b == 4:
                dels = none
            t = time.perf_counter()
            st = e.apply_batch(dels, adds, staged=b == 5)
            _check(st, 1e3 * (time.perf_counter() - t), (algo, kw, b))
            oracle_apply(og, dels, adds)
            if algo != "pr":
                assert np.array_equal(e.values(), oracle_values(og, algo)), b
            if b < 3:  # (component unions have no propagation: the inserts' unions are their seeds)
                assert st["mutate_ms"] > 0 and st["seed_ms"] + st["propagate_ms"] > 0, b


def test_stage_times_of_sources_and_queries():
    print("[gpu-case] stage times of sources", flush=True)
    g = cg.rmat_graph(11, 8, seed=5)
    s = cg.rmat_stream(g, 11, 3, 200, 200, seed=6)
    for n_stream in (1, 3):
        with cg.Engine("sssp", n_stream=n_stream) as e:
            e.load_graph(g)
            e.init_graph([0, 1, 2, 3, 4])
            e.start()
            for b in range(3):
                t = time.perf_counter()
                st = e.apply_batch(*s.batch(b))
                _check(st, 1e3 * (time.perf_counter() - t), (n_stream, b))
                assert st["mutate_ms"] > 0 and st["propagate_ms"] > 0
