"""Queries on an engine whose own frontier is still pending (initialised and
not solved yet, or stopped by a round cap): the distances equal the oracle's,
and the engine's next calls continue from where they stood."""
import numpy as np
import pytest

import coincgraph_amd as cg
from tests.helpers import check_traversal, oracle_apply, oracle_graph, oracle_values, pr_errors

pytestmark = pytest.mark.gpu

N, SCALE = 1 << 11, 11


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


def _check_queries(e, og):
    for algo in ("sssp", "bfs"):
        for sources in ([3], [5, 0, 77, 5, 1031]):
            got = e.query(algo, sources)
            for i, s in enumerate(sources):
                assert np.array_equal(got[i], oracle_values(og, algo, s)), (algo, s)


@pytest.mark.parametrize("algo,sources,kw", [
    ("sssp", 0, {}), ("bfs", 0, {}), ("cc", 0, {}),
    ("sssp", [0, 9, 100], {}), ("bfs", [0, 9, 100], {}),
    ("sssp", 0, dict(flags=cg.CFG_COOPERATIVE)), ("sssp", 0, dict(flags=cg.CFG_SCAN_REPAIR)),
    ("sssp", 0, dict(flags=cg.CFG_ORDERED_REPAIR))])
def test_query_between_init_and_start(algo, sources, kw):
    print(f"[gpu-case] query before start {algo} {sources} {kw}", flush=True)
    g = cg.rmat_graph(SCALE, 16, seed=81)
    og = oracle_graph(g)
    s = cg.rmat_stream(g, SCALE, 1, 200, 200, seed=82)
    with cg.Engine(algo, **kw) as e:
        e.load_graph(g)
        e.init_graph(sources)
        _check_queries(e, og)
        e.start()
        for b in range(2):
            if isinstance(sources, list):
                got = e.values()
                for i, src in enumerate(sources):
                    assert np.array_equal(got[i], oracle_values(og, algo, src)), (b, src)
            else:
                check_traversal(e, og, algo, 0, where=f"step {b}")
            if b == 0:
                e.apply_batch(*s.batch(0))
                oracle_apply(og, *s.batch(0))


@pytest.mark.parametrize("algo", ["sssp", "bfs", "cc"])
@pytest.mark.parametrize("split", [0, 64])
def test_query_of_a_capped_engine(algo, split):
    """One round a call; with the small split the cap leaves tiles pending too."""
    print(f"[gpu-case] query of a capped engine {algo} split={split}", flush=True)
    g = cg.rmat_graph(SCALE, 16, seed=83)
    og = oracle_graph(g)
    with cg.Engine(algo, max_rounds=1, split_degree=split, adapt_split=split and 1) as e:
        e.load_graph(g)
        e.init_graph(0)
        for i in range(60):
            e.start()
            if i < 4:
                _check_queries(e, og)
        check_traversal(e, og, algo, 0, where="after 60 rounds")


@pytest.mark.parametrize("cap,kw", [
    (1, {}), (3, {}), (3, dict(flags=cg.CFG_PR_PUSH_ONLY)), (3, dict(flags=cg.CFG_COOPERATIVE)),
    (1, dict(pr_pull_divisor=2)), (3, dict(pr_pull_divisor=1 << 30))])
def test_query_of_a_capped_pagerank(cap, kw):
    """The gathered rounds leave their frontier as flags without a list."""
    print(f"[gpu-case] query of a capped PageRank cap={cap} {kw}", flush=True)
    kw = dict(kw, flags=kw.get("flags", 0) | cg.CFG_PR_KEEP_IDS)
    g = cg.rmat_graph(SCALE, 16, seed=84)
    s = cg.rmat_stream(g, SCALE, 1, 200, 200, seed=85)
    og = oracle_graph(g)
    with cg.Engine("pr", pr_epsilon=1e-7, pr_max_rounds=cap, **kw) as e:
        e.load_graph(g)
        e.init_graph()
        _check_queries(e, og)
        for b in range(2):
            for i in range(400):
                st = e.start()
                if st["converged"]:
                    break
                if i < 3 or i % 10 == 0:
                    _check_queries(e, og)
            assert st["converged"]
            assert pr_errors(e.values(), og.pagerank()[0])[0] <= 1e-6, b
            if b == 0:
                st = e.apply_batch(*s.batch(0))
                oracle_apply(og, *s.batch(0))
                _check_queries(e, og)
