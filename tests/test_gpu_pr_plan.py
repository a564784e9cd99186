"""PageRank's pull plan at its edges: incoming rows around every size class,
the tile split and several tiles, few vertices, frontiers that a dense round
leaves to a sparse one, solves cut short by the round cap and continued.
Normalised L1 <= 1e-6 against FP64 with epsilon 1e-7, as the other PageRank
tests."""
import numpy as np
import pytest

import coincgraph_amd as cg
from tests.helpers import oracle_apply, oracle_graph, pr_errors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


EDGES = [0, 1, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 128, 129, 255, 256, 257, 2047, 2048, 2049, 4097]


def _graph(n, seed):
    """Vertex v < len(EDGES) has EDGES[v] in-edges (as far as n allows distinct
    sources do not matter: parallel edges count), the others a few."""
    rng = np.random.default_rng(seed)
    ind = rng.integers(0, 6, n)
    k = min(n, len(EDGES))
    ind[:k] = EDGES[:k]
    v = np.repeat(np.arange(n), ind)
    u = rng.integers(0, n, len(v))
    order = np.lexsort((v, u))
    off = np.zeros(n + 1, dtype=np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=n))
    return cg.HostGraph(n, off, v[order].astype(np.uint32))


def _check(e, og, where):
    l1, _ = pr_errors(e.values(), og.pagerank()[0])
    assert l1 <= 1e-6, f"{where}: normalised L1 {l1}"


@pytest.mark.parametrize("flags", [0, cg.CFG_PR_KEEP_IDS])
@pytest.mark.parametrize("n", [1, 63, 65, 1000, 40000])
@pytest.mark.parametrize("divisor,cap", [(0, 1000), (2, 1000), (0, 7), (2, 5), (1 << 30, 1000)])
def test_pull_plan_edges(n, flags, divisor, cap):
    print(f"[gpu-case] pull plan n={n} flags={flags} divisor={divisor} cap={cap}", flush=True)
    g = _graph(n, n)
    og = oracle_graph(g)
    rng = np.random.default_rng(n + 1)
    with cg.Engine("pr", pr_epsilon=1e-7, pr_max_rounds=cap, pr_pull_divisor=divisor, flags=flags) as e:
        e.load_graph(g)
        e.init_graph()

        def settle(st):
            for _ in range(400):
                if st["converged"]:
                    return
                st = e.start()
            raise AssertionError("PageRank did not converge")

        settle(e.start())
        _check(e, og, "initial")
        for b in range(2):
            off, dst = og.csr()
            m = int(off[-1])
            at = rng.permutation(m)[:m // 10]
            u = (np.searchsorted(off, at, side="right") - 1).astype(np.uint32)
            dels = cg.edges_array(u, dst[at])
            adds = cg.edges_array(rng.integers(0, n, len(at) + 3), rng.integers(0, min(n, 40), len(at) + 3))
            settle(e.apply_batch(dels, adds))
            oracle_apply(og, dels, adds)
            _check(e, og, f"batch {b}")


@pytest.mark.parametrize("flags", [0, cg.CFG_PR_KEEP_IDS])
@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 1])
def test_mask_rule_edge(n, flags):
    """The vertex count from which sparse sweeps test the source mask: a solve
    whose frontier shrinks through every form, then a batch whose rounds start
    sparse."""
    print(f"[gpu-case] mask rule n={n} flags={flags}", flush=True)
    g = _graph(n, n)
    og = oracle_graph(g)
    rng = np.random.default_rng(n)
    with cg.Engine("pr", pr_epsilon=1e-7, pr_max_rounds=1000, flags=flags) as e:
        e.load_graph(g)
        e.init_graph()
        assert e.start()["converged"]
        _check(e, og, "initial")
        off, dst = og.csr()
        at = rng.permutation(int(off[-1]))[:3000]
        u = (np.searchsorted(off, at, side="right") - 1).astype(np.uint32)
        dels = cg.edges_array(u, dst[at])
        adds = cg.edges_array(rng.integers(0, n, 3000).astype(np.uint32), rng.integers(0, n, 3000).astype(np.uint32))
        assert e.apply_batch(dels, adds)["converged"]
        oracle_apply(og, dels, adds)
        _check(e, og, "batch")
