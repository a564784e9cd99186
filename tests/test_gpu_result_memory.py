"""Reading results takes no device memory: values, parents and a renumbered
PageRank engine's fields, of 4 MiB and more, leave the free device memory as
it was."""
import ctypes as C

import numpy as np
import pytest

import coincgraph_amd as cg
from tests.test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


def _free(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _chain(n):
    """0 -> 1 -> 2 and no other edge."""
    off = np.full(n + 1, 2, dtype=np.uint64)
    off[0], off[1] = 0, 1
    return cg.HostGraph(n, off, np.array([1, 2], dtype=np.uint32))


@pytest.mark.parametrize("algo", ["bfs", "pr"])
def test_results_take_no_device_memory(algo):
    print(f"[gpu-case] result memory {algo}", flush=True)
    hip = _hip()
    read = (lambda e: (e.values(), e.parents())) if algo == "bfs" else (lambda e: (e.values(), e.residuals()))
    with cg.Engine(algo) as warm:  # the kernels and the copy path have run once
        warm.load_graph(_chain(1 << 20))
        warm.init_graph(0)
        warm.start()
        read(warm)
    n = 1 << 23
    with cg.Engine(algo) as e:
        e.load_graph(_chain(n))
        e.init_graph(0)
        e.start()
        before = _free(hip)
        a, b = read(e)
        assert _free(hip) == before
    if algo == "bfs":
        assert a[:4].tolist() == [0, 1, 2, cg.INF] and (a[3:] == cg.INF).all()
        assert b[:4].tolist() == [cg.INF, 0, 1, cg.INF] and (b[3:] == cg.INF).all()
    else:
        assert np.allclose(a[:4], [0.15, 0.2775, 0.385875, 0.15], rtol=1e-6, atol=0) and (a[3:] == a[0]).all()
        assert (np.abs(b) <= 1e-6).all()


def test_pagerank_of_a_second_graph_with_more_long_rows():
    """An engine's second graph needs fewer tiles than its first but has more
    incoming rows of several tiles."""
    print("[gpu-case] PageRank of a second graph", flush=True)
    from tests.helpers import oracle_graph, pr_errors
    rng = np.random.default_rng(95)

    def graph(n, u, v):
        order = np.argsort(u, kind="stable")
        off = np.zeros(n + 1, dtype=np.uint64)
        off[1:] = np.cumsum(np.bincount(u, minlength=n))
        return cg.HostGraph(n, off, v[order].astype(np.uint32))

    with cg.Engine("pr", pr_epsilon=1e-7, pr_max_rounds=1000, pool_slack=1) as e:
        for n, rows, length in ((3, 3, 700_000), (2000, 60, 3000)):
            v = np.concatenate([np.repeat(np.arange(rows), length), rng.integers(0, n, n)])
            g = graph(n, rng.integers(0, n, len(v)), v)
            e.load_graph(g)
            e.init_graph()
            assert e.start()["converged"]
            assert pr_errors(e.values(), oracle_graph(g).pagerank()[0])[0] <= 1e-6, n


@pytest.mark.parametrize("n", [1, 2, 257, 65535, 65536, 65537, 131072, 131073, 262145, 524288, 524289])
def test_results_around_their_routes(n):
    """Results of up to 2 MiB are formed in host memory, two buffers by turns;
    longer ones are copied."""
    print(f"[gpu-case] short results n={n}", flush=True)
    rng = np.random.default_rng(n)
    off = np.zeros(n + 1, dtype=np.uint64)
    off[1:] = np.cumsum(rng.integers(0, 4, n))
    g = cg.HostGraph(n, off, rng.integers(0, n, int(off[-1])).astype(np.uint32))
    from tests.helpers import check_traversal, oracle_graph, pr_errors
    og = oracle_graph(g)
    with cg.Engine("sssp") as e:
        e.load_graph(g)
        e.init_graph(0)
        e.start()
        for _ in range(2):
            check_traversal(e, og, "sssp", 0)
    for flags in (0, cg.CFG_PR_KEEP_IDS):
        with cg.Engine("pr", pr_epsilon=1e-7, pr_max_rounds=1000, flags=flags) as e:
            e.load_graph(g)
            e.init_graph()
            assert e.start()["converged"]
            assert pr_errors(e.values(), og.pagerank()[0])[0] <= 1e-6
            assert (np.abs(e.residuals()) <= 1e-7).all()
