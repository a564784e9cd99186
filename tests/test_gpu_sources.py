"""Multi-source runs at the edges of their tiles: vertex counts around the
64-vertex tiles of the result transpose, source counts around the source
groups of a wave, rows around the long-row split. Queries, the no-allocation
query and 64-bit state of maintained sources, bit-exact against the oracle."""
import numpy as np
import pytest

import coincgraph_amd as cg
from oracle import oracle as O
from tests.helpers import oracle_graph
from tests.test_zz_no_alloc import DeviceWords, _hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


def _graph(n, seed):
    """Random directed multigraph of n vertices; vertices 0 and 1 (when there
    are that many) have rows of 63..65, 127..129 or more slots."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 6, n)
    deg[0] = [1, 63, 64, 65, 129, 700][seed % 6]
    if n > 1:
        deg[1] = [127, 128, 129, 2049, 64, 1][seed % 6]
    off = np.zeros(n + 1, dtype=np.uint64)
    off[1:] = np.cumsum(deg)
    return cg.HostGraph(n, off, rng.integers(0, n, int(off[-1])).astype(np.uint32))


def _sources(n, k, seed):
    s = np.random.default_rng(seed).integers(0, n, k).astype(np.uint32)
    s[0] = 0
    return s


def _distances(og, algo, s):
    return og.bfs(int(s)) if algo == "bfs" else og.sssp(int(s), O.W_HASH64, 5)


@pytest.mark.parametrize("n,k", [(1, 1), (2, 3), (63, 4), (64, 5), (65, 64), (127, 31), (129, 33), (3000, 2), (4097, 63),
                                 (16384, 64), (70001, 17)])
@pytest.mark.parametrize("algo", ["bfs", "sssp"])
def test_queries_at_tile_edges(algo, n, k):
    print(f"[gpu-case] query {algo} n={n} k={k}", flush=True)
    g = _graph(n, n + k)
    src = _sources(n, k, k)
    og = oracle_graph(g)
    exp = np.stack([_distances(og, algo, s) for s in src])
    hip = _hip()
    with cg.Engine("sssp", weight_mode=cg.WEIGHT_HASH64, weight_seed=5) as e:
        e.load_graph(g)
        for _ in range(2):  # the second run starts from what the first left behind
            assert np.array_equal(e.query(algo, src), exp)
            buf = DeviceWords(hip, k * n)
            try:
                e.query_noalloc(algo, src, buf.p.value, 4 * k * n)
                assert np.array_equal(buf.read().reshape(k, n), exp)
            finally:
                buf.free()


@pytest.mark.parametrize("n,k", [(2, 2), (65, 64), (129, 33), (4097, 63), (16384, 64), (70001, 5)])
@pytest.mark.parametrize("algo", ["bfs", "sssp"])
def test_maintained_sources_at_tile_edges(algo, n, k):
    print(f"[gpu-case] sources {algo} n={n} k={k}", flush=True)
    g = _graph(n, n + k)
    src = _sources(n, k, k)
    og = oracle_graph(g)
    rng = np.random.default_rng(k)
    with cg.Engine(algo, weight_mode=cg.WEIGHT_HASH64, weight_seed=5) as e:
        e.load_graph(g)
        e.init_graph(src)
        e.start()
        for b in range(3):
            off, dst = og.csr()
            m = int(off[-1])
            at = rng.permutation(m)[:max(1, m // 20)]
            u = (np.searchsorted(off, at, side="right") - 1).astype(np.uint32)
            dels = cg.edges_array(u, dst[at])
            adds = cg.edges_array(rng.integers(0, n, len(at)), rng.integers(0, n, len(at)))
            if b == 2:
                dels = dels[:0]  # inserts alone
            e.apply_batch(dels, adds)
            og.apply_deletes(dels["u"], dels["v"])
            og.apply_adds(adds["u"], adds["v"])
            exp = np.stack([_distances(og, algo, s) for s in src])
            assert np.array_equal(e.values(), exp), f"batch {b}"
            par = e.parents()
            for i in (0, k - 1):
                res = og.check_parent(exp[i], par[i], int(src[i]), O.W_UNIT if algo == "bfs" else O.W_HASH64, 5)
                assert res.invalid_vertices == 0, f"batch {b} source {i}"


@pytest.mark.parametrize("n", [524287, 524288, 524289, 1048576, 1048577, 4 * 1048576 + 3, 5 * 1048576, 9 * 1048576 + 1])
def test_result_copy_at_buffer_edges(n):
    """Results of 4 B a vertex around the direct copy's limit (2 MiB) and the
    bounce buffers' edges (4 MiB each, a ring of four)."""
    print(f"[gpu-case] result copy n={n}", flush=True)
    off = np.zeros(n + 1, dtype=np.uint64)
    off[n - 1:] = 1
    g = cg.HostGraph(n, off, np.array([n - 1], dtype=np.uint32))  # one edge, n-2 -> n-1
    exp = np.arange(n, dtype=np.uint32)
    par = np.full(n, cg.INF, dtype=np.uint32)
    exp[n - 1] = par[n - 1] = n - 2
    with cg.Engine("cc") as e:
        e.load_graph(g)
        e.init_graph()
        e.start()
        for _ in range(2):
            assert np.array_equal(e.values(), exp)
        assert np.array_equal(e.parents(), par)
