"""Multi-source passes under a split and a tile length beyond every row: a row
of 1,300,000 slots (63 sources: its (edge, source) pairs are more than a lane's
item division is exact for) and a vertex with as many incoming edges. Queries
and maintained sources, bit-exact against the oracle."""
import numpy as np
import pytest

import coincgraph_amd as cg
from oracle import oracle as O
from tests.helpers import oracle_apply, oracle_graph

pytestmark = pytest.mark.gpu

N, HUB = 4096, 1_300_000


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


@pytest.fixture(scope="module")
def graph():
    rng = np.random.default_rng(91)
    u = np.concatenate([np.full(HUB, 7), rng.integers(0, N, HUB + 4 * N)])
    v = np.concatenate([rng.integers(0, N, HUB), np.full(HUB, 11), rng.integers(0, N, 4 * N)])
    order = np.argsort(u, kind="stable")
    off = np.zeros(N + 1, dtype=np.uint64)
    off[1:] = np.cumsum(np.bincount(u, minlength=N))
    return cg.HostGraph(N, off, v[order].astype(np.uint32))


def _distances(og, algo, s):
    return og.bfs(int(s)) if algo == "bfs" else og.sssp(int(s), O.W_HASH64, 5)


KW = [dict(split_degree=0xFFFFFFFF), dict(split_degree=0xFFFFFFFF, tile_len=1 << 30), dict(split_degree=1 << 20)]


@pytest.mark.parametrize("kw", KW)
@pytest.mark.parametrize("algo", ["bfs", "sssp"])
def test_rows_longer_than_the_pairs_allow(graph, algo, kw):
    print(f"[gpu-case] long rows {algo} {kw}", flush=True)
    og = oracle_graph(graph)
    rng = np.random.default_rng(92)
    src = rng.integers(0, N, 63).astype(np.uint32)
    src[0] = 7
    with cg.Engine(algo, weight_mode=cg.WEIGHT_HASH64, weight_seed=5, **kw) as e:
        e.load_graph(graph)
        e.init_graph(src)
        e.start()
        for b in range(2):
            exp = np.stack([_distances(og, algo, s) for s in src])
            assert np.array_equal(e.values(), exp), b
            assert np.array_equal(e.query(algo, src), exp), b
            if b == 0:
                off, dst = og.csr()
                at = np.concatenate([int(off[7]) + rng.permutation(HUB)[:60], rng.permutation(int(off[-1]))[:60]])
                du = (np.searchsorted(off, at, side="right") - 1).astype(np.uint32)
                dels = cg.edges_array(du, dst[at])
                adds = cg.edges_array(rng.integers(0, N, 100), rng.integers(0, N, 100))
                e.apply_batch(dels, adds)
                oracle_apply(og, dels, adds)
