"""Delete claims around the batch size that decides between one launch and
one per kind of row: rows of every kind (tiny, medium with few and with many
deletes, long) in both tiers, repeated and missing records, bit-exact against
the oracle. The call's statistics are folded by the same kernels on both
sides."""
import numpy as np
import pytest

import coincgraph_amd as cg
from tests.helpers import check_incoming, check_topology, check_traversal, oracle_apply, oracle_graph

pytestmark = pytest.mark.gpu

ONE = 1 << 14  # delete records, mirrors included


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if cg.device_count() < 1:
        pytest.skip("no HIP device")


@pytest.mark.parametrize("nd", [1, 255, 256, 257, ONE // 2 - 1, ONE // 2, ONE // 2 + 1])
@pytest.mark.parametrize("tier", ["hbm", "host"])
def test_claims_around_the_launch_rule(tier, nd):
    print(f"[gpu-case] claims {tier} nd={nd}", flush=True)
    rng = np.random.default_rng(nd)
    n = 3000
    deg = rng.integers(0, 60, n)
    deg[:8] = [63, 64, 65, 255, 257, 4096, 4097, 20000]
    off = np.zeros(n + 1, dtype=np.uint64)
    off[1:] = np.cumsum(deg)
    m = int(off[-1])
    g = cg.HostGraph(n, off, rng.integers(0, n, m).astype(np.uint32))
    src = np.repeat(np.arange(n, dtype=np.uint32), deg)
    og = oracle_graph(g)
    with cg.Engine("sssp", weight_mode=cg.WEIGHT_HASH64, weight_seed=5,
                   cache_bytes=m if tier == "host" else 0) as e:
        e.load_graph(g)
        e.init_graph(0)
        e.start()
        for b in range(2):
            pick = rng.choice(m, nd, replace=False)
            dels = np.zeros(nd, dtype=cg.EDGE_DTYPE)
            dels["u"], dels["v"] = src[pick], g.dst[pick]
            dels["u"][: nd // 8] = 7  # many deletes of one long row, some of them missing
            dels["v"][nd // 4: nd // 4 + nd // 16] = dels["v"][nd // 4]
            adds = dels[:: 3].copy()
            adds["v"] = rng.integers(0, n, len(adds))
            st = e.apply_batch(dels, adds)
            miss, inval = oracle_apply(og, dels, adds)
            assert (st["missing_deletes"], st["invalid_updates"]) == (miss, inval), b
            assert (st["deletes_applied"], st["adds_applied"]) == (nd - miss, len(adds)), b
            check_topology(e, og, f"batch {b}")
            check_incoming(e, og, f"batch {b}")
            check_traversal(e, og, "sssp", 0, cg.WEIGHT_HASH64, 5, where=f"batch {b}")


@pytest.mark.parametrize("others", [0, ONE])  # below and above the one-launch limit
@pytest.mark.parametrize("tier", ["hbm", "host"])
def test_short_rows_at_their_request_limits(tier, others):
    """Rows of 0 to 65 slots with up to 17 deletes each, around the 8 and 16
    that decide who claims: distinct, repeated and missing destinations."""
    print(f"[gpu-case] short rows {tier} others={others}", flush=True)
    rng = np.random.default_rng(others + 7)
    kinds = [(d, k) for d in (0, 1, 3, 4, 5, 15, 16, 17, 63, 64, 65) for k in (1, 7, 8, 9, 16, 17)]
    n = 4000
    deg = rng.integers(0, 60, n)
    deg[-4:] = 5000  # the budget goes to these
    deg[:len(kinds)] = [d for d, _ in kinds]
    off = np.zeros(n + 1, dtype=np.uint64)
    off[1:] = np.cumsum(deg)
    m = int(off[-1])
    g = cg.HostGraph(n, off, rng.integers(0, n, m).astype(np.uint32))
    g.dst[int(off[40]):int(off[len(kinds)])] %= 50  # parallel edges in the longer rows
    src = np.repeat(np.arange(n, dtype=np.uint32), deg)
    og = oracle_graph(g)
    with cg.Engine("sssp", weight_mode=cg.WEIGHT_HASH64, weight_seed=5,
                   cache_bytes=m if tier == "host" else 0) as e:
        e.load_graph(g)
        e.init_graph(0)
        e.start()
        for b in range(2):
            off, dst = og.csr()
            u, v = [], []
            for x, (_, k) in enumerate(kinds):
                row = dst[int(off[x]):int(off[x + 1])]
                take = rng.permutation(row)[:k]
                take = np.concatenate([take, rng.integers(0, n, k - len(take))])  # missing ones
                if k > 2 and x % 3 == 0:
                    take[-1] = take[0]  # one asked for twice
                u.append(np.full(k, x)), v.append(take)
            u, v = np.concatenate(u), np.concatenate(v)
            pick = rng.choice(m, others, replace=False)
            order = rng.permutation(len(u) + others)
            dels = cg.edges_array(np.concatenate([u, src[pick]])[order], np.concatenate([v, g.dst[pick]])[order])
            adds = cg.edges_array(rng.integers(0, len(kinds), 500), rng.integers(0, n, 500))
            st = e.apply_batch(dels, adds)
            miss, inval = oracle_apply(og, dels, adds)
            assert (st["missing_deletes"], st["invalid_updates"]) == (miss, inval), b
            assert st["deletes_applied"] == len(dels) - miss, b
            check_topology(e, og, f"batch {b}")
            check_incoming(e, og, f"batch {b}")
            check_traversal(e, og, "sssp", 0, cg.WEIGHT_HASH64, 5, where=f"batch {b}")
