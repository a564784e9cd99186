// Incremental BFS / SSSP from up to 64 sources at once.
//
// The reference maintains one source per engine (InitGraph takes the source,
// framework.cuh:991-1041; the batch path is update_tree_del / update_tree_add,
// framework.cuh:2139-2348, 2752-2894). Here one engine keeps k <= 64 sources
// current through every batch with the same steps as the single-source path
// (mutation, invalidation of parent-tree dependents, pull repair, insert
// seeding, push relaxation), each step done for all sources in one pass over
// the rows it touches:
//   st[v*k + s]  8 B  value << 32 | parent of v for source s (vertex-major:
//                     the k states of a vertex share cache lines)
//   act[v]       8 B  sources whose value at v improved, pending expansion
//   snap[v]      8 B  the round's snapshot of act (or of pinv)
//   affm[v]      8 B  sources for which v is affected in the current call
//   pinv[v]      8 B  affected bits not yet expanded by an invalidation wave
// Every per-edge step takes (edge, source) pairs, one per lane (pair_chunk):
// the states of one edge's sources lie next to each other, so a wave reads
// whole lines, and no lane idles whatever the masks are. Record steps take
// (record, source) pairs the same way. A vertex is queued exactly when its
// pending mask (act, or pinv in the invalidation) is non-zero: the lane whose
// atomicOr finds it zero appends the vertex. Bound by the latency of the
// rounds, whose frontiers are small, and by the random state reads: a lane
// per edge that walked the sources read 64 lines per load, and long rows took
// a third launch per round (64 sources of 2^18 vertices, batches of 6250 +
// 6250: 2.4 ms a batch, now 1.5).
#pragma once

namespace cig {
namespace dev {

struct MsiArgs {
    Ctl *ctl;
    const Row *rows;
    const Row *in_rows;  // incoming rows (rows + n, or rows for a symmetric graph)
    unsigned long long *st;
    unsigned long long *act, *snap, *affm, *pinv;
    uint32_t *q0, *q1;
    Tile *tiles;
    uint32_t *alist;
    ExpandCfg cfg;
    const cig_edge *dels;
    uint32_t nd;
    const cig_edge *adds;
    uint32_t na;
    const uint8_t *add_skip, *del_skip;  // grouped batches: cancelled records (may be null)
    uint32_t n, k;
    uint64_t seed;
    uint32_t ts;  // stage markers the kernel (or a chain's first round) notes
};

constexpr unsigned long long kMsiNone = ~0ull;  // value kInf, parent kNone

__device__ __forceinline__ uint32_t msi_bit(unsigned long long &m) {
    const uint32_t s = uint32_t(__ffsll(m) - 1);
    m &= m - 1;
    return s;
}

// Appends v to the pending frontier's queue, for few lanes.
__device__ __forceinline__ void msi_queue(const MsiArgs &a, uint32_t r, uint32_t v) {
    const uint32_t at = atomicAdd(&a.ctl->qcount[r % 3], 1u);
    ((r & 1) ? a.q1 : a.q0)[at] = v;
}

// Sources: state (0, none) and the first frontier. The host has set every
// state word to kMsiNone and every mask to 0.
__global__ void k_msi_init(MsiArgs a, SrcList sources) {
    const uint32_t r = a.ctl->round;
    for (uint32_t s = gthread(); s < a.k; s += gthreads()) {
        const uint32_t v = sources.v[s];
        a.st[uint64_t(v) * a.k + s] = uint64_t(kNone);  // value 0, no parent
        if (atomicOr(&a.act[v], 1ull << s) == 0ull) msi_queue(a, r, v);
    }
}

// Marks bits `m` of y affected and leaves the newly affected ones pending for
// the next invalidation wave; true when y had none pending (append it).
__device__ __forceinline__ bool msi_affect(unsigned long long *affm, unsigned long long *pinv, uint32_t y,
                                           unsigned long long m) {
    const unsigned long long gained = m & ~atomicOr(&affm[y], m);
    return gained && atomicOr(&pinv[y], gained) == 0ull;
}

// (record, source) pairs: a lane group of the next power of two >= k takes
// one record's sources, the loads of kMsiRecs records per group in flight
// together; the group's first lane acts for the record.
constexpr uint32_t kMsiRecs = 4;
struct MsiGroup {
    uint32_t s, rec, per;  // this lane's source, its record among the wave's `per` records a step
    unsigned long long sel;
    uint32_t shift;
};
__device__ __forceinline__ MsiGroup msi_group(uint32_t k) {
    uint32_t kw = 1;
    while (kw < k) kw <<= 1;
    MsiGroup g;
    g.s = lane_id() & (kw - 1);
    g.rec = lane_id() / kw;
    g.per = kWave / kw;
    g.shift = g.rec * kw;
    g.sel = kw == 64 ? ~0ull : (1ull << kw) - 1ull;
    return g;
}
// The sources of this lane's record whose flag is set.
__device__ __forceinline__ unsigned long long msi_bits(const MsiGroup &g, bool f) {
    return (__ballot(f) >> g.shift) & g.sel;
}

// reset_del_edges (driver.cuh:371-411) per source: a deleted (u,v) whose v
// has parent u for source s makes (v, s) affected. Parallel copies of (u,v)
// are treated conservatively, as in the single-source path.
__global__ __launch_bounds__(kBlock) void k_msi_inval_seed(MsiArgs a) {
    __shared__ ListStage stage;
    stamp_marks(a.ctl, a.ts);
    const uint32_t r = a.ctl->round;
    const StagedOut<1024, 2> out{Sink{(r & 1) ? a.q1 : a.q0, &a.ctl->qcount[r % 3]}, TileSink{nullptr, &a.ctl->scount},
                                 &stage};
    out_init(out);
    const MsiGroup g = msi_group(a.k);
    for (uint32_t base = gwave() * g.per * kMsiRecs; base < a.nd; base += gwaves() * g.per * kMsiRecs) {
        uint32_t u[kMsiRecs], v[kMsiRecs], par[kMsiRecs];
        bool on[kMsiRecs], push[kMsiRecs];
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            const uint32_t i = base + j * g.per + g.rec;
            on[j] = i < a.nd && !(a.del_skip && a.del_skip[i]);
            u[j] = v[j] = kNone;
            if (on[j]) {
                u[j] = a.dels[i].u;
                v[j] = a.dels[i].v;
            }
            on[j] = on[j] && g.s < a.k && u[j] < a.n && v[j] < a.n;
        }
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) par[j] = on[j] ? uint32_t(a.st[uint64_t(v[j]) * a.k + g.s]) : kNone;
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            const unsigned long long m = msi_bits(g, on[j] && par[j] == u[j]);
            push[j] = g.s == 0 && m != 0ull && msi_affect(a.affm, a.pinv, v[j], m);
        }
        out_push<kMsiRecs>(out, push, v);
    }
    out_flush(out);
}

// Invalidation wave (RelaxCTADB_del + PushFunctorDB_Del, sync_push_dd.cuh:
// 1220-1303): for each source s newly affected at x, a child y whose parent
// for s is x becomes affected for s.
struct MsiInvalOp {
    static constexpr int kGroup = 1, kUnroll = 4;
    using Loaded = uint32_t;
    const unsigned long long *snap;
    const unsigned long long *st;
    unsigned long long *affm, *pinv;
    uint32_t k;
    __device__ unsigned long long mask(uint32_t v) const { return snap[v]; }
    // a slot claimed by a delete of the same batch (the claims may run
    // beside the waves) holds kNone and no vertex
    __device__ void load(uint32_t, uint32_t y, uint32_t s, Loaded &x) const {
        x = y != kNone ? uint32_t(st[uint64_t(y) * k + s]) : kNone;
    }
    __device__ unsigned long long apply(uint32_t v, uint32_t, uint32_t s, unsigned long long, const Loaded &x) const {
        return x == v ? 1ull << s : 0ull;
    }
    __device__ bool mark(uint32_t y, unsigned long long m) const { return msi_affect(affm, pinv, y, m); }
};

// Push relaxation for every source pending at the expanding vertex
// (SyncPushDDB relax + AccumulateBuffer per source): an improvement is a
// 64-bit minimum of value << 32 | parent. A source counts as improved when its
// candidate beat the value read; if another lane lowered it further
// meanwhile, w is merely expanded once more for that source.
template <int W>
struct MsiRelaxOp {
    static constexpr int kGroup = 1, kUnroll = 4;
    struct Loaded {
        uint32_t du, dw;
    };
    unsigned long long *st;
    unsigned long long *act;
    const unsigned long long *snap;
    uint32_t k;
    uint64_t seed;
    __device__ unsigned long long mask(uint32_t v) const { return snap[v]; }
    __device__ void load(uint32_t u, uint32_t w, uint32_t s, Loaded &x) const {
        x.du = uint32_t(st[uint64_t(u) * k + s] >> 32);
        x.dw = uint32_t(st[uint64_t(w) * k + s] >> 32);
    }
    __device__ unsigned long long apply(uint32_t u, uint32_t w, uint32_t s, unsigned long long, const Loaded &x) const {
        const uint64_t c = uint64_t(x.du) + weight<W>(u, w, seed);
        if (c >= x.dw) return 0ull;  // also rejects c >= kInf
        __hip_atomic_fetch_min(&st[uint64_t(w) * k + s], (c << 32) | u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return 1ull << s;
    }
    __device__ bool mark(uint32_t w, unsigned long long m) const { return atomicOr(&act[w], m) == 0ull; }
};

// Round round+seq-1, phase 1 (relaxation or invalidation): snapshot and
// clear the pending masks `from` of the frontier and cut its long rows into
// tiles; workgroup 0 posts progress.
__global__ __launch_bounds__(kBlock) void k_msi_consume(MsiArgs a, unsigned long long *from, uint64_t *prog,
                                                        uint64_t tag, uint32_t seq) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->qcount[(r + 2) % 3] = 0;
        c->tcount[(r + 2) % 3] = 0;
        if (nq) c->rounds += 1;
        if (seq == 1) stamp_marks(c, a.ts);
        post_progress(prog, tag, nq != 0);
    }
    const uint32_t *qin = (r & 1) ? a.q1 : a.q0;
    Counters ctr;
    for (uint32_t base = blockIdx.x * blockDim.x; base < nq; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        const bool on = i < nq;
        uint32_t v = 0;
        Row row{};
        if (on) {
            v = qin[i];
            row = a.rows[v];
            a.snap[v] = from[v];
            from[v] = 0ull;
            ctr.scanned += row.deg;
            ctr.vexp += row.deg ? 1 : 0;
            if (row.off & kHostTier) ctr.host += row.deg;
        }
        pair_cut(a.cfg, pair_tile_len(a.cfg), v, row, on, a.tiles, &c->tcount[r % 3], scratch);
    }
    if (nq) flush_counters(ctr, a.cfg.stats, a.cfg.stage);
}

template <int W, bool INV>
__device__ __forceinline__ auto msi_op(const MsiArgs &a) {
    if constexpr (INV) return MsiInvalOp{a.snap, a.st, a.affm, a.pinv, a.k};
    else return MsiRelaxOp<W>{a.st, a.act, a.snap, a.k, a.seed};
}

// Phase 2: expand the frontier's rows and tiles. INV selects the invalidation
// wave, else the relaxation of weight kind W.
template <int W, bool INV>
__global__ __launch_bounds__(kBlock) void k_msi_expand(MsiArgs a, uint32_t seq) {
    using Op = decltype(msi_op<W, INV>(a));
    __shared__ PairLds<64> lds[kWavesPerBlock];
    __shared__ ListStage stage;
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    if (nq == 0) return;
    const Op op = msi_op<W, INV>(a);
    const StagedOut<1024, 2> out{Sink{(r & 1) ? a.q0 : a.q1, &c->qcount[(r + 1) % 3]}, TileSink{nullptr, &c->scount},
                                 &stage};
    out_init(out);
    PairLds<64> &L = lds[wave_in_block()];
    pair_range<1, Op::kUnroll>(op, a.cfg, a.rows, (r & 1) ? a.q1 : a.q0, nq, L, out);
    pair_tiles<1, Op::kUnroll>(op, a.cfg, a.tiles, c->tcount[r % 3], L, out);
    out_flush(out);
}

// reset_affected_values (driver.cuh:418-433) per source, over every vertex:
// each affected (v, s) restarts from (kInf, none), and v joins the affected
// list that the repair and the end-of-call clear walk.
__global__ void k_msi_reset(MsiArgs a) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    for (uint32_t base = blockIdx.x * blockDim.x; base < a.n; base += gthreads()) {
        const uint32_t v = base + threadIdx.x;
        unsigned long long m = v < a.n ? a.affm[v] : 0ull;
        const bool hit = m != 0ull;
        unsigned long long *sv = a.st + uint64_t(v) * a.k;
        while (m) sv[msi_bit(m)] = kMsiNone;
        block_append(hit, v, a.alist, &a.ctl->acount, scratch);
    }
}

// GpuAffectedPullRelax (framework.cuh:137-204) per source: each affected
// (y, s) takes the minimum over in-neighbours x not affected for s.
template <int W>
struct MsiPullOp {
    static constexpr int kGroup = 1, kUnroll = 4;
    struct Loaded {
        uint32_t vx, vy;
        bool ok;
    };
    unsigned long long *st;
    const unsigned long long *affm;
    unsigned long long *best;  // tiles: the wave's minimum per source, in LDS
    uint32_t k;
    uint64_t seed;
    __device__ unsigned long long mask(uint32_t y) const { return affm[y]; }
    __device__ void load(uint32_t y, uint32_t x, uint32_t s, Loaded &l) const {
        l.ok = ((affm[x] >> s) & 1ull) == 0ull;
        l.vx = uint32_t(st[uint64_t(x) * k + s] >> 32);
        l.vy = uint32_t(st[uint64_t(y) * k + s] >> 32);
    }
    __device__ unsigned long long apply(uint32_t y, uint32_t x, uint32_t s, unsigned long long, const Loaded &l) const {
        const uint64_t c = uint64_t(l.vx) + weight<W>(x, y, seed);
        if (l.ok && c < l.vy) {  // also rejects c >= kInf
            if (best) atomicMin(&best[s], (c << 32) | x);
            else __hip_atomic_fetch_min(&st[uint64_t(y) * k + s], (c << 32) | x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return 0ull;
    }
    __device__ bool mark(uint32_t, unsigned long long) const { return false; }
};

// The incoming rows of the affected vertices: short rows here, long rows cut
// into tiles for k_msi_repair_tiles.
template <int W>
__global__ __launch_bounds__(kBlock) void k_msi_repair(MsiArgs a) {
    __shared__ PairLds<64> lds[kWavesPerBlock];
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    Ctl *c = a.ctl;
    stamp_marks(c, a.ts);
    const uint32_t na = ld_acquire(&c->acount);
    if (na == 0) return;
    Counters ctr;
    for (uint32_t base = blockIdx.x * blockDim.x; base < na; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        uint32_t y = 0;
        Row row{};
        if (i < na) {
            y = a.alist[i];
            row = a.in_rows[y];
            ctr.scanned += row.deg;
            ctr.vexp += row.deg ? 1 : 0;
            if (row.off & kHostTier) ctr.host += row.deg;
        }
        pair_cut(a.cfg, pair_tile_len(a.cfg), y, row, i < na, a.tiles, &c->scount, scratch);
    }
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    const MsiPullOp<W> op{a.st, a.affm, nullptr, a.k, a.seed};
    pair_range<1, MsiPullOp<W>::kUnroll>(op, a.cfg, a.in_rows, a.alist, na, lds[wave_in_block()],
                                         DirectOut{Sink{nullptr, &c->scount}, TileSink{nullptr, &c->scount}});
}

// A tile's minimum per source is taken in LDS and leaves the wave as one
// atomic: all the tiles of a hub row start from kInf together, and an atomic
// per (edge, source) that beats it queues thousands of them at one address
// (64 sources, 2^18 vertices: 8 launches took 0.93 ms, now 0.47).
template <int W>
__global__ __launch_bounds__(kBlock) void k_msi_repair_tiles(MsiArgs a) {
    __shared__ PairLds<64> lds[kWavesPerBlock];
    __shared__ unsigned long long best_lds[kWavesPerBlock][kWave];
    Ctl *c = a.ctl;
    stamp_marks(c, a.ts);
    const uint32_t nt = ld_acquire(&c->scount);
    const uint32_t lane = lane_id();
    unsigned long long *best = best_lds[wave_in_block()];
    const MsiPullOp<W> op{a.st, a.affm, best, a.k, a.seed};
    const DirectOut none{Sink{nullptr, &c->scount}, TileSink{nullptr, &c->scount}};
    for (uint32_t t = gwave(); t < nt; t += gwaves()) {
        const Tile tile = a.tiles[t];
        best[lane] = kMsiNone;
        wave_lds_sync();
        pair_chunk<1, MsiPullOp<W>::kUnroll>(op, a.cfg.pools, tile.v, tile.start, lane == 0 ? tile.len : 0u,
                                             lane == 0 ? a.affm[tile.v] : 0ull, lds[wave_in_block()], none);
        wave_lds_sync();
        const unsigned long long b = best[lane];
        if (b != kMsiNone)
            __hip_atomic_fetch_min(&a.st[uint64_t(tile.v) * a.k + lane], b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// After the repair: every affected (y, s) that has a value again is pending
// expansion, and y joins the frontier of the current round.
__global__ __launch_bounds__(kBlock) void k_msi_repair_done(MsiArgs a) {
    __shared__ ListStage stage;
    const uint32_t cnt = ld_acquire(&a.ctl->acount);
    const uint32_t r = a.ctl->round;
    if (threadIdx.x == 0 && blockIdx.x == 0) a.ctl->scount = 0;
    if (cnt == 0) return;
    const StagedOut<1024, 2> out{Sink{(r & 1) ? a.q1 : a.q0, &a.ctl->qcount[r % 3]}, TileSink{nullptr, &a.ctl->scount},
                                 &stage};
    out_init(out);
    const MsiGroup g = msi_group(a.k);
    for (uint32_t base = gwave() * g.per * kMsiRecs; base < cnt; base += gwaves() * g.per * kMsiRecs) {
        uint32_t y[kMsiRecs], val[kMsiRecs];
        bool on[kMsiRecs], push[kMsiRecs];
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            const uint32_t i = base + j * g.per + g.rec;
            on[j] = i < cnt && g.s < a.k;
            y[j] = on[j] ? a.alist[i] : 0u;
        }
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            on[j] = on[j] && ((a.affm[y[j]] >> g.s) & 1ull);
            val[j] = on[j] ? uint32_t(a.st[uint64_t(y[j]) * a.k + g.s] >> 32) : kInf;
        }
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            const unsigned long long f = msi_bits(g, val[j] != kInf);
            push[j] = g.s == 0 && f != 0ull && atomicOr(&a.act[y[j]], f) == 0ull;
        }
        out_push<kMsiRecs>(out, push, y);
    }
    out_flush(out);
}

// SeedAddedEdgeFrontier (framework.cuh:238-294) per source: an inserted
// (u,v) offers value_s(u) + w to v for every source s not affected at u (an
// affected u re-expands its whole row once repaired).
template <int W>
__global__ __launch_bounds__(kBlock) void k_msi_insert_seed(MsiArgs a, uint32_t skip_affected) {
    __shared__ ListStage stage;
    stamp_marks(a.ctl, a.ts);
    const uint32_t r = a.ctl->round;
    const StagedOut<1024, 2> out{Sink{(r & 1) ? a.q1 : a.q0, &a.ctl->qcount[r % 3]}, TileSink{nullptr, &a.ctl->scount},
                                 &stage};
    out_init(out);
    const MsiGroup g = msi_group(a.k);
    for (uint32_t base = gwave() * g.per * kMsiRecs; base < a.na; base += gwaves() * g.per * kMsiRecs) {
        uint32_t u[kMsiRecs], v[kMsiRecs], du[kMsiRecs], dv[kMsiRecs];
        bool on[kMsiRecs], push[kMsiRecs];
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            const uint32_t i = base + j * g.per + g.rec;
            on[j] = i < a.na && !(a.add_skip && a.add_skip[i]);
            u[j] = v[j] = kNone;
            if (on[j]) {
                u[j] = a.adds[i].u;
                v[j] = a.adds[i].v;
            }
            on[j] = on[j] && g.s < a.k && u[j] < a.n && v[j] < a.n;
        }
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            if (skip_affected) on[j] = on[j] && !((a.affm[u[j]] >> g.s) & 1ull);
            du[j] = on[j] ? uint32_t(a.st[uint64_t(u[j]) * a.k + g.s] >> 32) : kInf;
            dv[j] = on[j] ? uint32_t(a.st[uint64_t(v[j]) * a.k + g.s] >> 32) : 0u;
        }
#pragma unroll
        for (uint32_t j = 0; j < kMsiRecs; ++j) {
            const uint64_t c = uint64_t(du[j]) + weight<W>(u[j], v[j], a.seed);
            const bool better = on[j] && c < dv[j];  // also rejects c >= kInf
            if (better)
                __hip_atomic_fetch_min(&a.st[uint64_t(v[j]) * a.k + g.s], (c << 32) | u[j], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long f = msi_bits(g, better);
            push[j] = g.s == 0 && f != 0ull && atomicOr(&a.act[v[j]], f) == 0ull;
        }
        out_push<kMsiRecs>(out, push, v);
    }
    out_flush(out);
}

// End of a call: the affected marks of the listed vertices go back to 0.
__global__ void k_msi_clear(MsiArgs a) {
    const uint32_t cnt = ld_acquire(&a.ctl->acount);
    for (uint32_t i = gthread(); i < cnt; i += gthreads()) {
        const uint32_t v = a.alist[i];
        a.affm[v] = 0ull;
        a.pinv[v] = 0ull;
    }
}

}  // namespace dev
}  // namespace cig
