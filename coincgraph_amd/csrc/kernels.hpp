// Kernels of the incremental graph engine. Included once, by engine.hip.
#pragma once
#include <hip/hip_cooperative_groups.h>
#include <hip/hip_runtime.h>

#include "../../include/cig.h"
#include "device.hpp"

namespace cig {
namespace dev {

namespace cg = cooperative_groups;

// LDS staging of the round kernels: 2048 frontier items and 128 tiles per
// workgroup (19 KB with the wave slots of a 256-thread workgroup).
using RoundStage = StageLds<2048, 128>;
// and of kernels that make no tiles: small, so that many workgroups fit on a CU.
using ListStage = StageLds<1024, 2>;

__device__ __forceinline__ uint64_t next_pow2_dev(uint64_t d) {
    uint64_t c = d < kMinRowCap ? kMinRowCap : d;
    return c <= 1 ? 1 : (1ull << (64 - __builtin_clzll(c - 1)));
}

__device__ __forceinline__ uint32_t gthread() { return blockIdx.x * blockDim.x + threadIdx.x; }
__device__ __forceinline__ uint32_t gthreads() { return gridDim.x * blockDim.x; }
__device__ __forceinline__ uint32_t gwave() { return blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; }
__device__ __forceinline__ uint32_t gwaves() { return gridDim.x * (blockDim.x / kWave); }

// ------------------------------------------------------------- small kernels
// Zero-fills a 32-bit range (used instead of hipMemsetAsync so the batch chain
// stays capturable in a HIP graph).
__global__ void k_fill32(uint32_t *p, uint64_t n, uint32_t value) {
    for (uint64_t i = gthread(); i < n; i += gthreads()) p[i] = value;
}

// Stage markers of a call: the kernel that follows a marker notes the device's
// constant-rate clock for it (bit k of mask: marker k) when it starts. An
// event record is a packet of its own that idles the stream for a few
// microseconds, and a call has up to ten markers. With k_end_call in
// place of three kernels, four phases of 500 records on 4,096 vertices and a
// result copy: 725 us before, 614 now; two calls of 1000 + 1000 on 65,536
// vertices and a result copy: 550 and 456 us.
__device__ __forceinline__ void stamp_marks(Ctl *c, uint32_t mask) {
    if (mask == 0 || blockIdx.x != 0 || threadIdx.x != 0) return;
    const uint64_t t = wall_clock64();
    for (uint32_t k = 0; k < 10; ++k)
        if ((mask >> k) & 1u) c->ts[k] = t;
}

// Markers that no kernel of the call's own can note.
__global__ void k_mark(Ctl *c, uint32_t mask) { stamp_marks(c, mask); }

// Per-call reset of the control block counters (not the round state).
// flags: kResetKeepRounds keeps the round state; kResetKeepMut keeps the
// mutation counters (the second stream resets those itself, k_reset_mut);
// kResetStamp: a call starts here.
constexpr uint32_t kResetKeepRounds = 1u, kResetKeepMut = 2u, kResetStamp = 4u;
__global__ void k_reset_ctl(Ctl *c, uint32_t flags) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (flags & kResetStamp) stamp_marks(c, 1u << 0);
    const bool keep_rounds = flags & kResetKeepRounds;
    c->acount = 0;
    c->icount[0] = c->icount[1] = c->icount[2] = 0;
    c->ifront[0] = c->ifront[1] = c->ifront[2] = 0;
    c->iround = 0;
    c->scount = 0;
    if (!(flags & kResetKeepMut)) {
        c->touched = 0;
        c->small_cnt = c->big_cnt = c->add_cnt = c->copy_cnt = c->overflow_cnt = 0;
        c->mid_cnt = c->mid_host_cnt = c->mid16_cnt = 0;
        c->dtile_cnt = c->ht_cursor = 0;
        c->group_cursor = 0;
    }
    c->pr_invalid = 0;
    c->pull_rounds = 0;
    c->edges_scanned = c->host_edges = c->vexp = 0;
    c->deletes_applied = c->missing = c->invalid = c->adds_applied = c->relocated = 0;
    c->touched_sources = 0;
    c->rounds = 0;
    c->residual_l1 = 0;
    c->converged = 0;
    for (int i = 0; i < 4; ++i) c->st_edges[i] = c->st_vexp[i] = c->st_host[i] = 0;
    if (!keep_rounds) {
        c->round = 1;
        for (int i = 0; i < 3; ++i) c->qcount[i] = c->tcount[i] = c->fscan[i] = c->flist[i] = 0;
    }
}

// Clears the per-mutation lists between the two stages of a staged batch.
__global__ void k_reset_mut(Ctl *c) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    c->touched = 0;
    c->small_cnt = c->big_cnt = c->add_cnt = c->copy_cnt = c->overflow_cnt = 0;
    c->mid_cnt = c->mid_host_cnt = c->mid16_cnt = 0;
    c->dtile_cnt = c->ht_cursor = 0;
    c->group_cursor = 0;
}

// InitGraph (driver.cuh:186-206): traversal state words and the first frontier.
// kind 0: single source (SSSP/BFS), kind 1: vertex seeds (CC, label = own id).
__global__ void k_init_traversal(uint64_t *state, uint32_t *stamp, uint32_t n, uint32_t kind,
                                 uint32_t source, uint32_t *q, Ctl *c) {
    const uint32_t r = c->round;
    for (uint32_t v = gthread(); v < n; v += gthreads()) {
        if (kind == 1) {
            state[v] = (uint64_t(v) << 32) | kNone;
            stamp[v] = r;
            q[v] = v;
        } else {
            state[v] = v == source ? (uint64_t(0) << 32 | kNone) : ~0ull;
            stamp[v] = v == source ? r : 0;
        }
    }
    if (gthread() == 0) {
        if (kind == 0) q[0] = source;
        c->qcount[r % 3] = kind == 1 ? n : 1;
    }
}

// pr::Initialize (pr_residual.cuh:44-53) with the Kahan compensation array.
__global__ void k_init_pr(float *rank, float *comp, float *res, uint32_t *queued, uint32_t *q,
                          uint32_t n, Ctl *c) {
    const uint32_t r = c->round;
    for (uint32_t v = gthread(); v < n; v += gthreads()) {
        rank[v] = 0.0f;
        comp[v] = 0.0f;
        res[v] = 0.15f;
        queued[v] = 1u;
        q[v] = v;
    }
    if (gthread() == 0) c->qcount[r % 3] = n;
}

// ------------------------------------------------------------------ mutation
// A batch's records in device memory. Launches replayed from a captured
// HIP graph read the records through it (the graph's arguments stay the
// same for every batch; a one-thread kernel before each replay fills it).
struct BatchRef {
    const cig_edge *dels;
    const cig_edge *adds;
    uint32_t nd, na;
};

__global__ void k_set_batch(BatchRef *ref, const cig_edge *dels, uint32_t nd, const cig_edge *adds, uint32_t na) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *ref = BatchRef{dels, adds, nd, na};
}

// Update records from the caller's vertex ids to a renumbered engine's;
// ids >= n stay as they are, so invalid records are still rejected.
__global__ void k_map_records(cig_edge *r, uint64_t cnt, const uint32_t *perm, uint32_t n) {
    for (uint64_t i = gthread(); i < cnt; i += gthreads()) {
        cig_edge e = r[i];
        if (e.u < n) e.u = perm[e.u];
        if (e.v < n) e.v = perm[e.v];
        r[i] = e;
    }
}

// Freed blocks of the pinned host tier, one stack per size class (class =
// log2 of the block's slots). A relocated host-tier row's old block is pushed
// once its slots have been copied (k_fl_release, after k_add_copy; tier
// moves: k_move_release after k_move_rows), and a later relocation or
// eviction of the same class pops it instead of growing the tail. Pushes and
// pops never share a launch. A full stack drops the block, which stays
// garbage until the tier is packed; packing the tier empties every stack.
struct FreeList {
    unsigned long long *off;  // [kFlClasses * cap] block offsets (tier bit clear); null: no list
    int *cnt;                 // [kFlClasses]
    uint32_t cap;
};
constexpr uint32_t kFlClasses = 32;

__device__ __forceinline__ uint32_t fl_class(uint64_t cap) { return 63u - uint32_t(__clzll(cap)); }

__device__ __forceinline__ bool fl_pop(const FreeList &f, uint32_t cls, uint64_t &off) {
    if (!f.off) return false;
    const int old = atomicSub(&f.cnt[cls], 1);
    if (old > 0) {
        off = f.off[uint64_t(cls) * f.cap + uint32_t(old - 1)];
        return true;
    }
    atomicAdd(&f.cnt[cls], 1);  // empty: undo (no push runs in the same launch)
    return false;
}

__device__ __forceinline__ void fl_push(const FreeList &f, uint32_t cls, uint64_t off) {
    if (!f.off) return;
    const int at = atomicAdd(&f.cnt[cls], 1);
    if (at < int(f.cap)) f.off[uint64_t(cls) * f.cap + uint32_t(at)] = off;
    else atomicSub(&f.cnt[cls], 1);  // full: the block stays garbage
}

struct MutArgs {
    Ctl *ctl;
    Row *rows;
    Pools pools;
    FreeList fl;       // host-tier free blocks (see FreeList)
    uint32_t n;
    uint32_t rev;      // 1: rows [n, 2n) hold the incoming rows and get every update mirrored
    const cig_edge *dels;
    uint32_t nd;
    const cig_edge *adds;
    uint32_t na;
    uint64_t *cnt64;   // per vertex: deletes (low) | adds (high) of this call
    uint32_t *rslot;   // per record: its rank among its row's deletes (or adds), from k_count
    uint64_t *gofs;    // per vertex offset of its group in `grouped`
    uint32_t *touched;
    uint32_t *grouped;
    uint32_t *small_list;
    uint32_t *mid_list;   // medium rows with deletes (k_del_rows): HBM-tier rows from the
                          // front, host-tier rows from the back (n << rev entries)
    uint32_t *mid16_list; // HBM-tier medium rows with 9-16 deletes (n << rev entries)
    uint32_t *big_list;
    uint32_t *add_list;
    uint32_t *overflow;
    // long-row deletes
    uint32_t *htoff;   // per vertex: offset of its delete table (kNone: none)
    uint32_t *hkeys;   // delete tables: destination + 1 (0 = empty)
    uint2 *hcnts;      // delete tables: (requested, claimed)
    uint32_t *hcnt;    // per vertex: holes found (zero between calls)
    uint8_t *dclass;   // per row: delete class of this call (kDelClass*)
    const uint8_t *skip;  // grouped batches: 1 = record cancelled (adds [0,na), deletes [na,na+nd)); may be null
    struct DelTile *dtiles;  // long-row delete scan tiles (DelTile below)
    struct AddPiece *pieces;  // copy pieces of the insert phase (AddPiece below)
    StatShard *stats;
    uint32_t *hot;     // per row activity of the current window (null: not counted)
    const BatchRef *ref;  // non-null: the records are read from here (graph replays)
    uint32_t ts;          // stage markers the hole fixes note
};

// The call's records: from the batch reference when there is one.
template <class A>
__device__ __forceinline__ uint32_t rec_nd(const A &a) { return a.ref ? a.ref->nd : a.nd; }
template <class A>
__device__ __forceinline__ uint32_t rec_na(const A &a) { return a.ref ? a.ref->na : a.na; }
template <class A>
__device__ __forceinline__ const cig_edge *rec_dels(const A &a) { return a.ref ? a.ref->dels : a.dels; }
template <class A>
__device__ __forceinline__ const cig_edge *rec_adds(const A &a) { return a.ref ? a.ref->adds : a.adds; }

// Deletes find their slot by row length (BuildDeletionPlan,
// source_local_chunk_store.h:670-723, restated for the device):
//  - tiny rows (<= 64 slots): one lane per delete record reads the whole row
//    and claims a matching slot with a CAS (slot := kNone); in the host tier
//    only those with more than kDelWaveMax deletes: a lane's 16-B reads cross
//    the host link one by one, a 16-lane group's as whole lines and once per
//    row (480k delete records of 500,009 vertices with 30% of the edges in
//    HBM: 4.2 -> 4.0 ms, which is the link's 53 GB/s);
//  - medium rows (<= 4096 slots, host-tier rows of any length up to that; <= kDelWaveMax deletes; HBM rows with up to
//    kDelWaveMax16 in a second kernel): a 16-lane group per row against all
//    of the row's deletes at once, 256 slots a step;
//  - other rows: tiles of kDelTile slots over the whole grid against the
//    row's delete multiset in an open-addressing table of 2^bits >= 2*nd
//    slots.
// Every claimed slot is recorded in the row's hole list (the row's group,
// whose delete records are not read again). Rows with at most 16 deletes
// (and no table) are then compacted by one thread, the others by a
// workgroup: live slots of the last k positions move into the holes below
// deg-k. Equal destinations are interchangeable, so the survivor multiset is
// the reference's; their order may differ (CompactSourceInPlace,
// source_local_chunk_store.h:733-780, keeps it).
constexpr uint32_t kDelTile = 4096;
constexpr uint32_t kDelLdsKeys = 2048;

// Everything a scan tile needs, written by k_plan so that the tile's row
// loads depend on one record read only.
struct DelTile {
    uint64_t off;   // pool offset of the tile's first slot (tier bit kept)
    uint32_t row, start, len, to, bits, pad;
};
static_assert(sizeof(DelTile) == 32, "DelTile layout");
constexpr uint32_t kDelTinyDeg = 64, kDelMediumDeg = 4096, kDelThreadFix = 16;
enum : uint8_t { kDelClassNone = 0, kDelClassTiny = 1, kDelClassMedium = 2, kDelClassLong = 3, kDelClassMedium16 = 4 };

// A medium row with many deletes is cheaper as one tile against its table
// than as one wave per delete (each of which may read the whole row).
constexpr uint32_t kDelWaveMax = 8;
// In large batches, HBM-tier medium rows with more deletes, up to this many,
// take a second medium-row pass whose groups hold 16 requests (one tile
// against the row's table costs far more for a row of a few thousand
// slots); the 8-request kernel keeps its registers. Batches of fewer delete
// records (mirrors included) than kMid16MinRecords have few such rows and
// keep the plain form, which saves them the extra classification and
// workgroups.
constexpr uint32_t kDelWaveMax16 = 16;
constexpr uint64_t kMid16MinRecords = 1u << 20;
// Batches of at most this many delete records (mirrors included; graph
// replays, whose count the host does not know, never) claim in one launch
// (k_del_claims): two batches of 2,000 records with a result copy 460 us in
// three launches, 425 in one; eight of 12,500 records on 64 maintained
// sources 8.50 and 8.35 ms. Larger ones want the waves that the kinds' own
// register and LDS needs allow: sixteen batches of 200,000 records 10.65 ms
// in three launches, 12.1 in one; 125,000 the same in both.
constexpr uint64_t kOneClaimRecords = 1u << 14;
static_assert(kOneClaimRecords < kMid16MinRecords, "k_del_claims has no 16-request rows");

template <bool M16>
__device__ __forceinline__ uint8_t del_class(uint32_t nd, uint32_t deg, bool host) {
    if (nd == 0) return kDelClassNone;
    if (deg <= kDelTinyDeg && !(host && nd <= kDelWaveMax)) return kDelClassTiny;
    if (deg > kDelMediumDeg) return kDelClassLong;
    if (nd <= kDelWaveMax) return kDelClassMedium;
    return M16 && nd <= kDelWaveMax16 && !host ? kDelClassMedium16 : kDelClassLong;
}

__device__ __forceinline__ uint32_t del_table_bits(uint32_t nd) {
    uint32_t bits = 4;
    while ((1ull << bits) < 2ull * nd) ++bits;
    return bits;
}

__device__ __forceinline__ uint32_t ht_hash(uint32_t x, uint32_t bits) {
    return (x * 0x9E3779B1u) >> (32 - bits);
}

// Record i of a mutation call: deletes then adds; with the incoming index on,
// records [nd+na, 2(nd+na)) are the same updates mirrored onto row n+v with
// destination u.
struct MutRecord {
    uint32_t row, dst;
    bool del, valid, bad, mirror;
};

__device__ __forceinline__ MutRecord mut_record(const MutArgs &a, uint32_t i) {
    const uint32_t nd = rec_nd(a), na = rec_na(a);
    const uint32_t total = nd + na;
    MutRecord r;
    r.mirror = i >= total;
    const uint32_t j = r.mirror ? i - total : i;
    r.del = j < nd;
    const cig_edge e = r.del ? rec_dels(a)[j] : rec_adds(a)[j - nd];
    r.bad = !(e.u < a.n && e.v < a.n);
    r.valid = !r.bad && !(a.skip && a.skip[r.del ? na + j : j - nd]);
    r.row = r.mirror ? a.n + e.v : e.u;
    r.dst = r.mirror ? e.u : e.v;
    return r;
}

__device__ __forceinline__ uint32_t mut_records(const MutArgs &a) { return (rec_nd(a) + rec_na(a)) << a.rev; }

// Delete record i of [0, nd << rev): the deletes, then their mirrors.
__device__ __forceinline__ MutRecord del_record(const MutArgs &a, uint32_t i) {
    const uint32_t nd = rec_nd(a);
    return mut_record(a, i < nd ? i : i - nd + nd + rec_na(a));
}

// GroupedUpdateBatch (effective_update_batch.h:35-87) on the device: count
// records per row and collect the touched rows. The count's atomic also
// ranks the record among its row's deletes (or adds), which k_scatter uses
// as its slot. A thread takes four records a step, so the touched-list
// reservation is one atomic per 1024 records.
__global__ void k_count(MutArgs a) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    constexpr uint32_t R = 4;
    const uint32_t total = mut_records(a);
    uint64_t bad_total = 0, fwd_touched = 0;
    for (uint32_t base = blockIdx.x * blockDim.x * R; base < total; base += gthreads() * R) {
        uint32_t u[R];
        bool first[R];
        uint32_t nf = 0;
#pragma unroll
        for (uint32_t k = 0; k < R; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            first[k] = false;
            u[k] = 0;
            bool bad = false;
            if (i < total) {
                const MutRecord r = mut_record(a, i);
                if (!r.valid) {
                    bad = r.bad && !r.mirror;
                } else {
                    u[k] = r.row;
                    const uint64_t old = atomicAdd((unsigned long long *)&a.cnt64[r.row],
                                                   r.del ? 1ull : (1ull << 32));
                    a.rslot[i] = r.del ? uint32_t(old) : uint32_t(old >> 32);
                    first[k] = old == 0;
                }
            }
            bad_total += uint32_t(__popcll(__ballot(bad)));
            fwd_touched += uint32_t(__popcll(__ballot(first[k] && u[k] < a.n)));
            nf += first[k] ? 1u : 0u;
        }
        uint32_t at = block_reserve<uint32_t>(nf, &a.ctl->touched, scratch);
#pragma unroll
        for (uint32_t k = 0; k < R; ++k)
            if (first[k]) a.touched[at++] = u[k];
    }
    StatShard *sh = stat_shard(a.stats);
    stat_add(&sh->invalid, bad_total);
    stat_add(&sh->touched, fwd_touched);
}

// Reserves each touched row's group and classifies its work; long rows
// with deletes also reserve their table and scan tiles. All cursors (eight,
// nine with M16: the 16-request medium rows of a large batch) are reserved
// together, one round trip per workgroup step.
template <bool M16>
__global__ void k_plan(MutArgs a) {
    constexpr int NC = M16 ? 9 : 8;
    __shared__ uint32_t scratch[NC * (kMaxWavesPerBlock + 1)];
    const uint32_t touched = ld_acquire(&a.ctl->touched);
    uint32_t *ctr[NC];
    ctr[0] = &a.ctl->group_cursor;
    ctr[1] = &a.ctl->ht_cursor;
    ctr[2] = &a.ctl->dtile_cnt;
    ctr[3] = &a.ctl->small_cnt;
    ctr[4] = &a.ctl->big_cnt;
    ctr[5] = &a.ctl->add_cnt;
    ctr[6] = &a.ctl->mid_cnt;
    ctr[7] = &a.ctl->mid_host_cnt;
    if constexpr (M16) ctr[8] = &a.ctl->mid16_cnt;
    for (uint32_t base = blockIdx.x * blockDim.x; base < touched; base += gthreads()) {
        const uint32_t t = base + threadIdx.x;
        uint32_t u = 0, nd = 0, na = 0, deg = 0;
        bool host = false;
        uint8_t cls = kDelClassNone;
        if (t < touched) {
            u = a.touched[t];
            const uint64_t c = a.cnt64[u];
            nd = uint32_t(c);
            na = uint32_t(c >> 32);
            const Row row = a.rows[u];
            deg = row.deg;
            host = (row.off & kHostTier) != 0;
            cls = del_class<M16>(nd, deg, host);
            a.dclass[u] = cls;
        }
        const bool table = cls == kDelClassLong;
        const bool thread_fix = nd != 0 && nd <= kDelThreadFix && !table;
        uint32_t x[NC];
        x[0] = nd + na;
        x[1] = table ? (1u << del_table_bits(nd)) : 0u;
        x[2] = table ? (deg + kDelTile - 1) / kDelTile : 0u;
        x[3] = thread_fix ? 1u : 0u;
        x[4] = (nd != 0 && !thread_fix) ? 1u : 0u;
        x[5] = na != 0 ? 1u : 0u;
        x[6] = cls == kDelClassMedium && !host ? 1u : 0u;
        x[7] = cls == kDelClassMedium && host ? 1u : 0u;
        if constexpr (M16) x[8] = cls == kDelClassMedium16 ? 1u : 0u;
        uint32_t at[NC];
        block_reserve_n<NC>(x, ctr, at, scratch);
        if (t < touched) {
            a.gofs[u] = at[0];
            a.htoff[u] = table ? at[1] : kNone;
            if (x[2]) {
                const uint64_t off = a.rows[u].off;
                const uint32_t bits = del_table_bits(nd);
                for (uint32_t j = 0; j < x[2]; ++j) {
                    DelTile dt;
                    dt.off = off + uint64_t(j) * kDelTile;
                    dt.row = u;
                    dt.start = j * kDelTile;
                    dt.len = min(kDelTile, deg - j * kDelTile);
                    dt.to = at[1];
                    dt.bits = bits;
                    dt.pad = 0;
                    a.dtiles[at[2] + j] = dt;
                }
            }
            if (x[3]) a.small_list[at[3]] = u;
            if (x[4]) a.big_list[at[4]] = u;
            if (x[5]) a.add_list[at[5]] = u;
            if (x[6]) a.mid_list[at[6]] = u;
            if (x[7]) a.mid_list[(a.n << a.rev) - 1u - at[7]] = u;
            if constexpr (M16)
                if (x[8]) a.mid16_list[at[8]] = u;
        }
    }
}

// Groups the records by source; deletes of long rows also enter their
// row's table (destination -> requested count).
__global__ void k_scatter(MutArgs a) {
    const uint32_t total = mut_records(a);
    for (uint32_t i = gthread(); i < total; i += gthreads()) {
        const MutRecord r = mut_record(a, i);
        if (!r.valid) continue;
        const uint32_t nd = uint32_t(a.cnt64[r.row]);
        const uint32_t slot = r.del ? a.rslot[i] : nd + a.rslot[i];
        a.grouped[a.gofs[r.row] + slot] = r.dst;
        const uint32_t to = r.del ? a.htoff[r.row] : kNone;
        if (to != kNone) {
            // at most nd distinct keys in 2^bits >= 2*nd slots: the probe ends
            const uint32_t bits = del_table_bits(nd), mask = (1u << bits) - 1u;
            uint32_t h = ht_hash(r.dst, bits);
            for (;;) {
                const uint32_t prev = atomicCAS(&a.hkeys[to + h], 0u, r.dst + 1u);
                if (prev == 0u || prev == r.dst + 1u) break;
                h = (h + 1u) & mask;
            }
            atomicAdd(&a.hcnts[to + h].x, 1u);
        }
    }
}

// Records a claimed slot in its row's hole list.
__device__ __forceinline__ void del_hole(const MutArgs &a, uint32_t row, uint32_t slot) {
    a.grouped[a.gofs[row] + atomicAdd(&a.hcnt[row], 1u)] = slot;
}

// Tiny rows: one lane per delete record.
__device__ void del_lane_body(const MutArgs &a, uint32_t bid, uint32_t nb) {
    const uint32_t total = rec_nd(a) << a.rev;
    for (uint32_t i = bid * blockDim.x + threadIdx.x; i < total; i += nb * blockDim.x) {
        const MutRecord r = del_record(a, i);
        if (!r.valid || a.dclass[r.row] != kDelClassTiny) continue;
        const Row row = a.rows[r.row];
        if (row.deg == 0) continue;  // nothing to delete: a missing record
        uint32_t *p = a.pools.row(row.off);
        const uint32_t nq = (row.deg + 3u) >> 2;  // 1..16
        uint32_t d[kDelTinyDeg / 4][4], live[kDelTinyDeg / 4];
#pragma unroll
        for (uint32_t q = 0; q < kDelTinyDeg / 4; ++q) {
            live[q] = load_quad(p, q < nq ? q : nq - 1, row.deg, d[q]);
            if (q >= nq) live[q] = 0;
        }
        // a row with one delete record has one claimant: a plain store
        // (for host-tier rows a CAS is an atomic over the host link)
        const bool sole = uint32_t(a.cnt64[r.row]) == 1u;
        bool done = false;
#pragma unroll
        for (uint32_t q = 0; q < kDelTinyDeg / 4; ++q)
#pragma unroll
            for (uint32_t s = 0; s < 4; ++s)
                if (!done && s < live[q] && d[q][s] == r.dst &&
                    (sole ? (p[4 * q + s] = kNone, true) : atomicCAS(&p[4 * q + s], r.dst, kNone) == r.dst)) {
                    del_hole(a, r.row, 4 * q + s);
                    done = true;
                }
    }
}

// Medium rows (HBM: 64 < deg <= 4096 slots, host tier: up to 4096, none
// included; at most K deletes: kDelWaveMax, or kDelWaveMax16 for the HBM rows
// of the second kernel): one
// 16-lane group per row (four rows per wave) reads the row once, 256 slots
// a step, against all of the row's requested destinations, which the
// group's lanes hold in registers (a destination requested twice is two
// requests). The group owns the row, so a slot equal to a destination with
// an open request is claimed with a plain store and its index goes to the
// row's hole list; the group stops as soon as every request is claimed. (A
// group per delete record would read the row once per request.) Q quads
// per lane a step: 4 for HBM rows; host-tier rows take 2 (HOST), since
// what a step reads past the last claim costs host-link bandwidth, which
// bounds them.
template <uint32_t Q, bool HOST, uint32_t K = kDelWaveMax>
__device__ void del_rows_body(const MutArgs &a, uint32_t bid, uint32_t nb) {
    constexpr uint32_t G = 16, GPW = kWave / G;
    static_assert(K <= G, "a group holds its row's requests");
    static_assert(!(HOST && K > kDelWaveMax), "the 16-request rows are HBM rows");
    constexpr bool M16 = K > kDelWaveMax;
    static_assert(4 * Q <= 32, "candidate bits fit one word");
    const uint32_t cnt = ld_acquire(M16 ? &a.ctl->mid16_cnt : HOST ? &a.ctl->mid_host_cnt : &a.ctl->mid_cnt);
    const uint32_t lane = lane_id(), g = lane / G, gl = lane % G;
    const uint64_t gmask = ((1ull << G) - 1ull) << (g * G);
    const uint32_t wpb = blockDim.x / kWave;
    for (uint32_t base = (bid * wpb + wave_in_block()) * GPW; base < cnt; base += nb * wpb * GPW) {
        const uint32_t i = base + g;
        uint32_t u = 0, nd = 0, nq = 0, deg = 0;
        uint32_t *grp = nullptr, *p = nullptr;
        if (i < cnt) {
            u = M16 ? a.mid16_list[i] : a.mid_list[HOST ? (a.n << a.rev) - 1u - i : i];
            nd = min(uint32_t(a.cnt64[u]), K);
            const Row row = a.rows[u];
            deg = row.deg;
            nq = (deg + 3u) >> 2;
            grp = a.grouped + a.gofs[u];  // the requests, then the hole list
            p = a.pools.row(row.off);
        }
        const uint32_t mine = gl < nd ? grp[gl] : kNone;
        uint32_t key[K];
#pragma unroll
        for (uint32_t j = 0; j < K; ++j) key[j] = __shfl(mine, int(g * G + j), kWave);
        // the most requests any of the wave's rows has: the match below
        // compares against that many keys only (most medium rows have one or
        // two deletes, so most waves skip most of the eight compares a slot)
        uint32_t wmax = nd;
        wmax = max(wmax, uint32_t(__shfl_xor(int(wmax), 16, kWave)));
        wmax = max(wmax, uint32_t(__shfl_xor(int(wmax), 32, kWave)));
        uint32_t open = (1u << nd) - 1u;  // uniform within the group
        uint32_t holes = 0;               // uniform within the group
        for (uint32_t q0 = 0; __ballot(open != 0u && q0 < nq) != 0; q0 += G * Q) {
            uint32_t d[Q][4], cand = 0;  // bit 4k+s: slot (k, s) equals an open request
            if (open != 0u && q0 < nq) {
                uint32_t livemask = 0;
#pragma unroll
                for (uint32_t k = 0; k < Q; ++k) {
                    const uint32_t q = q0 + k * G + gl;
                    uint32_t live = load_quad(p, q < nq ? q : nq - 1, deg, d[k]);
                    if (q >= nq) live = 0;
                    livemask |= ((1u << live) - 1u) << (4 * k);
                }
                // claimed and unused requests hold kNone, which no live slot holds
#pragma unroll
                for (uint32_t j = 0; j < K; ++j) {
                    if (j >= wmax) break;  // wave-uniform
#pragma unroll
                    for (uint32_t k = 0; k < Q; ++k)
#pragma unroll
                        for (uint32_t s = 0; s < 4; ++s)
                            if (key[j] == d[k][s]) cand |= 1u << (4 * k + s);
                }
                cand &= livemask;
            }
            // each group claims its candidates one at a time, in lane order
            for (;;) {
                const uint64_t any = __ballot(cand != 0u);
                if (any == 0) break;
                const uint64_t mineg = any & gmask;
                const uint32_t leader = mineg ? uint32_t(__ffsll((unsigned long long)mineg) - 1) : g * G;
                uint32_t claimed = kNone, slot = 0;
                if (mineg && lane == leader) {
                    const uint32_t b = uint32_t(__ffs(cand) - 1);
                    cand &= cand - 1u;
                    const uint32_t x = d[b >> 2][b & 3u];
                    uint32_t m = 0;
#pragma unroll
                    for (uint32_t j = 0; j < K; ++j) m |= (key[j] == x ? 1u : 0u) << j;
                    m &= open;
                    if (m) {
                        claimed = uint32_t(__ffs(m) - 1);
                        slot = 4u * (q0 + (b >> 2) * G + gl) + (b & 3u);
                        p[slot] = kNone;
                    }
                }
                claimed = __shfl(claimed, int(leader), kWave);
                slot = __shfl(slot, int(leader), kWave);
                if (claimed != kNone) {
                    open &= ~(1u << claimed);
#pragma unroll
                    for (uint32_t j = 0; j < K; ++j)
                        if (j == claimed) key[j] = kNone;
                    if (gl == 0) grp[holes] = slot;  // the requests were read into registers above
                    ++holes;
                }
                if (open == 0u) cand = 0;
            }
        }
        if (i < cnt && gl == 0) a.hcnt[u] = holes;  // zero before the call; this group is its only writer
    }
}

template <uint32_t Q, bool HOST, uint32_t K = kDelWaveMax>
__global__ __launch_bounds__(kBlock) void k_del_rows(MutArgs a) { del_rows_body<Q, HOST, K>(a, blockIdx.x, gridDim.x); }

// The tiny-row claims and the host-tier medium rows in one launch (disjoint
// rows): workgroups [0, split) take the records of tiny rows, [split,
// split2) the host-tier rows, whose reads wait on the host link. With M16
// (a large batch) the workgroups from split2 on take the HBM medium rows
// with 9-16 deletes (a launch of their own would add a kernel boundary).
template <bool M16>
__global__ __launch_bounds__(kBlock) void k_del_lane_host(MutArgs a, uint32_t split, uint32_t split2) {
    if (blockIdx.x < split) del_lane_body(a, blockIdx.x, split);
    else if (!M16 || blockIdx.x < split2) del_rows_body<2, true>(a, blockIdx.x - split, split2 - split);
    else if constexpr (M16) del_rows_body<4, false, kDelWaveMax16>(a, blockIdx.x - split2, gridDim.x - split2);
}

// Compaction of rows with at most kDelThreadFix deletes, one thread per row.
// bid / nb: this workgroup's index among the nb workgroups that share the
// work (the whole grid, or its part in k_del_fix_both).
__device__ void del_fix_rows_body(const MutArgs &a, uint32_t bid, uint32_t nb) {
    const uint32_t cnt = ld_acquire(&a.ctl->small_cnt);
    uint64_t applied = 0, missing = 0;
    for (uint32_t t = bid * blockDim.x + threadIdx.x; t < cnt; t += nb * blockDim.x) {
        const uint32_t u = a.small_list[t];
        const uint32_t nd = uint32_t(a.cnt64[u]);
        const uint32_t k = a.hcnt[u];
        if (k) {
            const Row r = a.rows[u];
            uint32_t *row = a.pools.row(r.off);
            const uint32_t *hl = a.grouped + a.gofs[u];
            const uint32_t newdeg = r.deg - k;
            // k <= kDelThreadFix: the k tail slots and the k holes are loaded
            // together first (the stores below go to holes under newdeg, never
            // to the tail), so a host-tier row costs one host-link round trip
            uint32_t tv[kDelThreadFix], hv[kDelThreadFix];
#pragma unroll
            for (uint32_t j = 0; j < kDelThreadFix; ++j) {
                tv[j] = j < k ? row[newdeg + j] : kNone;
                hv[j] = j < k ? hl[j] : kNone;
            }
            // as many holes lie below newdeg as live slots lie at or above
            // it: the j-th live tail slot fills the j-th hole below newdeg
            uint32_t rt = 0;
#pragma unroll
            for (uint32_t j = 0; j < kDelThreadFix; ++j) {
                const bool live = tv[j] != kNone;
                uint32_t target = kNone, rh = 0;
#pragma unroll
                for (uint32_t i = 0; i < kDelThreadFix; ++i) {
                    const bool below = hv[i] < newdeg;
                    if (below && rh == rt) target = hv[i];
                    rh += below ? 1u : 0u;
                }
                if (live && target != kNone) row[target] = tv[j];
                rt += live ? 1u : 0u;
            }
            a.rows[u].deg = newdeg;
            a.hcnt[u] = 0;
        }
        if (u < a.n) {
            applied += k;
            missing += nd - k;
        }
    }
    StatShard *sh = stat_shard(a.stats);
    stat_add(&sh->deletes_applied, wave_sum64(applied));
    stat_add(&sh->missing, wave_sum64(missing));
}

// Exclusive scan of a 0/1 flag over a 256-thread workgroup; *total gets the
// sum. Contains barriers: every thread of the workgroup must call it.
__device__ __forceinline__ uint32_t block_flag_scan(bool f, uint32_t *wsum, uint32_t &total) {
    const uint64_t m = __ballot(f);
    const uint32_t w = wave_in_block();
    if (lane_id() == 0) wsum[w] = uint32_t(__popcll(m));
    __syncthreads();
    uint32_t before = 0;
    total = 0;
    for (uint32_t i = 0; i < blockDim.x / kWave; ++i) {
        if (i < w) before += wsum[i];
        total += wsum[i];
    }
    __syncthreads();
    return before + uint32_t(__popcll(m & __lanemask_lt()));
}

// Long rows, scan phase: one workgroup per kDelTile-slot tile. A slot whose
// destination is in the row's table claims one requested occurrence (first
// claims win). The tile's row loads are issued before the table is staged
// in LDS (tables of more than kDelLdsKeys slots are probed in place).
// An 8192-bit filter of the staged table's keys: a slot whose bit is clear
// matches no request and skips the probe (most slots of a long row match
// nothing, and a wave runs each probe loop as long as its longest chain).
constexpr uint32_t kDelBloomWords = 256;
__device__ __forceinline__ uint32_t del_bloom_bit(uint32_t x) { return (x * 0x85EBCA6Bu) >> 19; }

__device__ void del_scan_body(const MutArgs &a, uint32_t bid, uint32_t nb) {
    __shared__ uint32_t keys[kDelLdsKeys];
    // two filters, alternating by tile: a tile fills one while it clears the
    // other for the next tile, so staging needs no barrier of its own
    __shared__ uint32_t blooms[2][kDelBloomWords];
    const uint32_t nt = ld_acquire(&a.ctl->dtile_cnt);
    const uint32_t tid = threadIdx.x;
    for (uint32_t k = tid; k < kDelBloomWords; k += blockDim.x) blooms[0][k] = 0u;
    uint32_t it = 0;
    for (uint32_t t = bid; t < nt; t += nb, ++it) {
        uint32_t *bloom = blooms[it & 1u], *next = blooms[(it + 1u) & 1u];
        const DelTile dt = a.dtiles[t];
        const uint32_t bits = dt.bits, mask = (1u << bits) - 1u, to = dt.to, len = dt.len;
        uint32_t *row = a.pools.row(dt.off);     // the tile start is a multiple of 4
        const uint32_t nq = (len + 3u) >> 2;     // <= 4 * blockDim.x
        uint32_t d[4][4], live[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t q = k * blockDim.x + tid;
            live[k] = load_quad(row, q < nq ? q : nq - 1, len, d[k]);
            if (q >= nq) live[k] = 0;
        }
        const bool in_lds = mask < kDelLdsKeys;
        __syncthreads();  // the previous tile is done with `keys` and with `next`
        for (uint32_t k = tid; k < kDelBloomWords; k += blockDim.x) next[k] = 0u;
        if (in_lds) {
            for (uint32_t k = tid; k <= mask; k += blockDim.x) {
                const uint32_t key = a.hkeys[to + k];
                keys[k] = key;
                if (key != 0u) {
                    const uint32_t b = del_bloom_bit(key - 1u);
                    atomicOr(&bloom[b >> 5], 1u << (b & 31u));  // cleared by the previous tile
                }
            }
        }
        __syncthreads();
        const uint32_t *gkeys = a.hkeys + to;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
#pragma unroll
            for (uint32_t s = 0; s < 4; ++s) {
                if (s >= live[k]) continue;
                const uint32_t x = d[k][s];
                if (in_lds) {
                    const uint32_t b = del_bloom_bit(x);
                    if (((bloom[b >> 5] >> (b & 31u)) & 1u) == 0u) continue;
                }
                uint32_t h = ht_hash(x, bits), hit = kNone;
                if (in_lds) {
                    for (uint32_t probe = 0; probe <= mask; ++probe, h = (h + 1u) & mask) {
                        const uint32_t key = keys[h];
                        if (key == 0u) break;
                        if (key == x + 1u) {
                            hit = h;
                            break;
                        }
                    }
                } else {
                    for (uint32_t probe = 0; probe <= mask; ++probe, h = (h + 1u) & mask) {
                        const uint32_t key = gkeys[h];
                        if (key == 0u) break;
                        if (key == x + 1u) {
                            hit = h;
                            break;
                        }
                    }
                }
                if (hit != kNone && atomicAdd(&a.hcnts[to + hit].y, 1u) < a.hcnts[to + hit].x) {
                    const uint32_t slot = 4u * (k * blockDim.x + tid) + s;
                    row[slot] = kNone;
                    del_hole(a, dt.row, dt.start + slot);
                }
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_del_scan(MutArgs a) { del_scan_body(a, blockIdx.x, gridDim.x); }

// Every claim of a small batch in one launch, a quarter of the workgroups to
// each kind of row (disjoint rows, so the kinds need no order): tiny rows,
// host-tier medium rows, HBM medium rows, long rows. A small batch is bound
// by the latency of each pass, not by how many waves fit: one after the other
// the three passes of 1000 deletes took 47 us, together 21. The
// grid is a multiple of four workgroups (a remainder would take scan tiles
// twice; testing for it here costs the fourth wave a SIMD: 131 registers).
__global__ __launch_bounds__(kBlock) void k_del_claims(MutArgs a) {
    const uint32_t nb = gridDim.x / 4u, part = blockIdx.x / nb, bid = blockIdx.x - part * nb;
    switch (part) {
    case 0: del_lane_body(a, bid, nb); break;
    case 1: del_rows_body<2, true>(a, bid, nb); break;
    case 2: del_rows_body<4, false>(a, bid, nb); break;
    default: del_scan_body(a, bid, gridDim.x - 3u * nb); break;
    }
}

// Compaction of rows with more than kDelThreadFix deletes (or a table), one
// workgroup per row: with k holes the row shrinks to deg-k and the live
// slots of the last k positions move into the holes below deg-k (O(k)
// stores). The row's table and hole counter are cleared for the next call.
__device__ void del_fix_body(const MutArgs &a, uint32_t bid, uint32_t nb) {
    __shared__ uint32_t wsum[256 / kWave];
    const uint32_t cnt = ld_acquire(&a.ctl->big_cnt);
    const uint32_t tid = threadIdx.x;
    uint64_t applied = 0, missing = 0;
    for (uint32_t j = bid; j < cnt; j += nb) {
        const uint32_t u = a.big_list[j];
        const Row r = a.rows[u];
        const uint32_t nd = uint32_t(a.cnt64[u]);
        const uint32_t k = a.hcnt[u];
        uint32_t *hl = a.grouped + a.gofs[u];
        uint32_t *row = a.pools.row(r.off);
        const uint32_t newdeg = r.deg - k;
        // 1. compact the holes below newdeg to the front of the hole list
        //    (write index <= read index, and the scan's barrier orders them)
        uint32_t run = 0;
        for (uint32_t b = 0; b < k; b += blockDim.x) {
            const uint32_t i = b + tid;
            const uint32_t h = i < k ? hl[i] : 0u;
            const bool front = i < k && h < newdeg;
            uint32_t tot;
            const uint32_t rk = block_flag_scan(front, wsum, tot);
            if (front) hl[run + rk] = h;
            run += tot;
        }
        __syncthreads();
        // 2. live slots of [newdeg, deg) fill those holes in order
        run = 0;
        for (uint32_t b = 0; b < k; b += blockDim.x) {
            const uint32_t i = b + tid;
            const uint32_t v = i < k ? row[newdeg + i] : kNone;
            const bool live = v != kNone;
            uint32_t tot;
            const uint32_t rk = block_flag_scan(live, wsum, tot);
            if (live && run + rk < k) row[hl[run + rk]] = v;
            run += tot;
        }
        // 3. clear the table (long rows) for the next call
        const uint32_t to = a.htoff[u], tsz = to != kNone ? 1u << del_table_bits(nd) : 0u;
        for (uint32_t s = tid; s < tsz; s += blockDim.x) {
            a.hkeys[to + s] = 0u;
            a.hcnts[to + s] = make_uint2(0u, 0u);
        }
        if (tid == 0) {
            a.rows[u].deg = newdeg;
            a.hcnt[u] = 0u;
        }
        if (u < a.n) {
            applied += k;
            missing += nd - k;
        }
        __syncthreads();
    }
    if (wave_in_block() == 0) {
        StatShard *sh = stat_shard(a.stats);
        stat_add(&sh->deletes_applied, applied);
        stat_add(&sh->missing, missing);
    }
}

// Both hole fixes in one launch (they own disjoint rows): the first `split`
// workgroups take the rows fixed by one thread each, the others one row per
// workgroup, so the short per-thread pass and the per-workgroup pass overlap.
__global__ __launch_bounds__(256) void k_del_fix_both(MutArgs a, uint32_t split) {
    stamp_marks(a.ctl, a.ts);
    if (blockIdx.x < split) del_fix_rows_body(a, blockIdx.x, split);
    else del_fix_body(a, blockIdx.x - split, gridDim.x - split);
}

// Insert phase (PatchOrInvalidateCachedAdjacency's grow path,
// csr_graph.cuh:1793-1821, and RewriteSourceToNewBlock,
// source_local_chunk_store.h:782-848): each touched source appends its adds;
// a row that outgrows its block moves to a block of the next power of two at
// the tail of its tier. k_add_plan decides per row (one thread each),
// reserves pool blocks and copy pieces with one atomic per workgroup and
// tier, and rewrites the descriptors; k_add_copy then moves every piece with
// whole waves. A row that cannot be placed is listed in `overflow` and left
// for the host to retry after compaction.
struct AddPiece {
    const uint32_t *src;
    uint32_t *dst;
    uint32_t len;
    uint32_t flags;  // kFlRelease | class: src is a host-tier block to list once copied
};
constexpr uint32_t kFlRelease = 0x80000000u;
constexpr uint32_t kPieceLen = 1024;

__device__ __forceinline__ uint32_t pieces_of(uint64_t len) { return uint32_t((len + kPieceLen - 1) / kPieceLen); }

__global__ void k_add_plan(MutArgs a, const uint32_t *list, const uint32_t *list_count) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    __shared__ unsigned long long scratch64[kMaxWavesPerBlock + 1];
    const uint32_t cnt = ld_acquire(list_count);
    uint64_t acc_adds = 0, acc_reloc = 0, acc_garbage[2] = {0, 0};
    for (uint32_t base = blockIdx.x * blockDim.x; base < cnt; base += gthreads()) {
        const uint32_t j = base + threadIdx.x;
        const bool on = j < cnt;
        uint32_t u = 0, nd = 0, na = 0, tier = 0;
        Row r{};
        uint64_t newdeg = 0, newcap = 0;
        bool grow = false;
        if (on) {
            u = list[j];
            const uint64_t c = a.cnt64[u];
            nd = uint32_t(c);
            na = uint32_t(c >> 32);
            r = a.rows[u];
            newdeg = uint64_t(r.deg) + na;
            tier = (r.off & kHostTier) ? 1u : 0u;
            grow = newdeg > r.cap;
            if (grow) newcap = next_pow2_dev(newdeg);
        }
        // a growing host-tier row takes a freed block of its new class when one is listed
        uint64_t popped = 0;
        const bool reuse = grow && tier == 1 && newcap <= 0xFFFFFFFFull && fl_pop(a.fl, fl_class(newcap), popped);
        const uint64_t o0 = block_reserve<unsigned long long>(grow && tier == 0 ? newcap : 0ull,
                                                              (unsigned long long *)&a.ctl->pool_tail[0], scratch64);
        const uint64_t o1 = block_reserve<unsigned long long>(grow && tier == 1 && !reuse ? newcap : 0ull,
                                                              (unsigned long long *)&a.ctl->pool_tail[1], scratch64);
        const uint64_t o = tier ? (reuse ? popped : o1) : o0;
        const bool over = grow && !reuse && (o + newcap > a.ctl->pool_cap[tier] || newcap > 0xFFFFFFFFull);
        block_append(over, u, a.overflow, &a.ctl->overflow_cnt, scratch);
        const bool go = on && !over && na != 0;
        const uint64_t noff = grow ? (o | (tier ? kHostTier : 0ull)) : r.off;
        const uint32_t np = go ? (grow ? pieces_of(r.deg) : 0u) + pieces_of(na) : 0u;
        const uint32_t pb = block_reserve<uint32_t>(np, &a.ctl->copy_cnt, scratch);
        if (go) {
            const uint32_t *old_row = a.pools.row(r.off);
            uint32_t *row = a.pools.row(noff);
            uint32_t k = pb;
            // the first piece of a relocated host-tier row carries the old
            // block's class: k_fl_release lists the block once it is copied
            if (grow)
                for (uint32_t p = 0; p < r.deg; p += kPieceLen)
                    a.pieces[k++] = AddPiece{old_row + p, row + p, min(kPieceLen, r.deg - p),
                                             p == 0 && tier == 1 ? kFlRelease | fl_class(r.cap) : 0u};
            const uint32_t *al = a.grouped + a.gofs[u] + nd;
            for (uint32_t p = 0; p < na; p += kPieceLen)
                a.pieces[k++] = AddPiece{al + p, row + r.deg + p, min(kPieceLen, na - p), 0u};
            if (grow) {
                Row nr;
                nr.off = noff;
                nr.deg = uint32_t(newdeg);
                nr.cap = uint32_t(newcap);
                a.rows[u] = nr;
                acc_garbage[tier] += r.cap;
                if (u < a.n) acc_reloc += 1;
            } else {
                a.rows[u].deg = uint32_t(newdeg);
            }
            if (u < a.n) acc_adds += na;
        }
    }
    StatShard *sh = stat_shard(a.stats);
    stat_add(&sh->adds_applied, wave_sum64(acc_adds));
    stat_add(&sh->relocated, wave_sum64(acc_reloc));
    stat_add(&sh->garbage[0], wave_sum64(acc_garbage[0]));
    stat_add(&sh->garbage[1], wave_sum64(acc_garbage[1]));
}

// Moves the pieces of the insert phase: a wave takes 64 pieces, scans their
// lengths and copies the concatenation 256 slots per step, so short pieces
// (a few adds) and long ones (a relocated row) keep every lane busy.
__global__ __launch_bounds__(kBlock) void k_add_copy(MutArgs a) {
    __shared__ uint32_t pref_lds[kWavesPerBlock][kWave];
    uint32_t *pref = pref_lds[wave_in_block()];
    const uint32_t cnt = ld_acquire(&a.ctl->copy_cnt);
    const uint32_t lane = lane_id();
    for (uint64_t base = uint64_t(gwave()) * kWave; base < cnt; base += uint64_t(gwaves()) * kWave) {
        const uint32_t i = uint32_t(base) + lane;
        AddPiece pc{nullptr, nullptr, 0u, 0u};
        if (i < cnt) pc = a.pieces[i];
        const uint32_t incl = wave_incl_scan(pc.len);
        const uint32_t total = __shfl(incl, kWave - 1, kWave);
        pref[lane] = incl - pc.len;
        wave_lds_sync();
        const unsigned long long src = (unsigned long long)pc.src, dst = (unsigned long long)pc.dst;
        for (uint32_t k0 = 0; k0 < total; k0 += kWave * 4) {
            uint32_t val[4], *dp[4];
            bool ok[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t k = k0 + uint32_t(e) * kWave + lane;
                ok[e] = k < total;
                const uint32_t kk = ok[e] ? k : total - 1;
                const uint32_t own = owner_of(pref, kk);
                const uint32_t off = kk - pref[own];
                const uint32_t *sp = reinterpret_cast<const uint32_t *>(__shfl(src, int(own), kWave));
                dp[e] = reinterpret_cast<uint32_t *>(__shfl(dst, int(own), kWave)) + off;
                val[e] = sp[off];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ok[e]) *dp[e] = val[e];
        }
        wave_lds_sync();
    }
}

// Lists the old blocks of the host-tier rows this insert phase relocated
// (their slots were copied by k_add_copy, which ran before).
__global__ void k_fl_release(MutArgs a) {
    const uint32_t cnt = ld_acquire(&a.ctl->copy_cnt);
    for (uint32_t i = gthread(); i < cnt; i += gthreads()) {
        const AddPiece pc = a.pieces[i];
        if (pc.flags & kFlRelease) fl_push(a.fl, pc.flags & 63u, uint64_t(pc.src - a.pools.host));
    }
}

// ------------------------------------------------------- grouped batches
// Several consecutive batches applied as one: every delete is matched to
// the latest earlier unmatched add of the same (u,v) in the group (adds of
// batch b come after its deletes); matched pairs cancel, since the delete
// removes an instance the add created. The records left then give the
// sequential result when all deletes are applied before all adds, so the
// group needs one mutation and one fixed point. Only (u,v) keys that occur
// both as add and as delete in the group are examined one by one.
struct GroupArgs {
    const cig_edge *dels;
    uint32_t nd;
    const cig_edge *adds;
    uint32_t na;
    const uint32_t *del_cut;  // nb+1 prefix of the deletes per batch
    const uint32_t *add_cut;  // nb+1 prefix of the adds per batch
    uint32_t nb;
    uint32_t n;
    unsigned long long *tkey;  // (u<<32 | v) + 1; 0 = empty
    uint32_t *thead;           // op list head (kNone = empty)
    uint8_t *tconf;            // key seen as add and as delete
    uint32_t tbits;
    uint32_t *next_op;         // ops: adds [0,na), deletes [na,na+nd)
    uint8_t *skip;             // 1 = cancelled op
    uint32_t *overflow;        // set when a key holds more than kGroupOps ops
    StatShard *stats;
};
constexpr uint32_t kGroupOps = 32;

__device__ __forceinline__ uint32_t key_hash(unsigned long long k, uint32_t bits) {
    return uint32_t((k * 0x9E3779B97F4A7C15ull) >> (64 - bits));
}

__global__ void k_group_adds(GroupArgs g) {
    const uint32_t mask = (1u << g.tbits) - 1u;
    for (uint32_t j = gthread(); j < g.na; j += gthreads()) {
        const cig_edge e = g.adds[j];
        if (e.u >= g.n || e.v >= g.n) continue;
        const unsigned long long key = ((unsigned long long)e.u << 32 | e.v) + 1ull;
        uint32_t h = key_hash(key, g.tbits);
        for (;;) {  // the table has >= 2 * na slots: the probe ends
            const unsigned long long prev = atomicCAS(&g.tkey[h], 0ull, key);
            if (prev == 0ull || prev == key) break;
            h = (h + 1u) & mask;
        }
        g.next_op[j] = atomicExch(&g.thead[h], j);
    }
}

__global__ void k_group_dels(GroupArgs g) {
    const uint32_t mask = (1u << g.tbits) - 1u;
    for (uint32_t i = gthread(); i < g.nd; i += gthreads()) {
        const cig_edge e = g.dels[i];
        if (e.u >= g.n || e.v >= g.n) continue;
        const unsigned long long key = ((unsigned long long)e.u << 32 | e.v) + 1ull;
        for (uint32_t h = key_hash(key, g.tbits), probe = 0; probe <= mask; ++probe, h = (h + 1u) & mask) {
            const unsigned long long k = g.tkey[h];
            if (k == 0ull) break;
            if (k == key) {
                g.tconf[h] = 1;
                g.next_op[g.na + i] = atomicExch(&g.thead[h], g.na + i);
                break;
            }
        }
    }
}

// Batch of entry `i` given the nb+1 prefix `cut` (largest b with cut[b] <= i).
__device__ __forceinline__ uint32_t batch_of(const uint32_t *cut, uint32_t nb, uint32_t i) {
    uint32_t lo = 0, hi = nb;  // cut[lo] <= i < cut[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (cut[mid] <= i) lo = mid;
        else hi = mid;
    }
    return lo;
}

// One thread per key seen as both add and delete: order its ops by time
// (delete of batch b at 2b, add at 2b+1) and cancel matched pairs.
__global__ void k_group_match(GroupArgs g) {
    const uint32_t cap = 1u << g.tbits;
    uint64_t cancel_d = 0, cancel_a = 0;
    for (uint32_t h = gthread(); h < cap; h += gthreads()) {
        if (!g.tconf[h]) continue;
        uint32_t op[kGroupOps], tm[kGroupOps], cnt = 0;
        bool over = false;
        for (uint32_t o = g.thead[h]; o != kNone; o = g.next_op[o]) {
            if (cnt == kGroupOps) {
                over = true;
                break;
            }
            const bool del = o >= g.na;
            tm[cnt] = del ? 2u * batch_of(g.del_cut, g.nb, o - g.na) : 2u * batch_of(g.add_cut, g.nb, o) + 1u;
            op[cnt++] = o;
        }
        if (over) {
            atomicExch(g.overflow, 1u);
            continue;
        }
        for (uint32_t x = 1; x < cnt; ++x)  // insertion sort by time
            for (uint32_t y = x; y > 0 && tm[y - 1] > tm[y]; --y) {
                const uint32_t t0 = tm[y]; tm[y] = tm[y - 1]; tm[y - 1] = t0;
                const uint32_t o0 = op[y]; op[y] = op[y - 1]; op[y - 1] = o0;
            }
        uint32_t stack[kGroupOps], top = 0;
        for (uint32_t x = 0; x < cnt; ++x) {
            if (op[x] < g.na) {
                stack[top++] = op[x];
            } else if (top) {
                g.skip[op[x]] = 1;
                g.skip[stack[--top]] = 1;
                ++cancel_d;
                ++cancel_a;
            }
        }
    }
    // a cancelled pair applied both records (the delete found the instance)
    StatShard *sh = stat_shard(g.stats);
    stat_add(&sh->deletes_applied, wave_sum64(cancel_d));
    stat_add(&sh->adds_applied, wave_sum64(cancel_a));
}

// End of a call: clears the per-row counters of the touched rows and, when
// `aff` is given, the affected bitmap words of the affected list. With
// activity counting on, every touched row (outgoing or incoming) adds its
// records of the call to its window count: a delete scans the row, so rows
// mutated often are worth keeping in HBM like rows expanded often.
__global__ void k_clear_touched(MutArgs a, uint32_t *aff, const uint32_t *alist) {
    const uint32_t touched = ld_acquire(&a.ctl->touched);
    for (uint32_t t = gthread(); t < touched; t += gthreads()) {
        const uint32_t u = a.touched[t];
        if (a.hot) {
            const uint64_t c = a.cnt64[u];
            a.hot[u] += uint32_t(min(uint64_t(255), (c & 0xFFFFFFFFull) + (c >> 32)));
        }
        a.cnt64[u] = 0;
    }
    if (aff) {
        const uint32_t cnt = ld_acquire(&a.ctl->acount);
        for (uint32_t i = gthread(); i < cnt; i += gthreads()) aff[alist[i] >> 5] = 0u;
    }
}

// The descriptor and the delete/add counts of each row listed in `list`
// (the rows whose adds found no room), for the host's compaction sizing.
struct RowCount {
    Row row;
    uint64_t cnt;
};
__global__ void k_gather_rows(const Row *rows, const uint64_t *cnt64, const uint32_t *list, uint32_t cnt,
                              RowCount *out) {
    for (uint32_t i = gthread(); i < cnt; i += gthreads()) {
        const uint32_t u = list[i];
        out[i] = RowCount{rows[u], cnt64[u]};
    }
}

// The affected-bit part of k_clear_touched alone.
__global__ void k_clear_aff(const Ctl *c, uint32_t *aff, const uint32_t *alist) {
    const uint32_t cnt = ld_acquire(&c->acount);
    for (uint32_t i = gthread(); i < cnt; i += gthreads()) aff[alist[i] >> 5] = 0u;
}

// ---------------------------------------------------- deletion invalidation
struct InvalArgs {
    Ctl *ctl;
    const Row *rows;
    const Row *in_rows;  // incoming rows: rows + n, or rows itself for a symmetric graph
    uint64_t *state;
    uint32_t *stamp;
    uint32_t *aff;
    uint32_t *alist;
    uint32_t *filt;  // global copy of the repair filter (kFilterWords words)
    uint32_t *q0, *q1;
    Tile *t0, *t1;
    ExpandCfg cfg;
    const cig_edge *dels;
    uint32_t nd;
    const cig_edge *adds;
    uint32_t na;
    uint32_t n;
    uint32_t kind;  // 0 = single source (SSSP/BFS), 1 = vertex seeds (CC)
    uint32_t max_rounds;
    uint64_t seed;
    const uint8_t *add_skip, *del_skip;  // grouped batches: cancelled records (may be null)
    const BatchRef *ref;                 // non-null: the records are read from here (graph replays)
    uint32_t ts;                         // stage markers the kernel notes
};

// reset_del_edges (driver.cuh:371-411): a deleted (u,v) whose v has parent u
// seeds the affected set. Parallel copies of (u,v) are treated conservatively.
__global__ void k_inval_seed(InvalArgs a) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    stamp_marks(a.ctl, a.ts);
    const uint32_t nd = rec_nd(a);
    const cig_edge *dels = rec_dels(a);
    for (uint32_t base = blockIdx.x * blockDim.x; base < nd; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        bool hit = false;
        uint32_t v = 0;
        if (i < nd) {
            const cig_edge e = dels[i];
            if (e.u < a.n && e.v < a.n && !(a.del_skip && a.del_skip[i]) && uint32_t(a.state[e.v]) == e.u) {
                v = e.v;
                hit = bit_claim(a.aff, v);
            }
        }
        block_append(hit, v, a.alist, &a.ctl->acount, scratch);
    }
}

// Invalidation waves (RunSyncPushDDB_del rounds, framework.cuh:2815-2853) as
// one persistent launch: the affected list grows in place; round k expands
// the items appended by round k-1.
template <int QPL>
__global__ __launch_bounds__(kBlock) void k_inval_loop(InvalArgs a) {
    __shared__ WaveLds lds[kWavesPerBlock];
    WaveLds &L = lds[wave_in_block()];
    Ctl *c = a.ctl;
    InvalidateOp op{a.rows, a.state, a.aff};
    Counters ctr;
    uint32_t b = 0;
    for (uint32_t k = 0; k < a.max_rounds; ++k) {
        const uint32_t e = ld_acquire(&c->acount);
        const uint32_t nt = ld_acquire(&c->icount[k % 3]);
        if (b == e && nt == 0) break;
        if (blockIdx.x == 0 && threadIdx.x == 0) c->icount[(k + 2) % 3] = 0;
        const DirectOut out{Sink{a.alist, &c->acount}, TileSink{(k & 1) ? a.t0 : a.t1, &c->icount[(k + 1) % 3]}};
        expand_range<QPL>(op, a.cfg, a.alist + b, e - b, out, L, ctr);
        expand_tiles<QPL>(op, a.cfg, (k & 1) ? a.t1 : a.t0, nt, out);
        b = e;
        cg::this_grid().sync();
    }
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
}

// One invalidation wave as an ordinary launch, the seq-th of its chain:
// round k expands its frontier alist[istart, istart+ifront) (the first round:
// the seeds, alist[0, acount)) and its deferred tiles, and appends the next
// frontier right behind it. Slots
// rotate mod 3: workgroup 0 opens slot k+1's start, clears slot k+2 and
// posts the round's progress word at the start, so no workgroup waits for
// another and the round needs no closing step.
template <int QPL>
__global__ __launch_bounds__(kBlock) void k_inval_round(InvalArgs a, uint64_t *prog, uint64_t tag, uint32_t seq) {
    __shared__ WaveLds lds[kWavesPerBlock];
    __shared__ RoundStage stage;
    Ctl *c = a.ctl;
    const uint32_t k = c->iround + seq - 1;
    // the first round's frontier is the seeds: alist[0, acount)
    const uint32_t start = seq == 1 ? 0u : c->istart[k % 3];
    const uint32_t cnt = seq == 1 ? c->acount : c->ifront[k % 3];
    const uint32_t nt = c->icount[k % 3];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->istart[(k + 1) % 3] = start + cnt;
        c->ifront[(k + 2) % 3] = 0;
        c->icount[(k + 2) % 3] = 0;
        c->acount = start + cnt;  // affected so far; final once a round finds nothing
        post_progress(prog, tag, cnt != 0 || nt != 0);
    }
    if (cnt == 0 && nt == 0) return;
    InvalidateOp op{a.rows, a.state, a.aff};
    Counters ctr;
    const StagedOut<2048, 128> out{Sink{a.alist + start + cnt, &c->ifront[(k + 1) % 3]},
                                   TileSink{(k & 1) ? a.t0 : a.t1, &c->icount[(k + 1) % 3]}, &stage};
    out_init(out);
    expand_range<QPL>(op, a.cfg, a.alist + start, cnt, out, lds[wave_in_block()], ctr);
    expand_tiles<QPL>(op, a.cfg, (k & 1) ? a.t1 : a.t0, nt, out);
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    out_flush(out);
}

// reset_affected_values (driver.cuh:418-433): affected vertices restart from
// the initial value (CC: own label), and all of them form the next frontier.
__device__ void reset_affected_body(const InvalArgs &a, uint32_t bid, uint32_t nb) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    const uint32_t cnt = ld_acquire(&a.ctl->acount);
    const uint32_t r = a.ctl->round;
    uint32_t *q = (r & 1) ? a.q1 : a.q0;
    for (uint32_t base = bid * blockDim.x; base < cnt; base += nb * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        bool push = false;
        uint32_t v = 0;
        if (i < cnt) {
            v = a.alist[i];
            a.state[v] = a.kind == 1 ? ((uint64_t(v) << 32) | kNone) : ~0ull;
            push = claim(a.stamp, v, r);
        }
        block_append(push, v, q, &a.ctl->qcount[r % 3], scratch);
    }
}

__global__ void k_reset_affected(InvalArgs a) { reset_affected_body(a, blockIdx.x, gridDim.x); }

// The reset beside the hole fixes of the same batch: the one writes vertex
// state and the frontier, the other rows, so where no wave runs between them
// they share a launch (first `split` workgroups: the reset; then, as in
// k_del_fix_both, up to `split2` the rows fixed by one thread each).
__global__ __launch_bounds__(256) void k_reset_and_fix(InvalArgs a, MutArgs m, uint32_t split, uint32_t split2) {
    stamp_marks(a.ctl, m.ts);
    if (blockIdx.x < split) reset_affected_body(a, blockIdx.x, split);
    else if (blockIdx.x < split2) del_fix_rows_body(m, blockIdx.x - split, split2 - split);
    else del_fix_body(m, blockIdx.x - split2, gridDim.x - split2);
}

// SeedAddedEdgeFrontier (framework.cuh:238-294): each inserted (u,v) offers
// value(u)+w to v; improved destinations join the pending frontier.
template <int W, bool kStrict>
__global__ void k_insert_seed(InvalArgs a, uint32_t skip_affected) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    stamp_marks(a.ctl, a.ts);
    const uint32_t r = a.ctl->round;
    uint32_t *q = (r & 1) ? a.q1 : a.q0;
    const uint32_t na = rec_na(a);
    const cig_edge *adds = rec_adds(a);
    for (uint32_t base = blockIdx.x * blockDim.x; base < na; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        bool push = false;
        uint32_t v = 0;
        if (i < na) {
            const cig_edge e = adds[i];
            if (e.u < a.n && e.v < a.n && !(a.add_skip && a.add_skip[i]) &&
                !(skip_affected && bit_test(a.aff, e.u))) {
                const uint32_t val = uint32_t(a.state[e.u] >> 32);
                if (val != kInf) {
                    const uint64_t cand = uint64_t(val) + weight<W>(e.u, e.v, a.seed);
                    if (cand < kInf && relax<kStrict>(a.state, e.v, uint32_t(cand), e.u)) {
                        v = e.v;
                        push = claim(a.stamp, v, r);
                    }
                }
            }
        }
        block_append(push, v, q, &a.ctl->qcount[r % 3], scratch);
    }
}

// -------------------------------------------------------------- repair scan
// The affected list is folded once into a bitmap filter of 2^18 bits (a
// multiplicative hash of the id) in global memory; every repair workgroup
// copies it into LDS. An edge whose destination misses the filter is not
// affected, so almost every edge of the scan is settled in LDS and only
// filter hits read the global affected bitmap. The filter is off when the
// affected list is too long to stay selective.
constexpr uint32_t kFilterBits = 18;
constexpr uint32_t kFilterWords = (1u << kFilterBits) / 32;
constexpr uint32_t kFilterMaxItems = 1u << 16;
constexpr uint32_t kRepairBlock = 512;

__device__ __forceinline__ uint32_t filter_hash(uint32_t v) { return (v * 0x9E3779B1u) >> (32 - kFilterBits); }

struct AffFilter {
    const uint32_t *lds;  // nullptr: filter off
    const uint32_t *aff;
    __device__ __forceinline__ bool test(uint32_t v) const {
        if (lds) {
            const uint32_t h = filter_hash(v);
            if (!((lds[h >> 5] >> (h & 31)) & 1u)) return false;
        }
        return bit_test(aff, v);
    }
};

// a.filt must be zero on entry (k_fill32 before this launch).
__global__ void k_build_filter(InvalArgs a) {
    const uint32_t na = ld_acquire(&a.ctl->acount);
    if (na > kFilterMaxItems) return;
    for (uint32_t i = gthread(); i < na; i += gthreads()) {
        const uint32_t h = filter_hash(a.alist[i]);
        atomicOr(&a.filt[h >> 5], 1u << (h & 31));
    }
}

__device__ __forceinline__ bool load_filter(uint32_t *lds, const uint32_t *g, uint32_t na) {
    if (na > kFilterMaxItems) return false;
    const uint4 *src = reinterpret_cast<const uint4 *>(g);
    uint4 *dst = reinterpret_cast<uint4 *>(lds);
    for (uint32_t w = threadIdx.x; w < kFilterWords / 4; w += blockDim.x) dst[w] = src[w];
    __syncthreads();
    return true;
}

template <int W, bool kStrict>
struct RepairScanOp {
    const Row *rows;
    uint64_t *state;
    AffFilter filt;
    uint64_t seed;
    __device__ bool source(uint32_t v, uint32_t, Row &row, uint32_t &pay) const {
        if (filt.test(v)) return false;
        const uint32_t val = uint32_t(state[v] >> 32);
        if (val == kInf) return false;
        row = rows[v];
        pay = val;
        return row.deg != 0;
    }
    __device__ bool tile_source(const Tile &t, uint32_t &pay) const {
        pay = uint32_t(state[t.v] >> 32);
        return pay != kInf;
    }
    // the LDS filter answers most edges without a global access
    __device__ uint64_t peek(uint32_t y) const {
        if (!filt.lds) return 1;
        const uint32_t h = filter_hash(y);
        return (filt.lds[h >> 5] >> (h & 31)) & 1u;
    }
    __device__ bool edge(uint32_t u, uint32_t val, uint32_t y, uint64_t maybe) const {
        if (!maybe || !bit_test(filt.aff, y)) return false;
        const uint64_t c = uint64_t(val) + weight<W>(u, y, seed);
        if (c < kInf) relax<kStrict>(state, y, uint32_t(c), u);
        return false;
    }
};

template <int W, bool kStrict, int QPL>
__global__ __launch_bounds__(kRepairBlock) void k_repair_scan(InvalArgs a) {
    __shared__ __align__(16) uint32_t filt[kFilterWords];
    __shared__ WaveLds lds[kRepairBlock / kWave];
    __shared__ StageLds<2, 160> stage;
    Ctl *c = a.ctl;
    const uint32_t na = ld_acquire(&c->acount);
    if (na == 0) return;
    const bool on = load_filter(filt, a.filt, na);
    RepairScanOp<W, kStrict> op{a.rows, a.state, AffFilter{on ? filt : nullptr, a.aff}, a.seed};
    Counters ctr;
    const StagedOut<2, 160> out{Sink{nullptr, &c->scount}, TileSink{a.t0, &c->scount}, &stage};
    out_init(out);
    expand_range<QPL>(op, a.cfg, nullptr, a.n, out, lds[wave_in_block()], ctr);
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    out_flush(out);
}

template <int W, bool kStrict, int QPL>
__global__ __launch_bounds__(kRepairBlock) void k_repair_tiles(InvalArgs a) {
    __shared__ __align__(16) uint32_t filt[kFilterWords];
    Ctl *c = a.ctl;
    const uint32_t na = ld_acquire(&c->acount);
    const uint32_t nt = ld_acquire(&c->scount);
    if (na == 0 || nt == 0) return;
    const bool on = load_filter(filt, a.filt, na);
    RepairScanOp<W, kStrict> op{a.rows, a.state, AffFilter{on ? filt : nullptr, a.aff}, a.seed};
    expand_tiles<QPL>(op, a.cfg, a.t0, nt, DirectOut{Sink{nullptr, &c->scount}, TileSink{nullptr, &c->scount}});
}

// -------------------------------------------------------------- pull repair
// With the incoming index on, the repair reads only the incoming rows of the
// affected vertices (GpuAffectedPullRelax, framework.cuh:137-204, over a
// device-resident reverse index instead of the CPU-materialised one of
// dynamic_reverse_index.h:223-274): y takes the minimum over its unaffected,
// reached in-neighbours x of value(x) + w(x, y), ties to the smaller x. This
// is the same candidate set the full scan offers y, so the state after the
// repair is identical.
template <int W, bool kStrict>
struct PullOp {
    const Row *in_rows;  // incoming rows
    uint64_t *state;
    const uint32_t *aff;
    uint64_t seed;
    __device__ bool source(uint32_t y, uint32_t, Row &row, uint32_t &pay) const {
        row = in_rows[y];
        pay = y;
        return row.deg != 0;
    }
    __device__ bool tile_source(const Tile &t, uint32_t &pay) const {
        pay = t.v;
        return true;
    }
    __device__ uint64_t peek(uint32_t x) const { return state[x]; }
    __device__ bool edge(uint32_t y, uint32_t, uint32_t x, uint64_t sx) const {
        const uint32_t vx = uint32_t(sx >> 32);
        if (vx == kInf || bit_test(aff, x)) return false;
        const uint64_t c = uint64_t(vx) + weight<W>(x, y, seed);
        if (c < kInf) relax<kStrict>(state, y, uint32_t(c), x);
        return false;
    }
};

template <int W, bool kStrict, int QPL>
__global__ __launch_bounds__(kBlock) void k_repair_pull(InvalArgs a) {
    __shared__ WaveLds lds[kWavesPerBlock];
    __shared__ StageLds<2, 128> stage;
    Ctl *c = a.ctl;
    stamp_marks(c, a.ts);
    const uint32_t na = ld_acquire(&c->acount);
    if (na == 0) return;
    PullOp<W, kStrict> op{a.in_rows, a.state, a.aff, a.seed};
    Counters ctr;
    const StagedOut<2, 128> out{Sink{nullptr, &c->scount}, TileSink{a.t0, &c->scount}, &stage};
    out_init(out);
    expand_range<QPL>(op, a.cfg, a.alist, na, out, lds[wave_in_block()], ctr);
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    out_flush(out);
}

template <int W, bool kStrict, int QPL>
__global__ __launch_bounds__(kBlock) void k_repair_pull_tiles(InvalArgs a) {
    Ctl *c = a.ctl;
    stamp_marks(c, a.ts);
    const uint32_t nt = ld_acquire(&c->scount);
    if (nt == 0) return;
    PullOp<W, kStrict> op{a.in_rows, a.state, a.aff, a.seed};
    expand_tiles<QPL>(op, a.cfg, a.t0, nt, DirectOut{Sink{nullptr, &c->scount}, TileSink{nullptr, &c->scount}});
}

// ------------------------------------------------- one-shot expansion passes
template <int QPL, class Op>
__global__ __launch_bounds__(kBlock) void k_expand_once(Op op, ExpandCfg cfg, const uint32_t *items,
                                                         const uint32_t *count_ptr, uint32_t count,
                                                         Sink sink, TileSink ts, const uint32_t *gate) {
    __shared__ WaveLds lds[kWavesPerBlock];
    __shared__ RoundStage stage;
    if (gate && ld_acquire(gate) == 0) return;
    Counters ctr;
    const uint32_t n = count_ptr ? ld_acquire(count_ptr) : count;
    const StagedOut<2048, 128> out{sink, ts, &stage};
    out_init(out);
    expand_range<QPL>(op, cfg, items, n, out, lds[wave_in_block()], ctr);
    flush_counters(ctr, cfg.stats, cfg.stage);
    out_flush(out);
}

template <int QPL, class Op>
__global__ __launch_bounds__(kBlock) void k_expand_tiles(Op op, ExpandCfg cfg, const Tile *tiles,
                                                          const uint32_t *ntiles, Sink sink) {
    __shared__ RoundStage stage;
    const StagedOut<2048, 128> out{sink, TileSink{nullptr, sink.count}, &stage};
    out_init(out);
    expand_tiles<QPL>(op, cfg, tiles, ld_acquire(ntiles), out);
    out_flush(out);
}

// ------------------------------------------------------ traversal fixed point
struct LoopArgs {
    Ctl *ctl;
    const Row *rows;
    uint64_t *state;
    uint32_t *stamp;
    uint32_t *hot;
    uint32_t *q0, *q1;
    Tile *t0, *t1;
    ExpandCfg cfg;
    uint64_t seed;
    uint32_t max_rounds;
    uint32_t delta;  // delta-ordered rounds (0: unordered)
    uint32_t ts;     // stage markers the chain's first round notes
};

// One persistent cooperative launch runs rounds until the frontier and the
// deferred tiles are empty (RunExactGpuClosure's grid.sync loop,
// framework.cuh:342-454, without host round trips). Round r consumes
// queue[r&1] / count slot r%3 and produces into the other queue and slot
// (r+1)%3; slot (r+2)%3 is cleared for round r+1. Tiles of long rows found in
// round r are expanded in round r+1 (re-reading the row owner's value).
template <int W, bool kStrict, int QPL>
__global__ __launch_bounds__(kBlock) void k_relax_loop(LoopArgs a) {
    __shared__ WaveLds lds[kWavesPerBlock];
    WaveLds &L = lds[wave_in_block()];
    Ctl *c = a.ctl;
    uint32_t r = ld_acquire(&c->round);
    Counters ctr;
    uint32_t it = 0;
    for (; it < a.max_rounds; ++it, ++r) {
        const uint32_t nq = ld_acquire(&c->qcount[r % 3]);
        const uint32_t nt = ld_acquire(&c->tcount[r % 3]);
        if (nq == 0 && nt == 0) break;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            c->qcount[(r + 2) % 3] = 0;
            c->tcount[(r + 2) % 3] = 0;
        }
        RelaxOp<W, kStrict> op{a.rows, a.state, a.stamp, a.hot, a.seed, r + 1};
        const uint32_t *qin = (r & 1) ? a.q1 : a.q0;
        const DirectOut out{Sink{(r & 1) ? a.q0 : a.q1, &c->qcount[(r + 1) % 3]},
                            TileSink{(r & 1) ? a.t0 : a.t1, &c->tcount[(r + 1) % 3]}};
        expand_range<QPL>(op, a.cfg, qin, nq, out, L, ctr);
        expand_tiles<QPL>(op, a.cfg, (r & 1) ? a.t1 : a.t0, nt, out);
        cg::this_grid().sync();
    }
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->round = r;
        c->rounds += it;
    }
}

// One relax round as an ordinary launch (the default driver), the seq-th of
// its chain: round r = round + seq - 1 consumes queue[r&1] / slot r%3 and
// appends to the other queue / slot (r+1)%3. Workgroup 0 clears slot
// (r+2)%3 and posts the round's progress word at the start; the host keeps
// a few rounds enqueued ahead and advances `round` after the chain, so no
// workgroup waits for another and a round has no closing step. A round
// whose frontier and deferred tiles are empty returns at once.
template <int W, bool kStrict, int QPL, int B = kBlock, bool ORD = false>
__global__ __launch_bounds__(B) void k_relax_round(LoopArgs a, uint64_t *prog, uint64_t tag, uint32_t seq) {
    __shared__ WaveLds lds[B / kWave];
    __shared__ RoundStage stage;
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3], nt = c->tcount[r % 3];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->qcount[(r + 2) % 3] = 0;
        c->tcount[(r + 2) % 3] = 0;
        if constexpr (ORD) c->bmin[(r + 1) % 3] = kInf;  // for the next round's k_ord_min
        if (seq == 1) stamp_marks(c, a.ts);
        if (nq || nt) c->rounds += 1;
        post_progress(prog, tag, nq != 0 || nt != 0);
    }
    if (nq == 0 && nt == 0) return;
    Counters ctr;
    RelaxOp<W, kStrict> op{a.rows, a.state, a.stamp, a.hot, a.seed, r + 1};
    const uint32_t *qin = (r & 1) ? a.q1 : a.q0;
    const StagedOut<2048, 128> out{Sink{(r & 1) ? a.q0 : a.q1, &c->qcount[(r + 1) % 3]},
                                   TileSink{(r & 1) ? a.t0 : a.t1, &c->tcount[(r + 1) % 3]}, &stage};
    out_init(out);
    if constexpr (ORD) {
        // Items above the round's smallest bucket wait for a later round
        // (PartitionActive, ordered_gpu_repair.cuh:33-48): re-listed here,
        // skipped by the expansion below. Tiles always expand: their rows
        // were cut in the previous round.
        op.delta = a.delta;
        op.bucket = c->bmin[r % 3];
        const uint32_t wpb = blockDim.x / kWave, gw = blockIdx.x * wpb + wave_in_block();
        for (uint32_t base = gw * kWave; base < nq; base += gridDim.x * wpb * kWave) {
            const uint32_t i = base + lane_id();
            bool f[1] = {false};
            uint32_t v[1] = {0};
            if (i < nq) {
                v[0] = qin[i];
                const uint32_t val = uint32_t(a.state[v[0]] >> 32);
                f[0] = val != kInf && val / a.delta > op.bucket && claim(a.stamp, v[0], r + 1);
            }
            out_push<1>(out, f, v);
        }
    }
    expand_range<QPL>(op, a.cfg, qin, nq, out, lds[wave_in_block()], ctr);
    expand_tiles<QPL>(op, a.cfg, (r & 1) ? a.t1 : a.t0, nt, out);
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    out_flush(out);
}

// Delta-ordered rounds (FindActiveBucket, ordered_gpu_repair.cuh:28-32):
// the smallest value / delta of round r's frontier, one atomic per wave.
// Values only fall, so a later read in the round can only find the bucket's
// items at or below it: the round always expands at least one row.
__global__ void k_ord_min(LoopArgs a, uint32_t seq) {
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    const uint32_t *qin = (r & 1) ? a.q1 : a.q0;
    uint32_t m = kInf;
    for (uint32_t i = gthread(); i < nq; i += gthreads()) {
        const uint32_t val = uint32_t(a.state[qin[i]] >> 32);
        if (val != kInf) m = min(m, val / a.delta);
    }
    for (int off = kWave / 2; off > 0; off >>= 1) m = min(m, uint32_t(__shfl_xor(int(m), off, kWave)));
    if (lane_id() == 0 && m != kInf) atomicMin(&c->bmin[r % 3], m);
}

__global__ void k_ord_reset(Ctl *c) {
    if (threadIdx.x < 3 && blockIdx.x == 0) c->bmin[threadIdx.x] = kInf;
}

// Moves the round counter past a finished chain of `by` rounds.
__global__ void k_advance_round(Ctl *c, uint32_t by) {
    if (threadIdx.x == 0 && blockIdx.x == 0) c->round += by;
}

// A query runs its rounds through the engine's queues, so a frontier pending
// there (of an engine that is initialised and not solved yet, or stopped by a
// round cap) is set aside first and listed again afterwards. It needs no copy:
// the frontier is the vertices whose mark is set, and a query touches no mark.
enum : uint32_t { kMarkStamp = 0, kMarkQueued = 1, kMarkAct = 2 };  // stamp = the round; PR's flag; msi.hpp's act

// The owners of pending tiles join the frontier: their whole rows are expanded
// again, which changes no fixed point, and the tiles need not be kept.
__global__ void k_park_tiles(Ctl *c, uint32_t *stamp, const Tile *t0, const Tile *t1) {
    const uint32_t r = c->round, nt = c->tcount[r % 3];
    const Tile *tiles = (r & 1) ? t1 : t0;
    for (uint32_t i = gthread(); i < nt; i += gthreads()) stamp[tiles[i].v] = r;
}

// No frontier in any slot; park != 0 notes the round of the one set aside.
__global__ void k_clear_frontier(Ctl *c, uint32_t park) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (park) c->parked = c->round;
    for (int i = 0; i < 3; ++i) c->qcount[i] = c->tcount[i] = c->fscan[i] = c->flist[i] = 0;
}

// Lists the frontier set aside as the current round's.
__global__ void k_list_frontier(Ctl *c, uint32_t kind, uint32_t *stamp, const unsigned long long *act, uint32_t *q0,
                                uint32_t *q1, uint32_t n) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    const uint32_t r = c->round, from = c->parked;
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gthreads()) {
        const uint32_t v = base + threadIdx.x;
        bool on = v < n;
        if (kind == kMarkAct) on = on && act[v] != 0ull;
        else if (kind == kMarkQueued) on = on && stamp[v] != 0u;
        else on = on && stamp[v] == from;
        if (on && kind == kMarkStamp) stamp[v] = r;
        block_append(on, v, (r & 1) ? q1 : q0, &c->qcount[r % 3], scratch);
    }
}

// ---------------------------------------------------------- PageRank rounds
// Pull plan of one solve. Incoming rows of up to kPullSplit slots are listed
// by size class: class c holds the rows of up to 4 << c slots, which 1 << c
// lanes read with one 16-B load each. Longer rows are cut into tiles of
// kPullTile slots; a row of several tiles also gets a PullRow, whose last tile
// to finish adds the tiles' partial sums up.
constexpr uint32_t kPullClasses = 7;
constexpr uint32_t kPullSplit = 4u << (kPullClasses - 1);
constexpr uint32_t kPullTile = 2048;

struct PullEntry {
    uint64_t off;
    uint32_t v, deg;
};

struct PullRow {
    uint32_t first, nt, done, pad;
};

// The plan's lists: the classes, then tiles and rows of several tiles.
constexpr uint32_t kPlanLists = kPullClasses + 2, kPlanTiles = kPullClasses, kPlanMulti = kPullClasses + 1;
constexpr uint32_t kPlanBlocks = 512;  // workgroups of the two plan kernels

struct PrArgs {
    Ctl *ctl;
    const Row *rows;
    float *rank, *comp, *res, *delta;
    uint32_t *queued;
    uint32_t *q0, *q1;
    Tile *t0, *t1;
    ExpandCfg cfg;
    float eps;
    uint32_t max_rounds;
    // pull form (incoming rows present): rounds whose frontier holds at
    // least pull_min vertices gather; pull_min = kNone disables it
    const Row *in_rows;
    uint32_t n, pull_min;
    PullEntry *pent;  // the classes' rows, class by class
    Tile *ptiles;
    PullRow *prow;
    uint32_t *pcnt;   // plan kernels: per workgroup, the length of each list
    unsigned long long *tpart;  // a word a tile (put_partial); 0 between passes
    // bit v set iff delta[v] != 0; pull passes of rounds with fewer than
    // mask_max frontier vertices (and amendments) test it before gathering
    unsigned long long *amask;
    uint32_t mask_max;
    // out-degrees of the current rows (k_pr_degrees, once per solve): the
    // dense consume reads 4 B per vertex here instead of its 16-B row
    uint32_t *odeg;
};

// Out-degree of every vertex for the dense consume passes of one solve.
__global__ void k_pr_degrees(const Row *rows, uint32_t n, uint32_t *odeg) {
    for (uint32_t v = gthread(); v < n; v += gthreads()) odeg[v] = rows[v].deg;
}

__device__ __forceinline__ bool pr_dense(const PrArgs &a, uint32_t nq) { return nq != 0 && nq >= a.pull_min; }

// Runtime::Converge (pr_residual.cuh:171-187) as one persistent launch:
// consume (rank += r with Kahan compensation, r = 0, contribution
// alpha*r/deg), grid barrier, scatter, grid barrier.
template <int QPL>
__global__ __launch_bounds__(kBlock) void k_pr_loop(PrArgs a) {
    __shared__ WaveLds lds[kWavesPerBlock];
    WaveLds &L = lds[wave_in_block()];
    Ctl *c = a.ctl;
    uint32_t r = ld_acquire(&c->round);
    Counters ctr;
    uint32_t it = 0;
    for (; it < a.max_rounds; ++it, ++r) {
        const uint32_t nq = ld_acquire(&c->qcount[r % 3]);
        if (nq == 0) break;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            c->qcount[(r + 2) % 3] = 0;
            c->tcount[(r + 2) % 3] = 0;
        }
        const uint32_t *qin = (r & 1) ? a.q1 : a.q0;
        Tile *tiles = (r & 1) ? a.t1 : a.t0;
        for (uint32_t i = gthread(); i < nq; i += gthreads()) {
            const uint32_t v = qin[i];
            const float rv = a.res[v];
            a.queued[v] = 0u;
            float d = 0.0f;
            if (!isfinite(rv) || !isfinite(a.rank[v])) atomicExch(&c->pr_invalid, 1u);
            if (fabsf(rv) > a.eps) {
                a.res[v] = 0.0f;
                const float x = a.rank[v];
                const float y = rv - a.comp[v];
                const float t = x + y;
                a.comp[v] = (t - x) - y;
                a.rank[v] = t;
                const Row row = a.rows[v];
                ctr.vexp += 1;
                if (row.deg) {
                    d = 0.85f * rv / float(row.deg);
                    if (row.deg >= a.cfg.split) {
                        const uint32_t nt = (row.deg + a.cfg.tile_len - 1) / a.cfg.tile_len;
                        const uint32_t t0 = atomicAdd(&c->tcount[r % 3], nt);
                        for (uint32_t j = 0; j < nt; ++j) {
                            Tile t;
                            t.start = row.off + uint64_t(j) * a.cfg.tile_len;
                            t.v = v;
                            t.len = min(a.cfg.tile_len, row.deg - j * a.cfg.tile_len);
                            t.payload = __float_as_uint(d);
                            t.pad = 0;
                            tiles[t0 + j] = t;
                        }
                        ctr.scanned += row.deg;
                        if (row.off & kHostTier) ctr.host += row.deg;
                        d = 0.0f;
                    }
                }
            }
            a.delta[i] = d;
        }
        cg::this_grid().sync();
        PrScatterOp op{a.rows, a.res, a.queued, a.delta, &c->pr_invalid, a.eps};
        // tiles of long rows were made while consuming; the scatter makes none
        const DirectOut out{Sink{(r & 1) ? a.q0 : a.q1, &c->qcount[(r + 1) % 3]}, TileSink{tiles, &c->scount}};
        Counters sctr;
        expand_range<QPL>(op, a.cfg, qin, nq, out, L, sctr);
        ctr.scanned += sctr.scanned;
        ctr.host += sctr.host;
        expand_tiles<QPL>(op, a.cfg, tiles, ld_acquire(&c->tcount[r % 3]), out);
        cg::this_grid().sync();
    }
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->round = r;
        c->rounds += it;
        c->converged = ld_acquire(&c->qcount[r % 3]) == 0 ? 1u : 0u;
    }
}

// PageRank round, consume phase (pr_residual.cuh:54-71) as an ordinary
// launch; long rows are cut into tiles for this round's scatter (one tile
// reservation per workgroup step).
__global__ __launch_bounds__(kBlock) void k_pr_consume(PrArgs a, uint64_t *prog, uint64_t tag, uint32_t seq) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->qcount[(r + 2) % 3] = 0;
        c->tcount[(r + 2) % 3] = 0;
        c->fscan[(r + 2) % 3] = 0;
        c->flist[(r + 2) % 3] = 0;
        if (nq) c->rounds += 1;
        post_progress(prog, tag, nq != 0);
    }
    if (nq == 0) return;
    Counters ctr;
    if (pr_dense(a, nq)) {
        // pull form: the queued flags are the frontier; every vertex gets its
        // contribution (0 when not consumed) in delta[v]
        if (blockIdx.x == 0 && threadIdx.x == 0) c->pull_rounds += 1;
        // a wave takes 64 consecutive vertices (one mask word) per step
        for (uint32_t base = gthread() - lane_id(); base < a.n; base += gthreads()) {
            const uint32_t v = base + lane_id();
            float d = 0.0f;
            if (v < a.n && a.queued[v]) {
                a.queued[v] = 0u;
                const float rv = a.res[v];
                if (!isfinite(rv) || !isfinite(a.rank[v])) atomicExch(&c->pr_invalid, 1u);
                if (fabsf(rv) > a.eps) {
                    a.res[v] = 0.0f;
                    const float x = a.rank[v];
                    const float y = rv - a.comp[v];
                    const float t = x + y;
                    a.comp[v] = (t - x) - y;
                    a.rank[v] = t;
                    const uint32_t deg = a.odeg[v];
                    ctr.vexp += 1;
                    if (deg) d = 0.85f * rv / float(deg);
                }
            }
            const unsigned long long bits = __ballot(d != 0.0f);
            if (v < a.n) a.delta[v] = d;
            if (lane_id() == 0) a.amask[base >> 6] = bits;
        }
        flush_counters(ctr, a.cfg.stats, a.cfg.stage);
        return;
    }
    uint32_t *qin = (r & 1) ? a.q1 : a.q0;
    Tile *tiles = (r & 1) ? a.t1 : a.t0;
    // a frontier that a pull pass left as flags: this scan writes the list
    const bool scan = c->fscan[r % 3] != 0;
    const uint32_t bound = scan ? a.n : nq;
    for (uint32_t base = blockIdx.x * blockDim.x; base < bound; base += gthreads()) {
        uint32_t i = base + threadIdx.x;
        uint32_t v = 0, nt = 0;
        Row row{};
        float d = 0.0f;
        bool on = i < bound;
        if (scan) {
            v = i;
            on = on && a.queued[v] != 0u;
            i = block_reserve<uint32_t>(on ? 1u : 0u, &c->flist[r % 3], scratch);
            if (on) qin[i] = v;
        } else if (on) {
            v = qin[i];
        }
        if (on) {
            const float rv = a.res[v];
            a.queued[v] = 0u;
            if (!isfinite(rv) || !isfinite(a.rank[v])) atomicExch(&c->pr_invalid, 1u);
            if (fabsf(rv) > a.eps) {
                a.res[v] = 0.0f;
                const float x = a.rank[v];
                const float y = rv - a.comp[v];
                const float t = x + y;
                a.comp[v] = (t - x) - y;
                a.rank[v] = t;
                row = a.rows[v];
                ctr.vexp += 1;
                if (row.deg) {
                    d = 0.85f * rv / float(row.deg);
                    if (row.deg >= a.cfg.split) nt = (row.deg + a.cfg.tile_len - 1) / a.cfg.tile_len;
                }
            }
        }
        const uint32_t t0 = block_reserve<uint32_t>(nt, &c->tcount[r % 3], scratch);
        for (uint32_t j = 0; j < nt; ++j) {
            Tile t;
            t.start = row.off + uint64_t(j) * a.cfg.tile_len;
            t.v = v;
            t.len = min(a.cfg.tile_len, row.deg - j * a.cfg.tile_len);
            t.payload = __float_as_uint(d);
            t.pad = 0;
            tiles[t0 + j] = t;
        }
        if (nt) {
            ctr.scanned += row.deg;
            if (row.off & kHostTier) ctr.host += row.deg;
            d = 0.0f;
        }
        if (on) a.delta[i] = d;
    }
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
}

// PageRank round, scatter phase (pr_residual.cuh:74-100) of round
// round + seq - 1; the consume phase of the same round posted its progress.
template <int QPL>
__device__ void pr_scatter_round(const PrArgs &a, uint32_t seq, WaveLds &lds, RoundStage &stage) {
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    if (nq == 0) return;
    const uint32_t nt = c->tcount[r % 3];
    const uint32_t *qin = (r & 1) ? a.q1 : a.q0;
    Tile *tiles = (r & 1) ? a.t1 : a.t0;
    PrScatterOp op{a.rows, a.res, a.queued, a.delta, &c->pr_invalid, a.eps};
    // tiles of long rows were made while consuming; the scatter makes none
    const StagedOut<2048, 128> out{Sink{(r & 1) ? a.q0 : a.q1, &c->qcount[(r + 1) % 3]},
                                   TileSink{tiles, &c->scount}, &stage};
    out_init(out);
    Counters ctr;
    expand_range<QPL>(op, a.cfg, qin, nq, out, lds, ctr);
    expand_tiles<QPL>(op, a.cfg, tiles, nt, out);
    flush_counters(ctr, a.cfg.stats, a.cfg.stage);
    out_flush(out);
}

template <int QPL>
__global__ __launch_bounds__(kBlock) void k_pr_scatter(PrArgs a, uint32_t seq) {
    __shared__ WaveLds lds[kWavesPerBlock];
    __shared__ RoundStage stage;
    pr_scatter_round<QPL>(a, seq, lds[wave_in_block()], stage);
}

// ------------------------------------------------ PageRank rounds, pull form
// The scatter of a round adds alpha*r(u)/deg(u) to r(w) for every edge (u,w)
// of a consumed u. When the frontier is dense the same sums are gathered
// along the incoming rows (rows n..2n-1, sources of each vertex's in-edges):
// w adds sum over its in-neighbours u of delta[u], which the consume phase
// wrote for every vertex (0 where nothing was consumed). Each r(w) then has
// a single writer, so the residual updates are plain loads and stores, not
// the scatter's per-edge atomics, and a vertex joins the next frontier when
// its residual crosses epsilon, as in the scatter. Only the summation order
// differs from the scatter's (whose atomic order is itself unspecified).

// The pull plan of the current incoming rows (they do not change during a
// solve), in two launches over the same vertex ranges: k_pr_plan_count counts
// what each workgroup adds to each list, k_pr_plan_fill adds the counts of the
// workgroups before it up and writes the lists, so neither needs an atomic on
// a shared cursor (one per 256 rows and list held the pass to 200 us at 2^22
// vertices; now 23 and 105). `gate` (when given) must be non-zero to run.
__device__ __forceinline__ uint32_t plan_range(uint32_t n, uint32_t &end) {
    const uint32_t per = (uint32_t((uint64_t(n) + kPlanBlocks - 1) / kPlanBlocks) + 255u) & ~255u;
    const uint64_t lo = uint64_t(blockIdx.x) * per;
    end = uint32_t(min(uint64_t(n), lo + per));
    return uint32_t(min(uint64_t(n), lo));
}

// The list of a row of deg >= 1 slots; tiles: how many it is cut into.
__device__ __forceinline__ uint32_t plan_list(uint32_t deg, uint32_t &tiles) {
    tiles = 0;
    if (deg > kPullSplit) {
        tiles = (deg + kPullTile - 1) / kPullTile;
        return kPlanTiles;
    }
    return deg <= 4 ? 0u : 30u - uint32_t(__clz(deg - 1));
}

__device__ __forceinline__ void plan_tally(const Row &row, uint32_t *cnt) {
    if (row.deg == 0) return;
    uint32_t tiles;
    const uint32_t l = plan_list(row.deg, tiles);
    atomicAdd(&cnt[l], l == kPlanTiles ? tiles : 1u);
    if (tiles > 1) atomicAdd(&cnt[kPlanMulti], 1u);
}

__global__ __launch_bounds__(kBlock) void k_pr_plan_count(PrArgs a, const uint32_t *gate) {
    __shared__ uint32_t cnt[kPlanLists];
    if (gate && *gate == 0) return;
    if (threadIdx.x < kPlanLists) cnt[threadIdx.x] = 0u;
    __syncthreads();
    uint32_t end;
    for (uint32_t v = plan_range(a.n, end) + threadIdx.x; v < end; v += kBlock) plan_tally(a.in_rows[v], cnt);
    __syncthreads();
    if (threadIdx.x < kPlanLists) a.pcnt[blockIdx.x * kPlanLists + threadIdx.x] = cnt[threadIdx.x];
}

__global__ __launch_bounds__(kBlock) void k_pr_plan_fill(PrArgs a, const uint32_t *gate) {
    __shared__ uint32_t cur[kPlanLists], tot[kPlanLists];
    if (gate && *gate == 0) return;
    const uint32_t lane = lane_id();
    for (uint32_t l = wave_in_block(); l < kPlanLists; l += kWavesPerBlock) {
        uint64_t all = 0, before = 0;
        for (uint32_t w = lane; w < kPlanBlocks; w += kWave) {
            const uint32_t x = a.pcnt[w * kPlanLists + l];
            all += x;
            before += w < blockIdx.x ? x : 0u;
        }
        all = wave_sum64(all);
        before = wave_sum64(before);
        if (lane == 0) {
            cur[l] = uint32_t(before);
            tot[l] = uint32_t(all);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (uint32_t l = 0; l < kPullClasses; ++l) {  // the classes share one array
            cur[l] += run;
            run += tot[l];
        }
        if (blockIdx.x == 0)
            for (uint32_t l = 0; l < kPlanLists; ++l) a.ctl->plan[l] = tot[l];
    }
    __syncthreads();
    uint32_t end;
    for (uint32_t v = plan_range(a.n, end) + threadIdx.x; v < end; v += kBlock) {
        const Row row = a.in_rows[v];
        if (row.deg == 0) continue;
        uint32_t nt;
        const uint32_t l = plan_list(row.deg, nt);
        if (l != kPlanTiles) {
            a.pent[atomicAdd(&cur[l], 1u)] = PullEntry{row.off, v, row.deg};
            continue;
        }
        const uint32_t at = atomicAdd(&cur[kPlanTiles], nt);
        uint32_t mi = kNone;
        if (nt > 1) {
            mi = atomicAdd(&cur[kPlanMulti], 1u);
            a.prow[mi] = PullRow{at, nt, 0u, 0u};
        }
        for (uint32_t j = 0; j < nt; ++j) {
            Tile t;
            t.start = row.off + uint64_t(j) * kPullTile;
            t.v = v;
            t.len = min(kPullTile, row.deg - j * kPullTile);
            t.payload = mi;
            t.pad = 0;
            a.ptiles[at + j] = t;
        }
    }
}

__device__ __forceinline__ float wave_sum_f(float x) {
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) x += __shfl_xor(x, d, kWave);
    return x;
}

// Where a pull pass finds the contributions: the first kPullHubs of them (the
// hubs of a renumbered engine) in LDS, the others in memory, behind the
// mask's bit when there is one (the mask is 1/32 of delta's size, so a sparse
// pass touches far fewer cache lines).
constexpr uint32_t kPullHubs = 32768;
constexpr uint32_t kPullHubBlock = 1024;
constexpr uint32_t kPullSets = 2;
// an LDS address as such: through a generic pointer the two reads of a slot
// merge into one flat load, which waits for both memories
using LdsFloat = __attribute__((address_space(3))) const float;
template <bool HUB>
struct PullSrc {
    const float *delta;
    const unsigned long long *mask;
    LdsFloat *hub;
};

// Sum of delta[] over the live slots of QPL quads whose loads are in flight
// together; dead slots (past the row's end or past the last quad) add 0. A
// slot that needs no memory read (a hub, a cleared mask bit) reads word 0, a
// line its wave shares, so the vector memory unit walks the others only.
template <int QPL, bool HUB>
__device__ __forceinline__ void pull_gather(const PullSrc<HUB> &p, const uint32_t (&d)[QPL][4],
                                            const uint32_t (&live)[QPL], float (&s)[QPL]) {
    float x[QPL][4];
    bool need[QPL][4];
#pragma unroll
    for (int q = 0; q < QPL; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) need[q][k] = !HUB || d[q][k] >= kPullHubs;
    if (p.mask) {
        uint32_t w[QPL][4];
        const uint32_t *m32 = reinterpret_cast<const uint32_t *>(p.mask);
#pragma unroll
        for (int q = 0; q < QPL; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k) w[q][k] = m32[need[q][k] ? d[q][k] >> 5 : 0u];
#pragma unroll
        for (int q = 0; q < QPL; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const bool on = (w[q][k] >> (d[q][k] & 31u)) & 1u;
                const float g = p.delta[need[q][k] && on ? d[q][k] : 0u];
                x[q][k] = on ? g : 0.0f;
            }
    } else {
#pragma unroll
        for (int q = 0; q < QPL; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k) x[q][k] = p.delta[need[q][k] ? d[q][k] : 0u];
    }
    if constexpr (HUB) {
#pragma unroll
        for (int q = 0; q < QPL; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float h = p.hub[need[q][k] ? 0u : d[q][k]];
                x[q][k] = need[q][k] ? x[q][k] : h;
            }
    }
#pragma unroll
    for (int q = 0; q < QPL; ++q) {
        s[q] = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) s[q] += uint32_t(k) < live[q] ? x[q][k] : 0.0f;
    }
}

// Adds `sum` to r(w), whose value before the pass is `old` (this lane is w's
// only writer), and reports whether w joins the next frontier.
__device__ __forceinline__ bool pull_add(const PrArgs &a, uint32_t w, float old, float sum) {
    if (sum == 0.0f) return false;
    const float now = old + sum;
    a.res[w] = now;
    if (!isfinite(now)) atomicExch(&a.ctl->pr_invalid, 1u);
    if (fabsf(old) <= a.eps && fabsf(now) > a.eps && a.queued[w] == 0u) {
        a.queued[w] = 1u;
        return true;
    }
    return false;
}

// A unit of the class lists: kPullSets sets of 64 >> c rows of class c, 1 << c
// lanes a row, one quad a lane. No search for a slot's row and no shared
// accumulator: a row's lanes add up by shuffles.
struct PullAt {
    uint32_t c, first, end;  // class, first row, end of the class's list (wave-uniform)
    bool on;
};
struct PullRows {
    PullEntry e[kPullSets];
    bool on[kPullSets];  // false: past the list's end (e repeats its last row)
};
struct PullQuads {
    uint32_t d[kPullSets][4], live[kPullSets];
    float old[kPullSets];
};

// Unit u of the lists whose lengths are cnt[].
__device__ __forceinline__ PullAt pull_at(const uint32_t (&cnt)[kPullClasses], uint32_t u) {
    PullAt p{0u, 0u, 0u, false};
    uint32_t base = 0;
#pragma unroll
    for (uint32_t c = 0; c < kPullClasses; ++c) {
        const uint32_t rows = kPullSets * (kWave >> c), units = (cnt[c] + rows - 1) / rows;
        if (!p.on && u < units) p = PullAt{c, base + u * rows, base + cnt[c], true};
        u -= p.on ? 0u : units;
        base += cnt[c];
    }
    return p;
}

__device__ __forceinline__ void pull_load_rows(const PrArgs &a, const PullAt &p, PullRows &r) {
#pragma unroll
    for (uint32_t s = 0; s < kPullSets; ++s) {
        const uint32_t i = p.first + s * (kWave >> p.c) + (lane_id() >> p.c);
        r.on[s] = p.on && i < p.end;
        r.e[s] = PullEntry{0ull, 0u, 0u};
        if (p.on) r.e[s] = a.pent[min(i, p.end - 1)];
    }
}

__device__ __forceinline__ void pull_load_quads(const PrArgs &a, const PullAt &p, const PullRows &r, PullQuads &q) {
    const uint32_t j = lane_id() & ((1u << p.c) - 1u);
#pragma unroll
    for (uint32_t s = 0; s < kPullSets; ++s) {
        const uint32_t deg = r.e[s].deg;
        const bool in = 4u * j < deg;
        q.live[s] = 0;
        q.old[s] = 0.0f;
        if (p.on) {
            // wave-uniform; lanes past the row's end read its first quad, whose
            // slots past deg (never written, any word) are aliased to its first
            const uint32_t live = load_quad_stream(a.cfg.pools.row(r.e[s].off), in ? j : 0u, deg, q.d[s]);
            q.live[s] = r.on[s] && in ? live : 0u;
            q.old[s] = a.res[r.e[s].v];
        }
    }
}

template <bool HUB>
__device__ __forceinline__ void pull_finish(const PrArgs &a, const PullSrc<HUB> &src, const PullAt &p, const PullRows &r,
                                            const PullQuads &q, uint32_t &joined, Counters &ctr) {
    float sum[kPullSets];
    pull_gather<kPullSets>(src, q.d, q.live, sum);
    const uint32_t j = lane_id() & ((1u << p.c) - 1u);
    for (uint32_t dd = (1u << p.c) >> 1; dd > 0; dd >>= 1)
#pragma unroll
        for (uint32_t s = 0; s < kPullSets; ++s) sum[s] += __shfl_xor(sum[s], int(dd), kWave);
#pragma unroll
    for (uint32_t s = 0; s < kPullSets; ++s) {
        const PullEntry &e = r.e[s];
        if (j == 0 && r.on[s]) {
            ctr.scanned += e.deg;
            ctr.vexp += 1;
            if (e.off & kHostTier) ctr.host += e.deg;
            joined += pull_add(a, e.v, q.old[s], sum[s]) ? 1u : 0u;
        }
    }
}

// A tile's partial sum travels in one 64-bit word with a flag above it, so the
// wave that adds the row up needs no order between the words and the row's
// counter (a release at the counter writes the L2 back for every tile: solve
// of 1,000,003 vertices 7.6 -> 10.7 ms, two batches of 62,500 + 62,500 over
// 2^22 29.7 -> 57.0). A word is 0 when its tile has not arrived and again once
// taken; a wave that takes one early waits for a store already issued.
__device__ __forceinline__ void put_partial(unsigned long long *p, float x) {
    __hip_atomic_store(p, (1ull << 32) | __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float take_partial(unsigned long long *p) {
    unsigned long long w;
    do w = ld_acquire(p);
    while ((w >> 32) == 0ull);
    __hip_atomic_store(p, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __uint_as_float(uint32_t(w));
}

// One tile of a long incoming row: all its loads in flight, then the gathers;
// a wave sum. A one-tile row is finished here; a longer row's tiles leave their
// partial sums behind, and the last one to count itself adds them up.
template <bool HUB>
__device__ void pull_tile(const PrArgs &a, const PullSrc<HUB> &src, const Tile &t, uint32_t ti, uint32_t &joined,
                          Counters &ctr) {
    constexpr int Q = kPullTile / (4 * kWave), P = 2;
    const uint32_t *p = a.cfg.pools.row(t.start);
    const uint32_t lane = lane_id();
    const uint32_t nq = (t.len + 3u) >> 2;
    uint32_t d[Q][4], live[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const uint32_t k = uint32_t(q) * kWave + lane;
        live[q] = 0;
        if (uint32_t(q) * kWave < nq) {  // wave-uniform
            live[q] = load_quad_stream(p, k < nq ? k : nq - 1, t.len, d[q]);
            if (k >= nq) live[q] = 0;
        }
    }
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < Q; q += P) {
        if (uint32_t(q) * kWave >= nq) break;
        uint32_t dd[P][4], ll[P];
        float s[P];
#pragma unroll
        for (int i = 0; i < P; ++i) {
            ll[i] = live[q + i];
#pragma unroll
            for (int k = 0; k < 4; ++k) dd[i][k] = uint32_t(q + i) * kWave < nq ? d[q + i][k] : 0u;
        }
        pull_gather<P>(src, dd, ll, s);
#pragma unroll
        for (int i = 0; i < P; ++i) acc += s[i];
    }
    acc = wave_sum_f(acc);
    if (lane == 0) {
        ctr.scanned += t.len;
        if (t.start & kHostTier) ctr.host += t.len;
    }
    if (t.payload != kNone) {
        PullRow &pr = a.prow[t.payload];
        uint32_t last = 0;
        if (lane == 0) {
            put_partial(&a.tpart[ti], acc);
            last = atomicAdd(&pr.done, 1u) + 1u == pr.nt ? 1u : 0u;
        }
        if (!__shfl(last, 0, kWave)) return;
        acc = 0.0f;
        for (uint32_t j = lane; j < pr.nt; j += kWave) acc += take_partial(&a.tpart[pr.first + j]);
        acc = wave_sum_f(acc);
        if (lane == 0) atomicExch(&pr.done, 0u);  // for the next pass
    }
    if (lane == 0) {
        ctr.vexp += 1;
        joined += pull_add(a, t.v, a.res[t.v], acc) ? 1u : 0u;
    }
}

// Where a pull pass appends and whether it runs. seq >= 1: the scatter phase
// of round round + seq - 1 when that round is dense, appending to the next
// round's frontier. seq = 0: a batch amendment (gated by amend_pull), whose
// contributions are the touched sources' +-alpha*x/deg, appending to the
// pending frontier of round `round`.
struct PullPass {
    bool run;
    uint32_t stage;
    uint32_t slot;  // of the frontier the vertices join
    const unsigned long long *mask;
};

__device__ __forceinline__ PullPass pull_pass(const PrArgs &a, uint32_t seq) {
    Ctl *c = a.ctl;
    if (seq == 0) {
        const uint32_t r = c->round;
        return PullPass{c->amend_pull != 0, kStageAmend, r % 3, a.amask};
    }
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    return PullPass{pr_dense(a, nq), kStageRepair, (r + 1) % 3, nq < a.mask_max ? a.amask : nullptr};
}

// The vertices that joined the frontier in a pull pass have their queued flag
// set; the frontier's count takes one atomic per workgroup, and its list is
// not written (flist = 0): a dense consume scans the flags anyway, a sparse
// one that finds no list scans them too. (A list cost up to an atomic per
// chunk on one address.) Every thread of the workgroup must call it.
__device__ __forceinline__ void frontier_count(Ctl *c, uint32_t slot, uint32_t joined, uint32_t *cnt) {
    if (threadIdx.x == 0) *cnt = 0u;
    __syncthreads();
    const uint32_t s = uint32_t(wave_sum64(joined));
    if (s && lane_id() == 0) atomicAdd(cnt, s);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (*cnt) atomicAdd(&c->qcount[slot], *cnt);
        if (blockIdx.x == 0) c->fscan[slot] = 1u;
    }
}

// What a round does with its contributions, or the amendment's sweep (seq 0;
// see pull_pass): gather along the incoming rows when the pass is dense, else
// scatter along the frontier's rows (a sparse round). One launch holds both
// forms: which one a round takes is known on the device only, and a launch
// that finds nothing to do costs the round 5 us and a gap.
//
// HUB (engines that number vertices by out-degree): one 1024-thread workgroup
// per CU holds the first 32768 contributions in LDS (R-MAT scale 20: the
// sources of 70% of the edges, scale 22: of 53%), since a gather from memory
// moves a 128-B line into L1 for 4 bytes. What bounds it: the lines of the
// other gathers (scale 22: 31 M, 3.9 GB into L1 per sweep) and the stream of
// source ids. Per dense sweep, scale 20 / 22: 110 / 285 us with 64 workgroups
// per CU that wrote the frontier's list, searched every slot's row and added
// quads up in LDS; now 56 / 265. Two sets of rows in flight per wave: one 62 /
// 280, four 76 / 335 (their lines displace each other in L1). Without HUB: 81
// / 360; it is held to the 128 registers of four waves a SIMD (132 and three
// waves: a solve of 2^20 vertices 12.6 -> 13.2 ms).
template <bool HUB>
__global__ __launch_bounds__(HUB ? kPullHubBlock : kBlock, 4) void k_pr_pull(PrArgs a, uint32_t seq) {
    constexpr uint32_t B = HUB ? kPullHubBlock : kBlock;
    struct ScatterLds {
        WaveLds w[B / kWave];
        RoundStage stage;
    };
    union Lds {
        float hub[HUB ? kPullHubs : 1];
        ScatterLds scatter;
        __device__ Lds() {}
    };
    __shared__ Lds lds;
    __shared__ uint32_t total;
    Ctl *c = a.ctl;
    const PullPass pass = pull_pass(a, seq);
    if (!pass.run) {
        if (seq) pr_scatter_round<1>(a, seq, lds.scatter.w[wave_in_block()], lds.scatter.stage);
        return;
    }
    // Neighbouring units go to different workgroups (the heavy ones are
    // neighbours). A wave's units are pipelined: a unit's row entries are read
    // two units ahead, its quads one ahead; the first loads go out before the
    // hubs are staged.
    const uint32_t gw = wave_in_block() * gridDim.x + blockIdx.x, nwaves = gridDim.x * (B / kWave);
    uint32_t cnt[kPullClasses];
#pragma unroll
    for (uint32_t l = 0; l < kPullClasses; ++l) cnt[l] = c->plan[l];
    const uint32_t nt = c->plan[kPlanTiles];
    PullAt p0 = pull_at(cnt, gw), p1 = pull_at(cnt, gw + nwaves);
    PullRows r0, r1;
    PullQuads q0;
    pull_load_rows(a, p0, r0);
    pull_load_rows(a, p1, r1);
    pull_load_quads(a, p0, r0, q0);
    if constexpr (HUB) {
        const uint32_t h = min(a.n, kPullHubs);
#pragma unroll 8
        for (uint32_t i = threadIdx.x; i < h; i += B) lds.hub[i] = a.delta[i];
        __syncthreads();
    }
    const PullSrc<HUB> src{a.delta, pass.mask, (LdsFloat *)lds.hub};
    Counters ctr;
    uint32_t joined = 0;
    for (uint32_t u = gw + 2 * nwaves; p0.on; u += nwaves) {
        const PullAt p2 = pull_at(cnt, u);
        PullRows r2;
        PullQuads q1;
        pull_load_quads(a, p1, r1, q1);
        pull_load_rows(a, p2, r2);
        pull_finish(a, src, p0, r0, q0, joined, ctr);
        p0 = p1;
        p1 = p2;
        r0 = r1;
        r1 = r2;
        q0 = q1;
    }
    if (gw < nt) {
        Tile next = a.ptiles[gw];
        for (uint32_t ti = gw; ti < nt; ti += nwaves) {
            const Tile t = next;
            if (ti + nwaves < nt) next = a.ptiles[ti + nwaves];
            pull_tile(a, src, t, ti, joined, ctr);
        }
    }
    flush_counters(ctr, a.cfg.stats, pass.stage);
    frontier_count(c, pass.slot, joined, &total);
}

// Batch amendment form (Engine::UpdatePageRank, framework.cuh:1660-1704):
// r += alpha (P_new^T - P_old^T) x over the touched sources, either scattered
// along their old and new rows (few touched rows) or gathered by two sweeps
// of the incoming rows, before and after the mutation (many touched rows: a
// hub-heavy batch touches most edges, and the scatter's atomics would cost
// several sweeps). `touched` counts outgoing and incoming rows.
__global__ void k_pr_amend_form(Ctl *c, uint32_t min_touched) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const uint32_t pull = c->touched >= min_touched ? 1u : 0u;
    c->amend_pull = pull;
    c->amend_push = 1u - pull;
}

// Pull amendment contributions: delta[u] = sign*alpha*x[u]/deg(u) along u's
// current row for every touched source u, with its mask bit (delta and the
// mask are zero elsewhere).
__global__ void k_pr_amend_delta(PrArgs a, const uint32_t *touched, float sign) {
    Ctl *c = a.ctl;
    if (!c->amend_pull) return;
    const uint32_t cnt = c->touched;
    for (uint32_t i = gthread(); i < cnt; i += gthreads()) {
        const uint32_t u = touched[i];
        if (u >= a.n) continue;  // an incoming row
        const uint32_t deg = a.rows[u].deg;
        const float x = a.rank[u];
        const float d = deg && x != 0.0f ? sign * 0.85f * x / float(deg) : 0.0f;
        a.delta[u] = d;
        if (d != 0.0f) atomicOr(&a.amask[u >> 6], 1ull << (u & 63u));
    }
}

// --------------------------------------------------- multi-source queries
// Up to 64 BFS / SSSP sources at once on the live graph: dist holds 64
// distances per vertex (vertex-major, `stride` words per vertex), act the
// sources whose distance at the vertex improved since it was last expanded.
// A round first takes each frontier vertex's mask (k_ms_consume: snap :=
// act, act := 0) and cuts its long rows into tiles, then expands rows and
// tiles (k_ms_expand): for every edge (u,w) and every source s in snap[u],
// dist[w][s] = min(dist[w][s], dist[u][s] + w(u,w)); a destination that
// improved for any source joins the next frontier. A vertex is queued exactly
// when its act is non-zero, so the lane whose gain finds act zero appends it.
// Label-correcting per source, so each distance is the exact shortest-path
// value. Bound by the random 16-B reads of the distances (L2 misses) and by
// the memory-side atomics; with a lane per edge that walked the sources, and
// long rows in a third launch, a round of 16 sources over 2^20 vertices took
// 320 us on average, now about 200 (64-source BFS over 200,003 vertices: 84
// and 54 us).
struct MsArgs {
    Ctl *ctl;
    const Row *rows;
    uint32_t *dist;
    unsigned long long *act, *snap;
    unsigned long long *reach;  // BFS, in place of act: (seen, done) per vertex
    uint32_t *q0, *q1;
    Tile *tiles;
    ExpandCfg cfg;
    uint32_t n, stride;
    uint64_t seed;
    // BFS pull rounds: incoming rows (null: push only), the frontier size from
    // which a round gathers, the run's source bits
    const Row *in_rows;
    uint32_t pull_min;
    unsigned long long all;
};

__device__ __forceinline__ bool ms_dense(const MsArgs &a, uint32_t nq) { return nq != 0 && nq >= a.pull_min; }

// A group is four sources: one 16-B load of the row owner's distances and one
// of the destination's.
template <int W>
struct MsOp {
    static constexpr int kGroup = 4, kUnroll = 2;
    struct Loaded {
        uint4 du, dw;
    };
    uint32_t *dist;
    unsigned long long *act;
    const unsigned long long *snap;
    uint32_t stride;
    uint64_t seed;
    __device__ unsigned long long mask(uint32_t v) const { return snap[v]; }
    __device__ void load(uint32_t u, uint32_t w, uint32_t g, Loaded &x) const {
        x.du = *reinterpret_cast<const uint4 *>(dist + uint64_t(u) * stride + 4u * g);
        x.dw = *reinterpret_cast<const uint4 *>(dist + uint64_t(w) * stride + 4u * g);
    }
    // A source counts as improved when its candidate beat the value read; if
    // another lane lowered it further meanwhile, w is merely expanded once
    // more for that source with its (smaller) current distance.
    __device__ unsigned long long apply(uint32_t u, uint32_t w, uint32_t g, unsigned long long bits,
                                        const Loaded &x) const {
        const uint32_t wt = weight<W>(u, w, seed);
        uint32_t *dw = dist + uint64_t(w) * stride + 4u * g;
        const uint32_t du[4] = {x.du.x, x.du.y, x.du.z, x.du.w}, cur[4] = {x.dw.x, x.dw.y, x.dw.z, x.dw.w};
        uint32_t gained = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint64_t c = uint64_t(du[i]) + wt;
            if (((uint32_t(bits) >> i) & 1u) && c < cur[i]) {  // also rejects c >= kInf
                __hip_atomic_fetch_min(&dw[i], uint32_t(c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                gained |= 1u << i;
            }
        }
        return static_cast<unsigned long long>(gained) << (4u * g);
    }
    __device__ bool mark(uint32_t w, unsigned long long gained) const { return atomicOr(&act[w], gained) == 0ull; }
};

// BFS from up to 64 sources, bit-parallel (one group): the rounds are
// level-synchronous (a round expands exactly the bits its vertices gained in
// the previous round, all at the same depth), so a destination's depth for
// source s is fixed when bit s first reaches it, and the next round's consume
// phase, which knows the depth, writes it for all of the vertex's new bits
// with whole-line stores. reach[2w] holds the sources that reached w,
// reach[2w+1] those among them that a consume phase has taken: the first
// atomicOr of a round that adds a bit finds the two equal and appends w.
struct MsBfsOp {
    static constexpr int kGroup = 64, kUnroll = 4;
    struct Loaded {
        ulonglong2 r;  // seen, done (seen only grows: a stale read under-reports it)
    };
    unsigned long long *reach;
    const unsigned long long *snap;
    __device__ unsigned long long mask(uint32_t v) const { return snap[v]; }
    __device__ void load(uint32_t, uint32_t w, uint32_t, Loaded &x) const {
        x.r = *reinterpret_cast<const ulonglong2 *>(reach + 2ull * w);
    }
    __device__ unsigned long long apply(uint32_t, uint32_t w, uint32_t, unsigned long long bits, const Loaded &x) const {
        if (!(bits & ~x.r.x)) return 0ull;
        const unsigned long long old = atomicOr(&reach[2ull * w], bits);
        return old == x.r.y ? bits & ~old : 0ull;
    }
    __device__ bool mark(uint32_t, unsigned long long) const { return true; }
};

template <int W>
__device__ __forceinline__ auto ms_op(const MsArgs &a) {
    if constexpr (W == 2) return MsBfsOp{a.reach, a.snap};
    else return MsOp<W>{a.dist, a.act, a.snap, a.stride, a.seed};
}

// The sources of a multi-source run, passed by value (256 B of kernel
// arguments), so that no device copy of them is needed.
struct SrcList {
    uint32_t v[64];
};

__global__ void k_ms_seed(MsArgs a, SrcList sources, uint32_t k, uint32_t ts) {
    stamp_marks(a.ctl, ts);
    const uint32_t r = a.ctl->round;
    for (uint32_t s = gthread(); s < k; s += gthreads()) {
        const uint32_t v = sources.v[s];
        if (!a.reach) a.dist[uint64_t(v) * a.stride + s] = 0;
        if (atomicOr(a.reach ? &a.reach[2ull * v] : &a.act[v], 1ull << s) == 0ull) {
            const uint32_t at = atomicAdd(&a.ctl->qcount[r % 3], 1u);
            ((r & 1) ? a.q1 : a.q0)[at] = v;
        }
    }
}

// Writes `depth` to the distances of v's sources in `mask`, for the 64
// (v, mask) pairs the wave's lanes hold: 16 B per lane, a row's lanes together.
__device__ __forceinline__ void ms_write_depths(uint32_t *dist, uint32_t stride, uint32_t v, unsigned long long mask,
                                                uint32_t depth) {
    if (__ballot(mask != 0ull) == 0) return;
    const uint32_t lane = lane_id(), quads = stride / 4;
    uint32_t g = 1;  // lanes per vertex
    while (g < quads) g <<= 1;
    const uint32_t q = lane & (g - 1);
    for (uint32_t i = lane / g; i < uint32_t(kWave); i += kWave / g) {
        const uint32_t vv = __shfl(v, int(i), kWave);
        const unsigned long long mm = __shfl(mask, int(i), kWave);
        const uint32_t nib = q < quads ? uint32_t(mm >> (4u * q)) & 15u : 0u;
        uint32_t *d = dist + uint64_t(vv) * stride + 4u * q;
        if (nib == 15u) {
            *reinterpret_cast<uint4 *>(d) = make_uint4(depth, depth, depth, depth);
        } else if (nib) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if ((nib >> j) & 1u) d[j] = depth;
        }
    }
}

// Round round+seq-1, phase 1: snapshot and clear the masks of the frontier,
// cut its long rows into tiles (so that phase 2 expands rows and tiles of one
// round in one launch); BFS: write the depths of the bits taken. A dense BFS
// round (ms_dense) walks every vertex instead of the list: its pull needs a
// snapshot of each (0 outside the frontier) and cuts the long incoming rows
// of the vertices that still miss sources. A frontier that a pull left
// without a list (fscan) is found the same way.
template <bool BFS>
__global__ __launch_bounds__(kBlock) void k_ms_consume(MsArgs a, uint64_t *prog, uint64_t tag, uint32_t seq) {
    __shared__ uint32_t scratch[kMaxWavesPerBlock + 1];
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    const bool dense = BFS && ms_dense(a, nq), scan = BFS && nq != 0 && (dense || c->fscan[r % 3] != 0);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        c->qcount[(r + 2) % 3] = 0;
        c->tcount[(r + 2) % 3] = 0;
        c->fscan[(r + 2) % 3] = c->flist[(r + 2) % 3] = 0;
        if (nq) c->rounds += 1;
        post_progress(prog, tag, nq != 0);
    }
    uint32_t *qin = (r & 1) ? a.q1 : a.q0;
    const uint32_t bound = scan ? a.n : nq;
    Counters ctr;
    for (uint32_t base = blockIdx.x * blockDim.x; base < bound; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        bool on = i < bound;
        uint32_t v = 0;
        Row row{};
        unsigned long long m = 0;
        if (on) {
            v = scan ? i : qin[i];
            if constexpr (BFS) {
                const ulonglong2 x = *reinterpret_cast<const ulonglong2 *>(a.reach + 2ull * v);
                m = x.x & ~x.y;
                if (m) a.reach[2ull * v + 1] = x.x;
                if (dense) {
                    a.snap[v] = m;
                    on = (a.all & ~x.x) != 0ull;  // this vertex gathers
                    if (on) row = a.in_rows[v];
                } else {
                    on = !scan || m != 0ull;  // every listed vertex leaves a snapshot
                }
            } else {
                m = a.act[v];
                a.act[v] = 0ull;
            }
            if (on && !dense) {
                row = a.rows[v];
                a.snap[v] = m;
            }
            if (on) {
                ctr.scanned += row.deg;
                ctr.vexp += row.deg ? 1 : 0;
                if (row.off & kHostTier) ctr.host += row.deg;
            }
        }
        if constexpr (BFS) {
            if (scan && !dense) {  // the list the expansion reads
                const uint32_t at = block_reserve<uint32_t>(on ? 1u : 0u, &c->flist[r % 3], scratch);
                if (on) qin[at] = v;
            }
        }
        pair_cut(a.cfg, dense ? a.cfg.tile_len : pair_tile_len(a.cfg), v, row, on, a.tiles, &c->tcount[r % 3], scratch);
        if constexpr (BFS) ms_write_depths(a.dist, a.stride, v, m, seq - 1);
    }
    if (nq) flush_counters(ctr, a.cfg.stats, a.cfg.stage);
}

// BFS pull: the sources that reach v in this round are the OR of its
// in-neighbours' snapshots, so a vertex is written once, by its own lane. In
// a dense push every edge into a hub that has not seen the hub's new bits yet
// queues an atomicOr at the hub (64 sources of 200,003 vertices: rounds of
// 125, 160, 95 and 36 us pushed, 46, 46, 46 and 42 gathered). Bound by the
// gathers, each of which moves a 128-B line into L1 for one snapshot: 3 M
// edges a round, 9 TB/s. 16, 32 and 64 vertices a wave: 50, 46 and 50 us.
constexpr uint32_t kPullVertices = 32;
struct MsPullLds {
    uint32_t pref[kWave], offlo[kWave], offhi[kWave];
    unsigned long long acc[kWave];
};

// The kPullVertices vertices from v0: those that miss sources and have a short row.
__device__ void ms_pull_chunk(const MsArgs &a, uint32_t v0, MsPullLds &L, uint32_t &joined) {
    constexpr uint32_t U = 4;
    const uint32_t lane = lane_id(), v = v0 + lane;
    unsigned long long missing = 0;
    uint32_t deg = 0;
    uint64_t off = 0;
    if (lane < kPullVertices && v < a.n) {
        const Row row = a.in_rows[v];  // with the mask's load, not behind it
        missing = a.all & ~a.reach[2ull * v];
        deg = missing && row.deg < a.cfg.split ? row.deg : 0u;
        off = row.off;
    }
    const uint32_t incl = wave_incl_scan(deg);
    const uint32_t total = __shfl(incl, kWave - 1, kWave);
    if (total == 0) return;
    L.pref[lane] = incl - deg;
    L.offlo[lane] = uint32_t(off);
    L.offhi[lane] = uint32_t(off >> 32);
    L.acc[lane] = 0ull;
    wave_lds_sync();
    for (uint32_t k0 = 0; k0 < total; k0 += kWave * U) {
        uint32_t own[U], rest[U], w[U];
        unsigned long long x[U];
        bool head[U];
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) {
            const uint32_t k = k0 + i * kWave + lane, kk = k < total ? k : total - 1;
            own[i] = owner_of(L.pref, kk);
            const uint32_t at = kk - L.pref[own[i]];
            const uint32_t end = own[i] + 1 < uint32_t(kWave) ? L.pref[own[i] + 1] : total;
            w[i] = a.cfg.pools.row((uint64_t(L.offhi[own[i]]) << 32) | L.offlo[own[i]])[at];
            rest[i] = min(end - 1u - kk, uint32_t(kWave) - 1u - lane);
            head[i] = k < total && (at == 0 || lane == 0);
        }
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) x[i] = a.snap[w[i]];
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) {
            if (__ballot(x[i] != 0ull) == 0) continue;
#pragma unroll
            for (uint32_t d = 1; d < uint32_t(kWave); d <<= 1) {
                const unsigned long long y = __shfl_down(x[i], d, kWave);
                if (d <= rest[i]) x[i] |= y;
            }
            if (head[i]) L.acc[own[i]] |= x[i];
            wave_lds_sync();
        }
    }
    wave_lds_sync();
    const unsigned long long gained = deg ? L.acc[lane] & missing : 0ull;
    if (gained) {
        a.reach[2ull * v] |= gained;
        ++joined;
    }
    wave_lds_sync();  // LDS is reused by the next chunk of this wave
}

// One tile of a long incoming row: one atomic per tile that adds sources.
__device__ void ms_pull_tile(const MsArgs &a, const Tile &t, uint32_t &joined) {
    constexpr uint32_t U = 8;
    const uint32_t lane = lane_id();
    const ulonglong2 cur = *reinterpret_cast<const ulonglong2 *>(a.reach + 2ull * t.v);
    const unsigned long long missing = a.all & ~cur.x;
    if (missing == 0ull) return;
    const uint32_t *p = a.cfg.pools.row(t.start);
    unsigned long long acc = 0;
    for (uint32_t k0 = 0; k0 < t.len; k0 += kWave * U) {
        uint32_t w[U];
        unsigned long long x[U];
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) w[i] = p[min(k0 + i * kWave + lane, t.len - 1)];
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) x[i] = a.snap[w[i]];
#pragma unroll
        for (uint32_t i = 0; i < U; ++i) acc |= x[i];
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) acc |= __shfl_xor(acc, d, kWave);
    if (lane != 0 || (acc & missing) == 0ull) return;
    // the first tile to add sources this round finds seen and done equal
    const unsigned long long old = atomicOr(&a.reach[2ull * t.v], acc & missing);
    if (old == cur.y && (acc & missing & ~old)) ++joined;
}

// Phase 2: expand the frontier's rows and tiles, or gather (a dense BFS round).
template <int W>
__global__ __launch_bounds__(kBlock) void k_ms_expand(MsArgs a, uint32_t seq) {
    using Op = decltype(ms_op<W>(a));
    struct Push {
        PairLds<64 / Op::kGroup> pair[kWavesPerBlock];
        ListStage stage;
    };
    union Lds {
        Push push;
        MsPullLds pull[W == 2 ? kWavesPerBlock : 1];
        __device__ Lds() {}
    };
    __shared__ Lds lds;
    Ctl *c = a.ctl;
    const uint32_t r = c->round + seq - 1;
    const uint32_t nq = c->qcount[r % 3];
    if (nq == 0) return;
    const uint32_t nt = c->tcount[r % 3];
    if constexpr (W == 2) {
        if (ms_dense(a, nq)) {
            __shared__ uint32_t total;
            uint32_t joined = 0;
            const uint32_t gw = wave_in_block() * gridDim.x + blockIdx.x, nw = gwaves();
            for (uint32_t t = gw; t < nt; t += nw) ms_pull_tile(a, a.tiles[t], joined);
            const uint32_t chunks = (a.n + kPullVertices - 1) / kPullVertices;
            for (uint32_t ch = gw; ch < chunks; ch += nw)
                ms_pull_chunk(a, ch * kPullVertices, lds.pull[wave_in_block()], joined);
            frontier_count(c, (r + 1) % 3, joined, &total);
            return;
        }
    }
    const Op op = ms_op<W>(a);
    const StagedOut<1024, 2> out{Sink{(r & 1) ? a.q0 : a.q1, &c->qcount[(r + 1) % 3]}, TileSink{nullptr, &c->scount},
                                 &lds.push.stage};
    out_init(out);
    PairLds<64 / Op::kGroup> &L = lds.push.pair[wave_in_block()];
    pair_range<Op::kGroup, Op::kUnroll>(op, a.cfg, a.rows, (r & 1) ? a.q1 : a.q0, nq, L, out);
    pair_tiles<Op::kGroup, Op::kUnroll>(op, a.cfg, a.tiles, nt, L, out);
    out_flush(out);
}

// Source-major result: out[s * n + v] = the word of (v, s) in `src`, whose
// vertex-major rows hold `stride` elements. FIELD: 0 = 32-bit words
// (distances), 1 / 2 = the value (high) / parent (low) half of 64-bit state
// words. A workgroup turns tiles of 64 vertices around in LDS, so both sides
// move whole lines: bound by HBM. Element by element in output order, each
// 4-B read fetched a line of its own and each element paid two 64-bit
// divisions (64 sources of 200,003 vertices, 102 MB moved: 224 us, now about 22).
template <int FIELD>
__global__ __launch_bounds__(kBlock) void k_ms_gather(const void *src, uint32_t n, uint32_t stride, uint32_t k,
                                                      uint32_t *out) {
    __shared__ uint32_t tile[kWave][kWave + 1];  // a column walks all banks
    const uint32_t lane = lane_id(), w = wave_in_block();
    uint32_t kw = 1;  // lanes of a vertex when reading
    while (kw < k) kw <<= 1;
    const uint32_t s = lane & (kw - 1), sub = lane / kw, vpw = kWave / kw;
    const uint32_t ntiles = (n + kWave - 1) / kWave;
    for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const uint32_t v0 = t * kWave, nv = min(uint32_t(kWave), n - v0);
#pragma unroll 4
        for (uint32_t v = w * vpw + sub; v < kWave; v += kWavesPerBlock * vpw) {
            if (v >= nv || s >= k) continue;
            const uint64_t at = uint64_t(v0 + v) * stride + s;
            if constexpr (FIELD == 0) tile[v][s] = static_cast<const uint32_t *>(src)[at];
            else tile[v][s] = static_cast<const uint32_t *>(src)[2 * at + (FIELD == 1 ? 1 : 0)];
        }
        __syncthreads();
#pragma unroll 4
        for (uint32_t j = w; j < k; j += kWavesPerBlock)
            if (lane < nv) out[uint64_t(j) * n + v0 + lane] = tile[lane][j];
        __syncthreads();
    }
}

// Results of one source: the value (high = 1) or parent half of each state
// word, so that 4 B a vertex leave the device instead of 8 B that the host
// then took apart (2^22 vertices: 8.6 ms for a gather, now 0.6).
__global__ void k_state_words(const uint64_t *state, uint32_t n, uint32_t high, uint32_t *out) {
    for (uint32_t v = gthread(); v < n; v += gthreads()) out[v] = uint32_t(high ? state[v] >> 32 : state[v]);
}

// out[v] = src[perm[v]]: a renumbered engine's words in the caller's order
// (perm null: as they are).
__global__ void k_permute_words(const uint32_t *src, const uint32_t *perm, uint32_t n, uint32_t *out) {
    for (uint32_t v = gthread(); v < n; v += gthreads()) out[v] = src[perm ? perm[v] : v];
}

// Plain streaming copy (16 B per lane per step): the HBM reference point for
// rocprofv3 FETCH_SIZE / WRITE_SIZE calibration and achievable bandwidth.
__global__ void k_copy_probe(const uint4 *src, uint4 *dst, uint64_t n16) {
    for (uint64_t i = gthread(); i < n16; i += gthreads()) dst[i] = src[i];
}

// Zero-copy read of pinned host memory (16 B per lane per step): the
// host-link reference point for rows in the host tier. The XOR of what each
// thread read goes to `sink` so that the loads stay.
__global__ void k_host_read_probe(const uint4 *src, uint64_t n16, uint32_t *sink) {
    uint32_t x = 0;
    for (uint64_t i = gthread(); i < n16; i += gthreads()) {
        const uint4 v = src[i];
        x ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    if (x == 0x9E3779B9u) sink[0] = x;  // practically never; keeps the loads
}

// FP64 residual norm sum |r| (the only FP64 arithmetic of the PR path).
__global__ void k_pr_l1(const float *res, uint32_t n, StatShard *stats) {
    double s = 0;
    for (uint32_t v = gthread(); v < n; v += gthreads()) s += fabs(double(res[v]));
    for (int d = kWave / 2; d > 0; d >>= 1) s += __shfl_xor(s, d, kWave);
    if (lane_id() == 0 && s != 0) atomicAdd(&stat_shard(stats)->l1, s);
}

// Folds the statistics shards into the control block (adding to its
// totals) and clears them. One wave: lane j reads shard j.
__device__ void reduce_stats(StatShard *stats, Ctl *c) {
    static_assert(kStatShards == kWave, "one lane per shard");
    const uint32_t j = threadIdx.x;
    uint64_t *w = reinterpret_cast<uint64_t *>(stats + j);
    uint64_t v[kStatWords];
#pragma unroll
    for (uint32_t f = 0; f < kStatWords; ++f) {
        v[f] = wave_sum64(w[f]);
        w[f] = 0;
    }
    double l1 = stats[j].l1;
    stats[j].l1 = 0;
    for (int d = kWave / 2; d > 0; d >>= 1) l1 += __shfl_xor(l1, d, kWave);
    if (j == 0) {
        for (int i = 0; i < 4; ++i) {
            c->st_edges[i] += v[i];
            c->st_vexp[i] += v[4 + i];
            c->st_host[i] += v[8 + i];
            c->edges_scanned += v[i];
            c->vexp += v[4 + i];
            c->host_edges += v[8 + i];
        }
        c->deletes_applied += v[12];
        c->missing += v[13];
        c->invalid += v[14];
        c->adds_applied += v[15];
        c->relocated += v[16];
        c->garbage[0] += v[17];
        c->garbage[1] += v[18];
        c->touched_sources += v[19];
        c->residual_l1 += l1;
    }
}

__global__ void k_reduce_stats(StatShard *stats, Ctl *c) { reduce_stats(stats, c); }

// End of a call, one wave: notes the last markers, advances the round counter
// past the call's last chain, folds the statistics, and publishes the control
// block to mapped pinned host memory, then its sequence number (system scope,
// after a system fence), so the host reads it by polling one word instead of
// a copy and a stream synchronisation.
struct CtlPub {
    Ctl c;
    uint64_t seq;
};
__global__ void k_end_call(Ctl *c, StatShard *stats, CtlPub *pub, uint64_t seq, uint32_t rounds, uint32_t ts) {
    static_assert(sizeof(Ctl) % 8 == 0, "whole words");
    constexpr uint32_t kWords = sizeof(Ctl) / 8;
    if (threadIdx.x == 0) {
        stamp_marks(c, ts);
        c->round += rounds;
    }
    reduce_stats(stats, c);
    __threadfence();
    __syncthreads();
    const uint64_t *src = reinterpret_cast<const uint64_t *>(c);
    uint64_t *dst = reinterpret_cast<uint64_t *>(&pub->c);
    for (uint32_t i = threadIdx.x; i < kWords; i += blockDim.x) dst[i] = ld_acquire(&src[i]);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(&pub->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Pool compaction: copies every row of `tier` to its new offset.
__global__ void k_relocate_rows(const Row *old_rows, Row *new_rows, uint32_t n, uint32_t tier,
                                const uint32_t *src_pool, uint32_t *dst_pool) {
    const uint32_t lane = lane_id();
    for (uint32_t v = gwave(); v < n; v += gwaves()) {
        const Row o = old_rows[v];
        const bool in_tier = ((o.off & kHostTier) != 0) == (tier == 1);
        if (!in_tier || o.deg == 0) continue;
        const Row nr = new_rows[v];
        const uint32_t *s = src_pool + (o.off & ~kHostTier);
        uint32_t *d = dst_pool + (nr.off & ~kHostTier);
        for (uint32_t q = lane; q < o.deg; q += kWave) d[q] = s[q];
    }
}

// ------------------------------------------------ in-place pool compaction
// Replaces the full-budget compaction copy (driver.cuh:236-247): the rows of
// one tier are bucketed by windows of `wslots` slots of their current offset.
// Window k's rows are packed into a staging buffer and then written to their
// final places, starting at the total capacity of the earlier windows. Rows
// do not overlap, so everything window k writes lies below its last row's
// end, i.e. below every row of window k+1 (not yet moved), and nothing is
// overwritten before it is read. No second pool and no host copy of the rows.
constexpr uint32_t kCmpMaxWin = 1024;
constexpr uint32_t kCmpChunk = 1u << 16;  // rows per workgroup of the bucketing passes

struct CmpJob {
    uint64_t from;   // current offset (tier bit kept)
    uint64_t spos;   // position in the staging buffer = offset within the window's packed range
    uint32_t len;    // live slots
    uint32_t row;
    uint32_t pfirst;  // first of the row's copy pieces
    uint32_t pad;
};

// Rows are copied in pieces of kCmpPiece slots, a wave per piece, so that a
// hub row of millions of slots is spread over the whole chip. Row blocks are
// powers of two of at least 4 slots at offsets that are sums of such blocks,
// so every row (and its staging place) starts 16-B aligned and rounding its
// length up to whole quads stays inside its block.
constexpr uint32_t kCmpPiece = 2048;

struct CmpArgs {
    Row *rows;
    uint32_t nrows, tier, nwin;
    uint64_t wslots;
    unsigned long long *wcnt, *wcap;  // per window: rows, capacity
    unsigned long long *lfill;        // per window: next free list position
    uint32_t *list;                   // row ids grouped by window
    Pools pools;
};

__device__ __forceinline__ bool cmp_in_tier(const Row &r, uint32_t tier) {
    return r.cap != 0 && ((r.off & kHostTier) != 0) == (tier == 1);
}

// Per window: rows and capacity (LDS counts per workgroup chunk).
__global__ void k_cmp_hist(CmpArgs a) {
    __shared__ unsigned long long cnt[kCmpMaxWin], cap[kCmpMaxWin];
    for (uint32_t w = threadIdx.x; w < a.nwin; w += blockDim.x) cnt[w] = cap[w] = 0;
    __syncthreads();
    const uint64_t lo = uint64_t(blockIdx.x) * kCmpChunk, hi = min<uint64_t>(a.nrows, lo + kCmpChunk);
    for (uint64_t v = lo + threadIdx.x; v < hi; v += blockDim.x) {
        const Row r = a.rows[v];
        if (!cmp_in_tier(r, a.tier)) continue;
        const uint32_t w = uint32_t((r.off & ~kHostTier) / a.wslots);
        atomicAdd(&cnt[w], 1ull);
        atomicAdd(&cap[w], (unsigned long long)r.cap);
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < a.nwin; w += blockDim.x) {
        if (cnt[w]) atomicAdd(&a.wcnt[w], cnt[w]);
        if (cap[w]) atomicAdd(&a.wcap[w], cap[w]);
    }
}

// Row ids grouped by window (lfill starts at each window's list base).
__global__ void k_cmp_scatter(CmpArgs a) {
    __shared__ unsigned long long cnt[kCmpMaxWin], base[kCmpMaxWin];
    for (uint32_t w = threadIdx.x; w < a.nwin; w += blockDim.x) cnt[w] = 0;
    __syncthreads();
    const uint64_t lo = uint64_t(blockIdx.x) * kCmpChunk, hi = min<uint64_t>(a.nrows, lo + kCmpChunk);
    for (uint64_t v = lo + threadIdx.x; v < hi; v += blockDim.x) {
        const Row r = a.rows[v];
        if (cmp_in_tier(r, a.tier)) atomicAdd(&cnt[uint32_t((r.off & ~kHostTier) / a.wslots)], 1ull);
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < a.nwin; w += blockDim.x) {
        base[w] = cnt[w] ? atomicAdd(&a.lfill[w], cnt[w]) : 0ull;
        cnt[w] = 0;
    }
    __syncthreads();
    for (uint64_t v = lo + threadIdx.x; v < hi; v += blockDim.x) {
        const Row r = a.rows[v];
        if (!cmp_in_tier(r, a.tier)) continue;
        const uint32_t w = uint32_t((r.off & ~kHostTier) / a.wslots);
        a.list[base[w] + atomicAdd(&cnt[w], 1ull)] = uint32_t(v);
    }
}

// One window: each row's place in the packed range (workgroup-aggregated
// reservations on the window's cursor), its copy pieces and its job.
__global__ void k_cmp_plan(CmpArgs a, const uint32_t *list, uint32_t cnt, unsigned long long *cursor,
                           uint32_t *pcursor, CmpJob *jobs, uint32_t *pjob) {
    __shared__ unsigned long long scratch64[kMaxWavesPerBlock + 1];
    __shared__ uint32_t scratch32[kMaxWavesPerBlock + 1];
    for (uint32_t base = blockIdx.x * blockDim.x; base < cnt; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        Row r{};
        uint32_t v = 0, np = 0;
        if (i < cnt) {
            v = list[i];
            r = a.rows[v];
            np = max(1u, (r.deg + kCmpPiece - 1) / kCmpPiece);  // an empty row still gets its offset
        }
        const uint64_t pos = block_reserve<unsigned long long>(i < cnt ? r.cap : 0ull, cursor, scratch64);
        const uint32_t pf = block_reserve<uint32_t>(np, pcursor, scratch32);
        if (i < cnt) {
            jobs[i] = CmpJob{r.off, pos, r.deg, v, pf, 0u};
            for (uint32_t k = 0; k < np; ++k) pjob[pf + k] = i;
        }
    }
}

// Copies slots [k*kCmpPiece, ...) of a row, whole quads, by one wave.
__device__ __forceinline__ void cmp_copy_piece(uint32_t *d, const uint32_t *s, uint32_t len, uint32_t k) {
    const uint32_t lo = k * kCmpPiece, hi = min(len, lo + kCmpPiece);
    if (hi <= lo) return;
    const uint32_t nq = (hi - lo + 3u) >> 2;
    const uint4 *sq = reinterpret_cast<const uint4 *>(s + lo);
    uint4 *dq = reinterpret_cast<uint4 *>(d + lo);
    for (uint32_t q = lane_id(); q < nq; q += kWave) dq[q] = sq[q];
}

// Live slots into the staging buffer (a wave per piece).
__global__ void k_cmp_in(CmpArgs a, const CmpJob *jobs, const uint32_t *pjob, const uint32_t *pcount,
                         uint32_t *stage) {
    const uint32_t np = *pcount;
    for (uint32_t p = gwave(); p < np; p += gwaves()) {
        const CmpJob jb = jobs[pjob[p]];
        cmp_copy_piece(stage + jb.spos, a.pools.row(jb.from), jb.len, p - jb.pfirst);
    }
}

// From the staging buffer to the final place, which the row now names.
__global__ void k_cmp_out(CmpArgs a, const CmpJob *jobs, const uint32_t *pjob, const uint32_t *pcount,
                          const uint32_t *stage, uint64_t newbase) {
    const uint64_t tbit = a.tier ? kHostTier : 0ull;
    const uint32_t np = *pcount;
    for (uint32_t p = gwave(); p < np; p += gwaves()) {
        const CmpJob jb = jobs[pjob[p]];
        const uint64_t off = (newbase + jb.spos) | tbit;
        cmp_copy_piece(a.pools.row(off), stage + jb.spos, jb.len, p - jb.pfirst);
        if (p == jb.pfirst && lane_id() == 0) a.rows[jb.row].off = off;
    }
}

// Lists the host-tier blocks that rows loaded into HBM vacated (k_move_rows,
// which copied them, ran before).
__global__ void k_move_release(const CopyJob *jobs, const uint32_t *njobs, FreeList fl) {
    const uint32_t cnt = ld_acquire(njobs);
    for (uint32_t j = gthread(); j < cnt; j += gthreads()) {
        const CopyJob jb = jobs[j];
        if ((jb.from & kHostTier) && jb.cap) fl_push(fl, fl_class(jb.cap), jb.from & ~kHostTier);
    }
}

// Moves rows between tiers (cache admission / eviction). Each job names a row
// whose descriptor has already been rewritten; `from` is the old location.
// A wave per copy piece (see kCmpPiece), whole quads.
__global__ void k_move_rows(const CopyJob *jobs, const uint32_t *pjob, const uint32_t *pcount, Pools pools) {
    const uint32_t np = ld_acquire(pcount);
    for (uint32_t p = gwave(); p < np; p += gwaves()) {
        const CopyJob jb = jobs[pjob[p]];
        cmp_copy_piece(pools.row(jb.to), pools.row(jb.from), jb.len, p - jb.pfirst);
    }
}

// ------------------------------------------------------- cache admission
// Device form of compute_hot_vertices + confirm_candidate_batch
// (framework.cuh:605-729): rows are admitted to HBM by decreasing activity
// score until 90% of the budget is used. Scores are sums of four 8-bit
// window counts (<= 1020), so a per-score capacity histogram replaces the
// reference's sort: the host walks it from the top to find the threshold
// score, rows above it are admitted, rows at it share what room is left.
constexpr uint32_t kScoreBuckets = 1024;

__global__ void k_adm_hist(const Row *rows, const uint32_t *score, uint32_t nrows, unsigned long long *hist) {
    __shared__ unsigned long long h[kScoreBuckets];
    for (uint32_t i = threadIdx.x; i < kScoreBuckets; i += blockDim.x) h[i] = 0ull;
    __syncthreads();
    for (uint32_t v = gthread(); v < nrows; v += gthreads()) {
        const uint32_t cap = rows[v].cap;
        if (cap) atomicAdd(&h[min(score[v], kScoreBuckets - 1)], (unsigned long long)cap);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kScoreBuckets; i += blockDim.x)
        if (h[i]) atomicAdd(&hist[i], h[i]);
}

struct AdmArgs {
    const Row *rows;
    const uint32_t *score;
    uint32_t nrows;
    uint32_t thr;              // rows scoring above thr are admitted, below it not
    unsigned long long room;   // slots for rows scoring exactly thr
    unsigned long long *acc;   // [0] room used, [1] evict slots, [2] load slots
    uint32_t *evict, *load;    // rows leaving / entering HBM
    uint32_t *evict_cnt, *load_cnt;
};

// Lists the rows that change tier. Rows scoring exactly thr take the room
// in two passes, rows already in HBM first (pass 0), so that a threshold
// bucket that fits moves nothing; the room is reserved per workgroup step.
__global__ void k_adm_mark(AdmArgs a, uint32_t pass) {
    __shared__ unsigned long long s64[kMaxWavesPerBlock + 1];
    __shared__ uint32_t s32[kMaxWavesPerBlock + 1];
    for (uint32_t base = blockIdx.x * blockDim.x; base < a.nrows; base += gthreads()) {
        const uint32_t v = base + threadIdx.x;
        Row r{};
        uint32_t sc = 0;
        if (v < a.nrows) {
            r = a.rows[v];
            sc = min(a.score[v], kScoreBuckets - 1);
        }
        const bool cached = r.cap && !(r.off & kHostTier);
        const bool cand = r.cap && sc == a.thr && (pass == 0 ? cached : !cached);
        const unsigned long long at =
            block_reserve<unsigned long long>(cand ? (unsigned long long)r.cap : 0ull, &a.acc[0], s64);
        bool decided = false, admit = false;
        if (r.cap && sc != a.thr && pass == 0) {
            decided = true;
            admit = sc > a.thr;
        } else if (cand) {
            decided = true;
            admit = at + r.cap <= a.room;
        }
        const bool ev = decided && cached && !admit, ld = decided && !cached && admit;
        block_reserve<unsigned long long>(ev ? (unsigned long long)r.cap : 0ull, &a.acc[1], s64);
        block_reserve<unsigned long long>(ld ? (unsigned long long)r.cap : 0ull, &a.acc[2], s64);
        block_append(ev, v, a.evict, a.evict_cnt, s32);
        block_append(ld, v, a.load, a.load_cnt, s32);
    }
}

// New blocks in `tier` for the listed rows (bump allocation from the tier's
// tail, one reservation per workgroup step), the copy jobs, the rows' new
// offsets; the vacated blocks become garbage of the other tier.
__global__ void k_move_plan(Row *rows, const uint32_t *list, const uint32_t *count, uint32_t tier, Ctl *c,
                            CopyJob *jobs, uint32_t *pcount, uint32_t *pjob, FreeList fl) {
    __shared__ unsigned long long s64[kMaxWavesPerBlock + 1];
    __shared__ uint32_t s32[kMaxWavesPerBlock + 1];
    const uint32_t cnt = ld_acquire(count);
    for (uint32_t base = blockIdx.x * blockDim.x; base < cnt; base += gthreads()) {
        const uint32_t i = base + threadIdx.x;
        Row r{};
        uint32_t v = 0, np = 0;
        uint64_t popped = 0;
        bool reuse = false;
        if (i < cnt) {
            v = list[i];
            r = rows[v];
            np = max(1u, (r.deg + kCmpPiece - 1) / kCmpPiece);
            // an evicted row takes a freed host-tier block of its class when one is listed
            reuse = tier == 1 && fl_pop(fl, fl_class(r.cap), popped);
        }
        const unsigned long long bumped = block_reserve<unsigned long long>(
            reuse ? 0ull : (unsigned long long)r.cap, reinterpret_cast<unsigned long long *>(&c->pool_tail[tier]),
            s64);
        const unsigned long long at = reuse ? popped : bumped;
        block_reserve<unsigned long long>((unsigned long long)r.cap,
                                          reinterpret_cast<unsigned long long *>(&c->garbage[1 - tier]), s64);
        const uint32_t pf = block_reserve<uint32_t>(np, pcount, s32);
        if (i < cnt) {
            CopyJob j;
            j.from = r.off;
            j.to = at | (tier ? kHostTier : 0ull);
            j.len = r.deg;
            j.pfirst = pf;
            j.cap = r.cap;
            j.pad = 0;
            jobs[i] = j;
            rows[v].off = j.to;
            for (uint32_t k = 0; k < np; ++k) pjob[pf + k] = i;
        }
    }
}

// Activity window (comp_hotness_sssp / reset_hotness, driver.cuh:462-521):
// history keeps four 8-bit saturating window counts; score = their sum.
__global__ void k_age_hotness(uint32_t *hot, uint32_t *hist, uint32_t *score, uint32_t n) {
    for (uint32_t v = gthread(); v < n; v += gthreads()) {
        const uint32_t h = min(hot[v], 255u);
        const uint32_t nh = (hist[v] << 8) | h;
        hist[v] = nh;
        hot[v] = 0;
        score[v] = (nh & 255u) + ((nh >> 8) & 255u) + ((nh >> 16) & 255u) + (nh >> 24);
    }
}

}  // namespace dev
}  // namespace cig
