// One query searched by the whole GPU (grid mode): the near/far piles of
// slot_search.h shared by a persistent grid.
//
// Open entries (f << 32 | node) sit in a near ring (f below a threshold) and
// a far pile.  A round takes the near entries (up to kPgRound); eight lanes
// expand one, and the chunks of eight entries a wave takes are dealt over the
// workgroups.  Rows longer than kPgSeg edges are
// cut into segments that the round's second step spreads over the whole grid:
// a power-law hub would otherwise keep one workgroup busy while the others
// wait at the barrier.  When the near ring is empty the threshold moves to the
// far pile's lower bound plus a window width, and one pass sends the entries
// under it to the near ring and compacts the other live ones into the second
// far buffer (which gives the next lower bound; it is exact up to entries that
// have gone stale since).  As in the slots this is a label-correcting search:
// an entry is dropped only when it is stale or cannot lead to anything below
// F(t), so the cost is exact for an admissible heuristic.  K sets the window:
// a width that fed fewer than K entries, or few a round (kPgFeed), doubles, one
// that fed more than 8K halves.
//
// Why piles and not the K lane heaps this replaced: a heap pop is a chain of
// dependent LDS and HBM accesses (8 us an iteration on the 100,000-node random
// graph, 41 us on R-MAT scale 20), an entry was expanded by its own lane's
// wave however long its row (R-MAT: 135 us, and 94 us of waiting for the
// workgroup with the hub), and K lanes were all the parallelism there was.
// Measured, whole call, heaps and piles: random graph of 100,000 nodes, K = 1,024,
// 1.5-3.1 and 0.39-0.43 ms; R-MAT scale 20, K = 16,384, 9.8-11.2 and 2.0-2.9 ms;
// 4,096 x 4,096 maze, K = 1,024, 26 and 18.7 ms.  What is left is latency: a round
// is six dependent round trips (the entry; its word, row and heuristic input;
// its edges; their ends' words and inputs; the atomics; places in the piles)
// and a barrier, 6 us.
//
// RESUME (DA*): the search starts from an open set -- the first entries of far0,
// counted on the device -- with F(t) read from the target's word, and a current
// entry that cannot beat F(t) goes to a dormant pile instead of being dropped:
// a later batch may raise F(t) again. On return the dormant pile holds the open
// set for the next resume.  Every relaxation is kept, whatever F(t) is.
//
// Everything workgroups share -- the (f, parent) words, the piles, the control
// words -- is accessed through agent-scope atomics only, as grid_sync needs.
// The workgroups are a team (grid_team.h): those of the launch that are resident
// together.  A round's steps each end with grid_sync; what a step appended is counted in
// one of three rotating slots, read by everybody after the barrier and cleared
// two steps later, so all workgroups take every decision from the same values.
#pragma once

#include "gastar.h"
#include "search_expand.h"

// Control words behind the result words of gastar.h (a 128-byte line each).
enum : int {
    PG_NEAR = 0, PG_FAR = 32, PG_TMIN = 64, PG_FMIN = 96, PG_HUBS = 128, PG_ERR = 129, PG_SLOT_WORDS = 160,
    PG_SLOTS = 128, PG_BAR = PG_SLOTS + 3 * PG_SLOT_WORDS, PG_TEAM = PG_BAR + GRID_SYNC_WORDS,
    PG_WORDS = PG_TEAM + TEAM_WORDS
};
static_assert(PG_WORDS <= GA_CTRL_WORDS, "control block too small");

constexpr int32_t kPgSeg = 64;    // edges per hub segment
constexpr int kPgLanes = 8;       // lanes per entry
constexpr int kPgUnroll = 2;      // edges per lane and step
constexpr int kPgBlock = 1024;
// Workgroups: 64 (a barrier of 1.9 us); one per CU (2.6 us) where a round scans
// hundreds of thousands of edges -- searches without a geometric heuristic on
// graphs of kPgWideEdges edges and more; 16 (1.4 us, and a launch that starts in a
// third of the time) below kPgSmallEdges edges.  A call in us with 16, 64 and 256
// workgroups:
//   random graph     6,000 edges   204   244   402     maze 64 x 64   198   235   397
//                  300,000         342   323   483     maze 256^2   1,638 1,681 2,014
//                  600,000         597   428   569     map, 200,000   589   619   818
//   R-MAT          196,000         384   380   532          1,000,000 1,254 1,275 1,542
//                  786,000         676   593   747
// (of a server's versioned view, with its insert lists, R-MAT of 196,000: 404 and 368)
// and in ms with 64, 128 and 256:
//   random graph   4.0M edges  0.58 0.58 0.66   R-MAT  2.1M  0.50 0.52 0.60
//                  8.0M        0.95 0.75 0.91          4.2M  1.10 1.02 1.05
//                 10.0M        1.23 0.84 0.85          8.4M  2.04 1.52 1.50
//                 16.0M        2.01 1.43 1.26         16.8M  3.75 2.23 1.70
//                 32.0M        2.05 1.37 1.46         33.6M  8.09 6.86 5.77
// A geometric heuristic keeps rounds small at any size (map of 20M edges, 64 and
// 256 workgroups without heuristic 5.7 and 6.4).
constexpr int kPgBlocks = 64, kPgSmallBlocks = 16;
constexpr int64_t kPgWideEdges = 1 << 22, kPgSmallEdges = 1 << 17;

// For a graph of E edges on a GPU of `cus` CUs.
inline int32_t pg_workgroups(int64_t E, bool geometric, int32_t cus)
{
    const int32_t most = E >= kPgWideEdges && !geometric ? cus : E < kPgSmallEdges ? kPgSmallBlocks : kPgBlocks;
    return most < cus ? most : cus;
}
// Near entries a round takes at most.  Taking the whole window at once saves
// rounds and costs little order, which the window's width keeps: 8,192 against
// 65,536 entries took 0.39 and 0.32 ms on the random graph (K = 1,024), 0.68
// and 0.36 ms on one of 300,000 nodes at K = 256.
constexpr uint32_t kPgRound = 65536;
// Near entries a window's rounds take on average at least: a window of fewer
// doubles too, however many it fed in all.  A round costs 6 us whatever it takes,
// and on a maze with the Manhattan heuristic a chain of thousands of rounds of 15
// entries passed the K test: 4,096 x 4,096 took 76 ms (12,477 rounds), now 26
// (3,928; K = 1,024); 512 x 512 8.8 and 6.0; a map of 1M nodes without heuristic 12.6
// and 6.5 (64 entries instead of 512: 12.6).  Random graphs, R-MAT and maps with
// their heuristic are the same within 1%.
constexpr uint32_t kPgFeed = 512;
// The first window: the mean weight, or 32 of them with the Manhattan heuristic.
// There f grows by two a detour, so windows of a few steps are chains of rounds of
// a handful of entries until they have doubled often enough: 21 mazes of 64 x 64
// to 1,500 x 1,500 (2 queries each, K = 1,024) took 0.74 to 1.6 times as long as on lane
// heaps, now 0.59 to 0.87; 4,096 x 4,096 25.9 and 18.7 ms.  Other searches keep the
// mean: wider ones make R-MAT of scale 16 0.59 -> 0.69 ms, and random graphs of
// 500,000 nodes 0.40 -> 0.69 from 8 on.
inline uint32_t pg_first_window(uint32_t mean, bool manhattan)
{
    const uint64_t d = (uint64_t)mean * (manhattan ? 32 : 1);
    return d < 0x7FFFFFFFu ? (uint32_t)d : 0x7FFFFFFFu;
}
// Near entries that count as stragglers: with 256 the split ran ahead of f
// order on mazes (703,000 expansions against 56,000 without early splits).
constexpr uint32_t kPgThin = 64;

struct PgArgs {
    GraphView g;
    HeurView h;
    uint64_t *gp;
    uint64_t *near;       // ring of nmask + 1 entries
    uint64_t *far0, *far1;
    uint64_t *hubs;       // 2 words per segment: start | length << 32, node | g << 32
    uint32_t nmask, fcap, hubcap;
    uint32_t *ctrl;
    unsigned long long *stats;
    // RESUME: the dormant pile (dcap entries) and its count, the live entries'
    // count and smallest f, and whether counting them overflowed
    uint64_t *dorm;
    uint32_t dcap;
    uint32_t *dorm_n;
    const uint32_t *live_n, *live_min, *live_ovf;
    // rebuild: piles that overflow are rebuilt from the N nodes' words (the ring
    // and each far buffer hold N entries at least)
    int32_t N, rebuild;
    int32_t t, maxit;
    uint32_t grow;        // K: a window that fed fewer entries doubles, one that fed 8 times as many halves
    uint32_t thr0, delta0;
    uint64_t barrier_ticks;
};

// Where a step's improvements go: staged in LDS, and placed with one atomic
// per workgroup and pile when the step ends; what LDS cannot hold is placed
// by its wave at once.
template <int B, bool RESUME>
struct PgStage {
    static constexpr uint32_t kCap = 2 * B;
    static constexpr int kPiles = RESUME ? 3 : 2;
    uint64_t q[kPiles][kCap];            // near, far, dormant
    uint32_t n[kPiles], base[kPiles];
    uint32_t tmin, fmin, err;
};

// Error bits beside GA_ERR_*: the piles overflowed and are to be rebuilt.
constexpr uint32_t PG_ERR_REBUILD = 0x100;

template <int B, bool RESUME>
struct PgPush {
    using Stage = PgStage<B, RESUME>;
    Stage *S;
    const PgArgs *a;
    uint32_t *slot;       // this step's counters
    uint32_t nbase, head; // ring positions where this step's appends start, and of the oldest entry
    uint64_t *far;
    uint32_t fbase;
    uint32_t thr, F;
    uint32_t fmin = 0xFFFFFFFFu;  // smallest f this lane sent to the far pile

    __device__ __forceinline__ uint32_t *counter(int pile) const
    {
        return pile == 0 ? slot + PG_NEAR : pile == 1 ? slot + PG_FAR : a->dorm_n;
    }
    // entry k of what this step appends to the pile (of the dormant pile: entry k)
    __device__ __forceinline__ void put(int pile, uint32_t k, uint64_t key) const
    {
        bool ok;
        if (pile == 0) {
            const uint32_t pos = nbase + k;
            ok = pos - head <= a->nmask;
            if (ok) st_u64(a->near + (pos & a->nmask), key);
        } else if (pile == 1) {
            const uint64_t pos = (uint64_t)fbase + k;
            ok = pos < a->fcap;
            if (ok) st_u64(far + pos, key);
        } else {
            ok = k < a->dcap;
            if (ok) st_u64(a->dorm + k, key);
        }
        if (!ok) atomicOr(&S->err, a->rebuild ? PG_ERR_REBUILD : (uint32_t)GA_ERR_HEAP);
    }
    __device__ __forceinline__ void target(uint32_t f) const { atomicMin(&S->tmin, f); }
    __device__ __forceinline__ void touch(int32_t, uint64_t) const {}
    template <int R>
    __device__ __forceinline__ void touch_all(const bool (&)[R], const int32_t (&)[R]) const {}
    // wave-collective
    template <int R>
    __device__ __forceinline__ void all(const bool (&has)[R], const uint64_t (&key)[R])
    {
#pragma unroll
        for (int pile = 0; pile < Stage::kPiles; ++pile) {
            bool sel[R];
            uint32_t pos[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t f = (uint32_t)(key[r] >> 32);
                sel[r] = has[r] && (f < F ? (f < thr ? 0 : 1) : 2) == pile;
                if (pile == 1 && sel[r] && f < fmin) fmin = f;
            }
            wave_append<R>(sel, &S->n[pile], pos);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (sel[r] && pos[r] < Stage::kCap) S->q[pile][pos[r]] = key[r];
                const bool over[1] = {sel[r] && pos[r] >= Stage::kCap};
                if (__any(over[0])) {
                    uint32_t k[1];
                    wave_append<1>(over, counter(pile), k);
                    if (over[0]) put(pile, k[0], key[r]);
                }
            }
        }
    }
    // block-collective: the staged entries to their piles
    __device__ __forceinline__ void flush()
    {
        const int lane = threadIdx.x;
        if (__any(fmin != 0xFFFFFFFFu)) {
            const uint32_t m = wave_min_u32(fmin);
            if ((lane & 63) == 0) atomicMin(&S->fmin, m);
        }
        __syncthreads();
        if ((lane & 63) == 0 && lane < 64 * Stage::kPiles) {  // a wave per pile, so that the round trips overlap
            const int pile = lane >> 6;
            const uint32_t m = S->n[pile] < Stage::kCap ? S->n[pile] : Stage::kCap;
            S->base[pile] = m ? add_u32(counter(pile), m) : 0;
        } else if (lane == 192) {
            if (S->fmin != 0xFFFFFFFFu)
                (void)__hip_atomic_fetch_min(slot + PG_FMIN, S->fmin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (S->tmin != 0xFFFFFFFFu)
                (void)__hip_atomic_fetch_min(slot + PG_TMIN, S->tmin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
#pragma unroll
        for (int pile = 0; pile < Stage::kPiles; ++pile) {
            const uint32_t m = S->n[pile] < Stage::kCap ? S->n[pile] : Stage::kCap;
            for (uint32_t k = lane; k < m; k += B) put(pile, S->base[pile] + k, S->q[pile][k]);
        }
        __syncthreads();
        if (lane == 0) {
            if (S->err) (void)__hip_atomic_fetch_or(slot + PG_ERR, S->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int pile = 0; pile < Stage::kPiles; ++pile) S->n[pile] = 0;
            S->tmin = S->fmin = 0xFFFFFFFFu;
            S->err = 0;
        }
    }
};

// The edges [start, start + len) of node u (g value gu) by the eight lanes of
// a group; every lane of the wave calls it (len = 0: nothing to do).
template <int B, int HK, bool RESUME>
__device__ __forceinline__ void pg_expand(const PgArgs &a, uint32_t start, uint32_t len, int32_t u, uint32_t gu,
                                          uint32_t Fb, ExpandCounters &C, PgPush<B, RESUME> &push)
{
    constexpr int U = kPgUnroll;
    const uint32_t sub = threadIdx.x % kPgLanes;
    for (uint32_t j = 0; __any(j < len); j += kPgLanes * U) {
        int32_t c[U], dv[U];
        uint32_t wt[U];
#pragma unroll
        for (int r = 0; r < U; ++r) {
            const uint32_t k = j + r * kPgLanes + sub;
            c[r] = -1;
            wt[r] = 0;
            dv[r] = INT32_MAX;
            if (k < len) {
                c[r] = a.g.col[start + k];
                wt[r] = a.g.w[start + k];
                if (a.g.dver) dv[r] = a.g.dver[start + k];
                C.edges++;
            }
        }
#pragma unroll
        for (int r = 0; r < U; ++r)
            if (a.g.dver && dv[r] <= a.g.ver) c[r] = -1;  // deleted at or before this version
        relax_window<U, HK>(a.g, a.h, a.gp, a.t, c, wt, [&](int) { return gu; }, [&](int) { return u; }, Fb, C, push);
    }
}

template <int B, int HK, bool RESUME = false>
__global__ void __launch_bounds__(B) ga_piles_kernel(PgArgs a)
{
    static_assert(B >= 256, "flush uses four waves");
    __shared__ PgStage<B, RESUME> S;
    __shared__ int32_t s_flag;
    __shared__ Team s_team;
    constexpr uint32_t kPerWave = 64 / kPgLanes, kWaves = B / 64;
    const int lane = threadIdx.x;
    const uint32_t wl = lane & 63, sub = lane % kPgLanes;
    uint32_t *ctrl = a.ctrl;
    const uint32_t rank = grid_arrive(ctrl + PG_TEAM);
    uint32_t gen = ld_u32(ctrl + PG_BAR + 32);
    // ring positions and far entries as of the last barrier, the same in every workgroup
    uint32_t head = 0, tail = 1, fn = 0, F = DDP_INF_F, thr = a.thr0, delta = a.delta0, phase_n = 0, phase_it = 0;
    uint32_t low = 0xFFFFFFFFu;  // no live far entry is below this
    uint64_t *far = a.far0, *far2 = a.far1;
    uint32_t step = 0, err = 0, err_seen = 0;
    int32_t it = 0;
    bool timeout = false;
    const Team tm = grid_team(ctrl + PG_TEAM, rank, a.barrier_ticks, &s_team, timeout);
    if (tm.n == 0) {  // the team was complete before this workgroup started
        if (timeout && lane == 0) atomicOr(ctrl + GA_RES_ERR, (uint32_t)GA_ERR_BARRIER);
        return;
    }
    ExpandCounters C;
    uint32_t stale = 0;
    if constexpr (RESUME) {
        tail = 0;
        fn = ld_u32(a.live_n);
        low = ld_u32(a.live_min);
        F = (uint32_t)(ld_gp(a.gp + a.t) >> 32);
        if (ld_u32(a.live_ovf) || fn > a.fcap) {  // the open set did not fit its buffers
            fn = 0;
            if (a.rebuild) err_seen = PG_ERR_REBUILD;
            else err = GA_ERR_HEAP;
        }
    }
    if (lane == 0) {
        for (int pile = 0; pile < PgStage<B, RESUME>::kPiles; ++pile) S.n[pile] = 0;
        S.tmin = S.fmin = 0xFFFFFFFFu;
        S.err = 0;
    }
    __syncthreads();
    // a step: its counters' slot; the next step's (last read two barriers ago) is cleared meanwhile
    auto begin = [&]() {
        if (tm.me == 0 && lane < 6) {
            uint32_t *ns = ctrl + PG_SLOTS + ((step + 1) % 3) * PG_SLOT_WORDS;
            if (lane < 5) st_u32(ns + 32 * lane, lane == 2 || lane == 3 ? 0xFFFFFFFFu : 0u);
            else st_u32(ns + PG_ERR, 0u);
        }
        return ctrl + PG_SLOTS + (step % 3) * PG_SLOT_WORDS;
    };
    auto add_sat = [](uint32_t x, uint32_t y) { return x > 0xFFFFFFFFu - y ? 0xFFFFFFFFu : x + y; };
    while (!err) {
        if (err_seen & PG_ERR_REBUILD) {
            // entries were lost: the piles start again from every node whose
            // word is below F(t) (RESUME: finite; nodes that were expanded at
            // that value already are expanded again, which is harmless)
            err_seen = 0;
            if (tm.me == 0 && lane == 0) {
                if constexpr (RESUME) st_u32(a.dorm_n, 0u);
                C.rebuilds++;
            }
            uint32_t *slot = begin();
            if (!grid_sync(ctrl + PG_BAR, tm, gen, a.barrier_ticks, &s_flag)) {
                timeout = true;
                break;
            }
            ++step;
            slot = begin();
            head = tail;
            PgPush<B, RESUME> push{&S, &a, slot, tail, head, far, 0u, thr, F};
            const uint32_t stride = tm.n * B, trips = ((uint32_t)a.N + stride - 1) / stride;
            for (uint32_t r = 0; r < trips; ++r) {
                const uint32_t v = r * stride + tm.me * B + lane;
                uint64_t key[1] = {0};
                bool live[1] = {false};
                if (v < (uint32_t)a.N && v != (uint32_t)a.t) {
                    const uint32_t f = (uint32_t)(ld_gp(a.gp + v) >> 32);
                    live[0] = f != DDP_INF_F;
                    key[0] = (uint64_t)f << 32 | v;
                }
                push.template all<1>(live, key);
            }
            push.flush();
            if (!grid_sync(ctrl + PG_BAR, tm, gen, a.barrier_ticks, &s_flag)) {
                timeout = true;
                break;
            }
            ++step;
            tail += ld_u32(slot + PG_NEAR);
            fn = ld_u32(slot + PG_FAR);
            low = ld_u32(slot + PG_FMIN);
            err_seen = ld_u32(slot + PG_ERR);
            err = err_seen & ~PG_ERR_REBUILD;
            continue;
        }
        const uint32_t avail = tail - head;
        if (avail == 0 && (fn == 0 || low >= F)) {  // nothing open can improve t
            if constexpr (RESUME) {
                // What is left of the far pile joins the dormant pile below.  If
                // they do not fit together (stale entries count too), a rebuild
                // leaves every node in one of them once.
                if (a.rebuild && (uint64_t)ld_u32(a.dorm_n) + fn > a.dcap) {
                    if (!grid_sync(ctrl + PG_BAR, tm, gen, a.barrier_ticks, &s_flag)) {
                        timeout = true;
                        break;
                    }  // everybody has read the count
                    err_seen |= PG_ERR_REBUILD;
                    continue;
                }
            }
            break;
        }
        // The far pile is split when the near ring is empty, or when all but
        // stragglers of a window that has fed its K entries are done and the
        // next window adjoins it (entries further out would run ahead of f
        // order): the stragglers' round and the split then share a barrier.
        const bool split = fn > 0 && (avail == 0 || (avail < kPgThin && phase_n >= a.grow && low < add_sat(thr, delta)));
        if (split) {
            if (avail == 0) {
                if (it > 0) {
                    if (phase_n < a.grow || phase_n < kPgFeed * phase_it) delta = add_sat(delta, delta);
                    else if (phase_n > 8 * a.grow && phase_n > 8 * kPgFeed * phase_it && delta > 1) delta >>= 1;
                }
                phase_n = 0;
                phase_it = 0;
            }
            const uint32_t nt = add_sat(low, delta);
            thr = nt > thr ? nt : thr;
            if (tm.me == 0 && lane == 0) C.refills++;
        }
        if (avail && it >= a.maxit) {
            err |= GA_ERR_ITERS;
            break;
        }
        if (avail) {
            ++it;
            ++phase_it;
        }
        const uint32_t n = avail < kPgRound ? avail : kPgRound;
        phase_n += n;
        // ---- step 1: the round's entries, hub rows cut into segments, and the split
        uint32_t *slot = begin();
        {
            PgPush<B, RESUME> push{&S, &a, slot, tail, head, split ? far2 : far, split ? 0u : fn, thr, F};
            const uint32_t chunks = (n + kPerWave - 1) / kPerWave;
            for (uint32_t ch = (lane >> 6) * tm.n + tm.me; ch < chunks; ch += kWaves * tm.n) {
                const uint32_t i = ch * kPerWave + wl / kPgLanes;
                int32_t u = -1;
                uint32_t gu = 0, start = 0, deg = 0;
                uint64_t link = ~0ull;  // head of the node's list of inserted edges
                bool dz[1] = {false};   // current, but hopeless now
                uint64_t dkey[1] = {0};
                if (i < n) {
                    const uint64_t key = ld_gp(a.near + ((head + i) & a.nmask));
                    const uint32_t f = (uint32_t)(key >> 32);
                    const int32_t node = (int32_t)(uint32_t)key;
                    // the node's word, row and heuristic input in one round trip
                    const uint64_t word = ld_gp(a.gp + node);
                    const int32_t rb = a.g.off[node], re = a.g.off[node + 1];
                    const int32_t hn = heur_eval<HK>(a.h, node);
                    if (a.g.lhead && sub == 0) link = ld_gp(a.g.lhead + node);
                    dz[0] = RESUME && f >= F && (uint32_t)(word >> 32) == f && node != a.t && sub == 0;
                    dkey[0] = key;
                    if (f < F && (uint32_t)(word >> 32) == f) {
                        u = node;
                        gu = f - (uint32_t)hn;
                        start = (uint32_t)rb;
                        deg = (uint32_t)(re - rb);
                        if (sub == 0) C.expanded++;
                    } else if (sub == 0) {
                        ++stale;
                    }
                }
                if constexpr (RESUME)
                    if (__any(dz[0])) push.template all<1>(dz, dkey);
                if (__any(deg > (uint32_t)kPgSeg)) {
                    uint32_t at = 0;
                    const uint32_t parts = (deg + kPgSeg - 1) / kPgSeg;
                    if (deg > (uint32_t)kPgSeg && sub == 0) at = add_u32(slot + PG_HUBS, parts);
                    at = __shfl(at, wl - sub, 64);
                    if (deg > (uint32_t)kPgSeg) {
                        // (a row the list has no room for stays with its group, its places empty)
                        const bool fits = at + parts <= a.hubcap;
                        for (uint32_t k = sub; k < parts && at + k < a.hubcap; k += kPgLanes) {
                            const uint32_t o = k * kPgSeg, len = deg - o < (uint32_t)kPgSeg ? deg - o : kPgSeg;
                            st_u64(a.hubs + 2 * (uint64_t)(at + k), (uint64_t)(fits ? len : 0) << 32 | (start + o));
                            st_u64(a.hubs + 2 * (uint64_t)(at + k) + 1, (uint64_t)gu << 32 | (uint32_t)u);
                        }
                        if (fits) deg = 0;
                    }
                }
                pg_expand<B, HK>(a, start, deg, u, gu, RESUME ? 0xFFFFFFFFu : F, C, push);
                if (a.g.lhead) {
                    // Versioned inserts: the group's first lane walks the node's
                    // list, oldest first, up to the first entry newer than this
                    // version (links carry the inserting version).
                    if (u < 0) link = ~0ull;
                    for (;;) {
                        bool active = false;
                        int32_t x = -1;
                        while ((uint32_t)link <= (uint32_t)a.g.ver) {
                            x = (int32_t)(link >> 32);
                            link = ld_gp(a.g.lnext + x);
                            if (a.g.ldel[x] > a.g.ver) {
                                active = true;
                                break;
                            }
                        }
                        if (!__any(active)) break;
                        bool has[1] = {false};
                        uint64_t key[1] = {0};
                        if (active) {
                            C.edges++;
                            const int32_t cn = a.g.lv[x];
                            const int32_t hcn = heur_eval<HK>(a.h, cn);
                            if (HK != DDP_H_ARRAY || hcn >= 0) {
                                const uint32_t cand = gu + a.g.lw[x] + (uint32_t)hcn;
                                uint64_t prev;
                                if (relax_gp(a.gp, cn, cand, (uint32_t)u, &prev)) {
                                    C.improved++;
                                    if (cn == a.t) {
                                        push.target(cand);
                                    } else {
                                        has[0] = true;
                                        key[0] = (uint64_t)cand << 32 | (uint32_t)cn;
                                    }
                                }
                            }
                        }
                        push.template all<1>(has, key);
                    }
                }
            }
            if (split) {
                const uint32_t stride = tm.n * B, trips = (fn + stride - 1) / stride;
                for (uint32_t r = 0; r < trips; ++r) {  // uniform: the appends are wave-wide
                    const uint64_t i = (uint64_t)r * stride + (uint64_t)tm.me * B + lane;
                    uint64_t key[1] = {0};
                    bool live[1] = {false};
                    if (i < fn) {
                        key[0] = ld_gp(far + i);
                        const uint32_t f = (uint32_t)(key[0] >> 32);
                        live[0] = (RESUME ? (int32_t)(uint32_t)key[0] != a.t : f < F) &&
                                  (uint32_t)(ld_gp(a.gp + (uint32_t)key[0]) >> 32) == f;
                        C.scanned++;
                    }
                    push.template all<1>(live, key);
                }
            }
            push.flush();
        }
        if (!grid_sync(ctrl + PG_BAR, tm, gen, a.barrier_ticks, &s_flag)) {
            timeout = true;
            break;
        }
        ++step;
        const uint32_t hubs0 = ld_u32(slot + PG_HUBS), hubs = hubs0 < a.hubcap ? hubs0 : a.hubcap;
        {
            const uint32_t tm = ld_u32(slot + PG_TMIN);
            F = tm < F ? tm : F;
            head += n;
            tail += ld_u32(slot + PG_NEAR);
            fn = (split ? 0 : fn) + ld_u32(slot + PG_FAR);
            const uint32_t fm = ld_u32(slot + PG_FMIN);
            low = !split && low < fm ? low : fm;
            err_seen |= ld_u32(slot + PG_ERR);
            err = err_seen & ~PG_ERR_REBUILD;
        }
        if (split) {
            uint64_t *tmp = far;
            far = far2;
            far2 = tmp;
        }
        if (hubs && !err) {
            // ---- step 2: the segments of long rows
            slot = begin();
            PgPush<B, RESUME> push{&S, &a, slot, tail, head, far, fn, thr, F};
            const uint32_t chunks = (hubs + kPerWave - 1) / kPerWave;
            for (uint32_t ch = (lane >> 6) * tm.n + tm.me; ch < chunks; ch += kWaves * tm.n) {
                const uint32_t i = ch * kPerWave + wl / kPgLanes;
                uint64_t row = 0, from = 0;
                if (i < hubs) {
                    row = ld_gp(a.hubs + 2 * (uint64_t)i);
                    from = ld_gp(a.hubs + 2 * (uint64_t)i + 1);
                }
                pg_expand<B, HK>(a, (uint32_t)row, (uint32_t)(row >> 32), (int32_t)(uint32_t)from,
                                 (uint32_t)(from >> 32), RESUME ? 0xFFFFFFFFu : F, C, push);
            }
            push.flush();
            if (!grid_sync(ctrl + PG_BAR, tm, gen, a.barrier_ticks, &s_flag)) {
                timeout = true;
                break;
            }
            ++step;
            const uint32_t tm = ld_u32(slot + PG_TMIN);
            F = tm < F ? tm : F;
            const uint32_t fm = ld_u32(slot + PG_FMIN);
            low = low < fm ? low : fm;
            tail += ld_u32(slot + PG_NEAR);
            fn += ld_u32(slot + PG_FAR);
            err_seen |= ld_u32(slot + PG_ERR);
            err = err_seen & ~PG_ERR_REBUILD;
        }
    }
    if constexpr (RESUME) {
        // what is left of the far pile cannot beat F(t): dormant.  Nobody
        // appends any more, so every workgroup reads the same count.
        const uint32_t dn = ld_u32(a.dorm_n);
        if ((uint64_t)dn + fn > a.dcap) err |= GA_ERR_HEAP;
        else
            for (uint32_t i = tm.me * B + lane; i < fn; i += tm.n * B) st_u64(a.dorm + dn + i, ld_gp(far + i));
        if (tm.me == 0 && lane == 0) ctrl[GA_RES_PLEN] = dn + fn;
    }
    if (timeout && lane == 0) atomicOr(ctrl + GA_RES_ERR, (uint32_t)GA_ERR_BARRIER);
    if (tm.me == 0 && lane == 0) {
        if (err) atomicOr(ctrl + GA_RES_ERR, err);
        ctrl[GA_RES_IT] = (uint32_t)it;
        ctrl[GA_RES_F] = F;
    }
    const uint64_t v0 = wave_sum_u64(C.expanded), v1 = wave_sum_u64(C.edges), v2 = wave_sum_u64(C.improved),
                   v3 = wave_sum_u64(stale), v4 = wave_sum_u64(C.rebuilds), v5 = wave_sum_u64(C.refills),
                   v6 = wave_sum_u64(C.scanned);
    if (wl == 0) {
        atomicAdd(a.stats + 0, (unsigned long long)v0);
        atomicAdd(a.stats + 1, (unsigned long long)v1);
        atomicAdd(a.stats + 2, (unsigned long long)v2);
        atomicAdd(a.stats + 3, (unsigned long long)v3);
        if (v4) atomicAdd(a.stats + 4, (unsigned long long)v4);
        if (v5) atomicAdd(a.stats + 5, (unsigned long long)v5);
        if (v6) atomicAdd(a.stats + 6, (unsigned long long)v6);
    }
}
