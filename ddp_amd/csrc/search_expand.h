// Block-cooperative expansion of the nodes popped in one GA* iteration.
//
// Each lane of the block brings at most one popped node u (its queue's pop).
// Out-degrees are prefix-summed across the block and the union of all rows is
// cut into one range of consecutive edges per wave, so lanes read consecutive
// CSR entries and a long row is split across the whole block instead of
// serialising one lane (the reference gives each thread its own row:
// GA_star/GA_v2.cu:109-167).  A wave takes its range R windows of 64 edges at
// a time and issues their loads stage by stage (row entries, then heuristic
// inputs and (f, parent) words), so R independent memory round trips overlap.
//
// Edges that beat their node's word are few (5% on R-MAT, a fifth on a road
// map), so a wave collects them in LDS and relaxes and queues 64 (128 up to 512 lanes) at a time.
// Not for the lane-owned heaps: their pushes have to stay spread over the
// lanes (collected, the C4 batch overflowed heaps of 2,048 entries, and with
// the lanes taking turns it took 96-117 ms instead of 79).
//
// What a wave issues bounds a round, not what it waits for: with every stage
// run for all R windows and the rows located by a binary search per edge (or by
// owner hints in small rounds), a 1,024-lane workgroup spent 10.1 us on 4,096
// edges in a batch of 256 queries on R-MAT (scale 20; a query 105 ms on
// average), now 7.1 us (74 ms); the C4 batch went from 19.3 to 16.1 ms.
#pragma once

#include "device_common.h"

// Edges handled per lane and trip (memory requests a lane keeps in flight
// per stage).  At 1,024 lanes two, three, four and six took 80, 78, 73 and 73
// ms a query on R-MAT (scale 20) and 16.1, 16.2, 16.2 and 16.7 ms for C4: three
// with the Euclidean heuristic, whose kernels run out of registers with four
// (20 bytes of scratch in the batch kernel).  At 512 lanes two: four take R-MAT
// bursts on a server 7% further, but the kernels past the 128 registers that let
// two workgroups share a CU.
template <int B, int HK = DDP_H_ZERO>
constexpr int expand_unroll()
{
    return B == 512 ? 2 : B == 1024 && HK == DDP_H_EUCLID ? 3 : 4;
}

// Collected edges a lane relaxes at once (atomics it keeps in flight).  Where most
// edges improve (a random graph with an h array) a narrow workgroup waits for
// one atomic round trip per 64: a search of 600,000 nodes took 36.9, 18.2, 10.9 and
// 8.2 ms with 64, 128, 256 and 512 lanes at one a lane, 32.5, 16.3, 9.9 and 7.7 at two
// (31.3, 15.7, 9.8 and - at four, which takes a map's batch from 4.1 to 4.3 ms).  The
// 1,024-lane kernels have no registers for a second one.
template <int B>
constexpr int relax_unroll()
{
    return B <= 512 ? 2 : 1;
}

// Rows of a round and its collected edges (expand_rows; COLLECT, else none).
// Only rows that have edges are listed, so incl ascends strictly.
template <int B, bool COLLECT>
struct RowsLds {
    static constexpr int CAP = COLLECT ? 64 * (expand_unroll<B>() + relax_unroll<B>()) : 1;  // collected edges of a wave
    int32_t incl[B];        // inclusive prefix of degrees
    int32_t rowb[B];        // row start - edges before the row
    uint32_t gu[B];         // g(u) = f(u) - h(u), unsigned as GA_v2.cu:137
    int32_t node[B];
    int2 tmp[B / 64];       // edges and rows of each wave
    int32_t split;          // rows of the lanes below n0 (list_rows)
    uint64_t key[B / 64 * CAP];  // candidate f << 32 | node
    uint16_t row[B / 64 * CAP];
};

// What expanding u needs besides u itself: its row and g(u).
struct RowSpan {
    int32_t b = 0, deg = 0;
    uint32_t gu = 0;
};

template <int HK>
__device__ __forceinline__ RowSpan row_span(const GraphView &G, const HeurView &H, int32_t u, uint32_t fu)
{
    RowSpan r;
    if (u >= 0) {
        r.gu = fu - (uint32_t)heur_eval<HK>(H, u);
        r.b = G.off[u];
        r.deg = G.off[u + 1] - r.b;
    }
    return r;
}

// Per-lane statistics, 32-bit to spare registers.  Kernels add them to the
// 64-bit device totals at exit, and slot kernels also whenever a wave's
// edge count passes 2^30 (no counter of theirs grows faster).
struct ExpandCounters {
    uint32_t expanded = 0, edges = 0, improved = 0;
    // grid searches (slots count these in LDS, RefillCounts):
    uint32_t rebuilds = 0;  // piles rebuilt after an overflow (lane 0 counts)
    uint32_t refills = 0;   // splits of the far pile (lane 0 counts)
    uint32_t scanned = 0;   // far-pile entries read by them
};

// A round's rows: edges and rows in all, and (in every 16 lanes) up to and with
// each wave.
struct RoundRows {
    int32_t total, nrows, we_sum, wr_sum;
};

// Lists the rows that the block's lanes bring (deg edges from row start b, of
// node u with g(u) = gu).  Every lane of the block calls it; it begins with
// L free and ends with a barrier.  L.split: the rows of lanes below n0.
template <int B, bool COLLECT>
__device__ __forceinline__ RoundRows list_rows(RowsLds<B, COLLECT> &L, int32_t deg, int32_t b, uint32_t gu, int32_t u,
                                               int32_t n0 = -1)
{
    constexpr int W = B / 64;
    const int lane = threadIdx.x, wl = lane & 63;
    const int wid = __builtin_amdgcn_readfirstlane(lane >> 6);
    // edges and non-empty rows before this lane's row: within the wave, then
    // over the waves, whose sums every 16 lanes scan
    const int32_t x = wave_incl_scan(deg);
    const uint64_t full = __ballot(deg > 0);
    if (wl == 63) L.tmp[wid] = make_int2(x, (int32_t)__popcll(full));
    __syncthreads();
    int2 ws = make_int2(0, 0);
    if ((wl & 15) < W) ws = L.tmp[wl & 15];
    RoundRows rr;
    rr.we_sum = row16_incl_scan(ws.x);
    rr.wr_sum = row16_incl_scan(ws.y);
    rr.total = __builtin_amdgcn_readlane(rr.we_sum, 15);
    rr.nrows = __builtin_amdgcn_readlane(rr.wr_sum, 15);
    const int32_t i = (wid ? __builtin_amdgcn_readlane(rr.wr_sum, wid - 1) : 0) + (int32_t)lane_rank(full);
    if (deg > 0) {
        const int32_t end = (wid ? __builtin_amdgcn_readlane(rr.we_sum, wid - 1) : 0) + x;
        L.incl[i] = end;
        L.rowb[i] = b - (end - deg);
        L.gu[i] = gu;
        L.node[i] = u;
    }
    if (lane == n0) L.split = i;
    __syncthreads();
    return rr;
}

// The row of edge e < total.  Every lane of the wave calls it.
template <int B, bool COLLECT>
__device__ __forceinline__ int32_t first_row(const RowsLds<B, COLLECT> &L, const RoundRows &rr, int32_t e)
{
    const int wl = threadIdx.x & 63;
    const int g = (int)__popcll(__ballot(wl < B / 64 && rr.we_sum <= e));  // waves whose rows all end before
    const int32_t at = (g ? __builtin_amdgcn_readlane(rr.wr_sum, g - 1) : 0) + wl;
    return at - wl + (int32_t)__popcll(__ballot(at < rr.nrows && L.incl[at < rr.nrows ? at : 0] <= e));
}

// Rows of 64 consecutive edges, found by a wave at once: lane i reads the end
// of row row + i and marks the lane of the edge after it; an edge's row is row
// plus the marks up to it.  row: the row of edge e0, moved on to that of
// e0 + 64.  Every lane of the wave calls it, with e0 below the last row's end.
template <int B, bool COLLECT>
__device__ __forceinline__ int32_t wave_rows(const RowsLds<B, COLLECT> &L, int32_t nrows, int32_t e0, int32_t &row)
{
    const int32_t wl = (int32_t)(threadIdx.x & 63), at = row + wl;
    const int32_t p = at < nrows ? L.incl[at] - e0 : INT32_MAX;  // >= 1: row holds e0
    const int32_t r0 = row;
    const int32_t p0 = __builtin_amdgcn_readfirstlane(p);
    if (p0 >= 64) {  // one row holds the window
        row += p0 == 64 ? 1 : 0;
        return r0;
    }
    row += (int32_t)__popcll(__ballot(p <= 64));
    // lane 0, which no mark is for, takes what the other lanes push
    const int32_t mark = __builtin_amdgcn_ds_permute((p < 64 ? p : 0) << 2, p < 64 ? 1 : 0);
    const uint64_t m = __ballot(wl != 0 && mark != 0);
    return r0 + (int32_t)lane_rank(m) + (int32_t)(m >> wl & 1);
}

// Relaxes Q candidates per lane (key: f << 32 | node, of a node at which it can
// improve the word) and hands the improvements to the push policy.  Every
// lane of the wave calls it.
template <int Q, class Push>
__device__ __forceinline__ void relax_collected(const GraphView &G, uint64_t *gp, int32_t t, const bool (&have)[Q],
                                                const uint64_t (&key)[Q], const int32_t (&par)[Q], ExpandCounters &C,
                                                Push &push)
{
    int32_t c[Q];
    bool ok[Q], first[Q], has[Q];
    uint64_t prev[Q];
    if (G.relax_min != 0) {  // uniform
        // one atomicMin: the smallest (f, parent) of the round wins with no
        // retry round trips
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (have[q])
                prev[q] = (uint64_t)atomicMin((unsigned long long *)(gp + (uint32_t)key[q]),
                                              (key[q] & 0xFFFFFFFF00000000ull) | (uint32_t)par[q]);
#pragma unroll
        for (int q = 0; q < Q; ++q) ok[q] = have[q] && (uint32_t)(prev[q] >> 32) > (uint32_t)(key[q] >> 32);
    } else {
#pragma unroll
        for (int q = 0; q < Q; ++q)
            ok[q] = have[q] &&
                    relax_gp(gp, (int32_t)(uint32_t)key[q], (uint32_t)(key[q] >> 32), (uint32_t)par[q], &prev[q]);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        c[q] = (int32_t)(uint32_t)key[q];
        if (ok[q]) {
            C.improved++;
            if (c[q] == t) push.target((uint32_t)(key[q] >> 32));
        }
        first[q] = ok[q] && (uint32_t)(prev[q] >> 32) == DDP_INF_F;
        has[q] = ok[q] && c[q] != t;
    }
    push.template touch_all<Q>(first, c);
    push.template all<Q>(has, key);
}

// Relaxes R edges per lane (grid engine, lane heaps): edge r leads to c[r] (< 0:
// none) with weight wt[r] from the node par(r), whose g is gu(r).  Loads are
// issued stage by stage (heuristic inputs and (f, parent) words, then one
// atomic per improving edge), and improvements go to the push policy.  Fb
// as in expand_rows.
template <int R, int HK, class GuOf, class ParOf, class Push>
__device__ __forceinline__ void relax_window(const GraphView &G, const HeurView &H, uint64_t *gp, int32_t t,
                                             int32_t (&c)[R], const uint32_t (&wt)[R], GuOf gu_of, ParOf par_of,
                                             uint32_t Fb, ExpandCounters &C, Push &push)
{
    // stage 2: heuristic inputs and the current (f, parent) words, all
    // loads issued before the first heuristic is computed.  hin, cur and
    // got below are only written and read by lanes whose edge takes part:
    // giving the others a value would make the compiler merge the two and
    // wait for each load (or CAS) before issuing the next.
    HeurIn hin[R];
    uint64_t cur[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if constexpr (HK == DDP_H_ZERO || HK == DDP_H_MANHATTAN)
            if (c[r] >= 0 && gu_of(r) + wt[r] + (uint32_t)heur_from<HK>(H, c[r], HeurIn{0, 0}) >= Fb)
                c[r] = -1;  // cannot beat the bound: no word read
        if (c[r] >= 0) {  // negative id = deleted edge
            hin[r] = heur_load<HK>(H, c[r]);
            cur[r] = ld_gp(gp + c[r]);
        }
    }
    int32_t hc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) hc[r] = c[r] >= 0 ? heur_from<HK>(H, c[r], hin[r]) : 0;
    // stage 3: one CAS attempt per improving edge, all issued together
    uint64_t want[R], got[R];
    bool tried[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        tried[r] = false;
        want[r] = 0;
        if (c[r] >= 0 && (HK != DDP_H_ARRAY || hc[r] >= 0)) {  // h = -1: cannot reach t
            const uint32_t cand = gu_of(r) + wt[r] + (uint32_t)hc[r];
            want[r] = ((uint64_t)cand << 32) | (uint32_t)par_of(r);
            tried[r] = (uint32_t)(cur[r] >> 32) > cand;
        }
    }
    // Every load above has returned by now (the comparisons used them);
    // saying so keeps the compiler from waiting again before each CAS.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    const bool by_min = G.relax_min != 0;  // uniform
    if (by_min) {
        // one atomicMin per improving edge: the smallest (f, parent) of
        // the round wins with no retry round trips
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (tried[r]) got[r] = (uint64_t)atomicMin((unsigned long long *)(gp + c[r]),
                                                       (unsigned long long)want[r]);
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (tried[r])
                got[r] = (uint64_t)atomicCAS((unsigned long long *)(gp + c[r]), (unsigned long long)cur[r],
                                             (unsigned long long)want[r]);
    }
    // stage 4: settle contended CASes, then hand improvements to the push policy
    bool has[R], first[R];
    uint64_t key[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        has[r] = false;
        first[r] = false;
        key[r] = 0;
        if (tried[r]) {
            const uint32_t cand = (uint32_t)(want[r] >> 32);
            bool ok = by_min ? (uint32_t)(got[r] >> 32) > cand : got[r] == cur[r];
            uint64_t prev = by_min ? got[r] : cur[r];
            if (!ok && !by_min) {
                uint64_t now = got[r];
                while ((uint32_t)(now >> 32) > cand) {
                    const uint64_t old = atomicCAS((unsigned long long *)(gp + c[r]), (unsigned long long)now,
                                                   (unsigned long long)want[r]);
                    if (old == now) {
                        ok = true;
                        prev = now;
                        break;
                    }
                    now = old;
                }
            }
            if (ok) {
                C.improved++;
                first[r] = (uint32_t)(prev >> 32) == DDP_INF_F;
                if (c[r] == t) {
                    push.target(cand);
                } else {
                    has[r] = true;
                    key[r] = ((uint64_t)cand << 32) | (uint32_t)c[r];
                }
            }
        }
    }
    push.template touch_all<R>(first, c);
    push.template all<R>(has, key);
}

// Push policy interface (kCollect: edges may reach it from any lane of their wave;
// members marked wave-wide: every lane of the wave calls them):
//   void target(uint32_t f)                    -- t improved to f (t is never queued)
//   void touch(int32_t c, uint64_t prev)       -- c's word was prev before the update
//   void operator()(bool has, uint64_t key)    -- wave-wide
//   void touch_all<R>(first[R], c[R])          -- wave-wide: touch() of R edges
//                                                 whose previous f was infinite
//   void all<R>(has[R], key[R])                -- wave-wide: operator() of R edges
// Each lane brings a node u (or -1) and its row span (row_span, or the same
// values loaded earlier by the caller).
//
// Without FINAL_SYNC the function returns without its closing barrier; the
// caller must pass a barrier before the next expand_rows (or before reading
// what the pushes wrote).
//
// Fb: an upper bound the caller no longer needs to beat (the target's f when
// it only wants the target's cost).  Where the heuristic needs no load (zero,
// Manhattan) an edge whose candidate f is already >= Fb is skipped before its
// (f, parent) word is read: it cannot lead to a cheaper path to t, and the
// word's random 8-byte read costs a whole cache line.  Callers that keep
// searching for a later, larger bound (a resumed DA* search) pass UINT32_MAX.
//
// DIRECT_OK (heuristics without loads, atomicMin relaxation): in a round of at
// most one edge per lane no word is read first; every edge that can still beat
// Fb issues its atomicMin, whose returned word says whether it improved.  A
// small round is a chain of dependent round trips, and this takes one out of
// it; a large round keeps the read, which spares the atomics of the many edges
// that cannot improve.
template <int B, int HK, class Push, bool FINAL_SYNC = true, bool DIRECT_OK = false>
__device__ __forceinline__ void expand_rows(const GraphView &G, const HeurView &H, uint64_t *gp, int32_t t,
                                            int32_t u, const RowSpan &rs, RowsLds<B, Push::kCollect> &L,
                                            ExpandCounters &C, Push &push, uint32_t Fb = 0xFFFFFFFFu)
{
    constexpr int R = expand_unroll<B, HK>(), Q = relax_unroll<B>(), W = B / 64;
    constexpr bool kNoLoad = HK == DDP_H_ZERO || HK == DDP_H_MANHATTAN;
    const int lane = threadIdx.x, wl = lane & 63;
    const int wid = __builtin_amdgcn_readfirstlane(lane >> 6);
    if (u >= 0) C.expanded++;
    const RoundRows rr = list_rows<B>(L, u >= 0 ? rs.deg : 0, rs.b, rs.gu, u);
    const int32_t total = rr.total, nrows = rr.nrows;
    // This wave's windows of 64 edges: consecutive ones, dealt out evenly, or
    // (lane heaps) every W-th, which mixes the rows over the heaps: with
    // consecutive ones the C4 batch's heaps kept each other's offspring and
    // expanded 20% more nodes.
    constexpr int STEP = Push::kCollect ? 64 : B;
    const int32_t nw = (int32_t)(((uint32_t)total + 63) / 64);
    int32_t we = Push::kCollect ? nw * wid / W * 64 : wid * 64, wend = total;
    if constexpr (Push::kCollect) {
        const int32_t we1 = nw * (wid + 1) / W * 64;
        wend = we1 < total ? we1 : total;
    }
    const bool direct = DIRECT_OK && kNoLoad && G.relax_min != 0 && total <= B;
    if (we < wend) {
        int32_t row = first_row(L, rr, we);
        uint64_t *const ck = L.key + wid * RowsLds<B, Push::kCollect>::CAP;
        uint16_t *const cr = L.row + wid * RowsLds<B, Push::kCollect>::CAP;
        int32_t cn = 0;  // collected edges
        while (we < wend) {
            int32_t c[R], jj[R], pos[R];
            uint32_t wt[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                pos[r] = -1;
                jj[r] = 0;
                const int32_t e0 = we + r * STEP;
                if (e0 >= wend) continue;
                if (STEP != 64) row = first_row(L, rr, e0);
                jj[r] = wave_rows(L, nrows, e0, row);
                if (e0 + wl < wend) {
                    pos[r] = L.rowb[jj[r]] + e0 + wl;
                    C.edges++;
                }
            }
            int32_t dv[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                c[r] = -1;
                wt[r] = 0;
                dv[r] = INT32_MAX;
                if (pos[r] >= 0) {
                    c[r] = G.col[pos[r]];
                    wt[r] = G.w[pos[r]];
                    if (G.dver) dv[r] = G.dver[pos[r]];
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (G.dver && dv[r] <= G.ver) c[r] = -1;  // deleted at or before this version
            if constexpr (!Push::kCollect) {
                we += STEP * R;
                relax_window<R, HK>(G, H, gp, t, c, wt, [&](int r) { return L.gu[jj[r]]; },
                                    [&](int r) { return L.node[jj[r]]; }, Fb, C, push);
                continue;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) wt[r] += pos[r] >= 0 ? L.gu[jj[r]] : 0;  // g of the edge's end
            // heuristic inputs and current (f, parent) words, all loads issued
            // before the first heuristic is computed.  hin and cur are only
            // written and read by lanes whose edge takes part: giving the
            // others a value would make the compiler merge the two and wait
            // for each load before issuing the next.
            HeurIn hin[R];
            uint64_t cur[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (kNoLoad) {
                    if (c[r] >= 0) {
                        wt[r] += (uint32_t)heur_from<HK>(H, c[r], HeurIn{0, 0});
                        if (wt[r] >= Fb) c[r] = -1;  // cannot beat the bound: no word read
                    }
                }
                if (c[r] >= 0) {  // negative id = deleted edge
                    if constexpr (!kNoLoad) hin[r] = heur_load<HK>(H, c[r]);
                    if (!direct) cur[r] = ld_gp(gp + c[r]);
                }
            }
            uint64_t key[R];
            bool tried[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                tried[r] = false;
                key[r] = 0;
                if (c[r] >= 0) {
                    const int32_t hc = kNoLoad ? 0 : heur_from<HK>(H, c[r], hin[r]);
                    if (HK != DDP_H_ARRAY || hc >= 0) {  // h = -1: cannot reach t
                        const uint32_t cand = wt[r] + (uint32_t)hc;
                        key[r] = ((uint64_t)cand << 32) | (uint32_t)c[r];
                        tried[r] = direct || (uint32_t)(cur[r] >> 32) > cand;
                    }
                }
            }
            we += STEP * R;
            if (total <= B) {  // at most one edge per lane: nothing to collect
                const bool one[1] = {tried[0]};
                const uint64_t key1[1] = {key[0]};
                const int32_t par1[1] = {tried[0] ? L.node[jj[0]] : 0};
                relax_collected<1>(G, gp, t, one, key1, par1, C, push);
                break;
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint64_t m = __ballot(tried[r]);
                if (tried[r]) {
                    const int32_t at = cn + (int32_t)lane_rank(m);
                    ck[at] = key[r];
                    cr[at] = (uint16_t)jj[r];
                }
                cn += (int32_t)__popcll(m);
            }
            while (cn >= 64 * Q || (cn > 0 && we >= wend)) {  // the last ones first, so the rest stays where it is
                const int32_t n = cn < 64 * Q ? cn : 64 * Q, at = cn - n + wl;
                bool have[Q];
                uint64_t k[Q];
                int32_t par[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    have[q] = 64 * q + wl < n;
                    k[q] = 0;
                    par[q] = 0;
                    if (have[q]) {
                        k[q] = ck[at + 64 * q];
                        par[q] = L.node[cr[at + 64 * q]];
                    }
                }
                relax_collected<Q>(G, gp, t, have, k, par, C, push);
                cn -= n;
            }
        }
    }
    if (G.lhead) {
        // Versioned inserts: each lane walks its own node's list, oldest
        // first, stopping at the first entry newer than this version (links
        // carry the inserting version, so newer entries are never read).
        const uint32_t gu = rs.gu;
        uint64_t link = u >= 0 ? __hip_atomic_load(G.lhead + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ~0ull;
        for (;;) {
            bool active = false, has = false;
            uint64_t key = 0;
            int32_t xe = -1;
            while ((uint32_t)link <= (uint32_t)G.ver) {
                xe = (int32_t)(link >> 32);
                link = __hip_atomic_load(G.lnext + xe, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (G.ldel[xe] > G.ver) {
                    active = true;
                    break;
                }
            }
            if (active) {
                C.edges++;
                const int32_t cn = G.lv[xe];
                const int32_t hcn = heur_eval<HK>(H, cn);
                if (HK != DDP_H_ARRAY || hcn >= 0) {
                    const uint32_t cand = gu + G.lw[xe] + (uint32_t)hcn;
                    uint64_t prev;
                    if (relax_gp(gp, cn, cand, (uint32_t)u, &prev)) {
                        C.improved++;
                        push.touch(cn, prev);
                        if (cn == t) {
                            push.target(cand);
                        } else {
                            has = true;
                            key = ((uint64_t)cand << 32) | (uint32_t)cn;
                        }
                    }
                }
            }
            push(has, key);
            if (!__syncthreads_or(active)) break;
        }
    }
    if constexpr (FINAL_SYNC) __syncthreads();
}

template <int B, int HK, bool DIRECT_OK = false, class Push>
__device__ __forceinline__ void expand_block(const GraphView &G, const HeurView &H, uint64_t *gp, int32_t t,
                                             int32_t u, uint32_t fu, RowsLds<B, Push::kCollect> &L,
                                             ExpandCounters &C, Push &push)
{
    expand_rows<B, HK, Push, true, DIRECT_OK>(G, H, gp, t, u, row_span<HK>(G, H, u, fu), L, C, push);
}
