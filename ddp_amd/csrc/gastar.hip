// Single-query GA*: planning, state and entry point.  Grid mode runs on piles over
// the whole GPU (grid_piles.h); the other modes keep the search in one workgroup
// (below): K lane heaps, piles (slot_search.h) or piles from both ends
// (bidi_search.h).
//
// Reference loop (GA_star/GA_v2.cu:488-559): per iteration the host launches
// extractMin, A_star_expand, keepHeapPQ, setNV (an O(N) flag scan), insertPQ,
// copies flags and all K queue sizes back, and runs checkMIN.  Here the whole
// loop is one kernel in every mode:
//   * an iteration expands its nodes cooperatively, and every improvement goes
//     into a packed (f << 32 | parent) word by one atomic -- no per-node locks;
//   * improved nodes are queued by the wave that improved them, with one counter
//     atomic per wave or workgroup, which replaces setNV's O(N) scan;
//   * termination is decided on the device: once no open entry can lead to
//     anything below F(t) (GA_v2.cu:277-289, 547-557).
// Stale entries (a node improved after it was queued) are skipped when they are
// taken; this replaces keepHeapPQ's in-place decrease-key repair.
#include <algorithm>
#include <chrono>
#include <cstring>

#include <type_traits>

#include "bidi_search.h"
#include "gastar.h"
#include "grid_piles.h"
#include "pile_sizes.h"

namespace {

enum : uint32_t {
    ERR_HEAP = GA_ERR_HEAP, ERR_ITERS = GA_ERR_ITERS, ERR_BARRIER = GA_ERR_BARRIER,
    ERR_PATH = 16
};

__global__ void fill_u64_kernel(uint64_t *p, int64_t n, uint64_t v)
{
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void unpack_parent_kernel(const uint64_t *gp, int32_t *par, int32_t N)
{
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        par[i] = (int32_t)(uint32_t)gp[i];
}

// Fresh search on piles: gp[s], s alone in the near ring, the control words.
__global__ void pg_seed_kernel(uint64_t *gp, uint64_t *near, uint32_t *ctrl, int32_t s, uint32_t hs)
{
    for (int k = threadIdx.x; k < PG_WORDS; k += blockDim.x) {
        const int w = k >= PG_SLOTS && k < PG_BAR ? (k - PG_SLOTS) % PG_SLOT_WORDS : -1;
        ctrl[k] = w == PG_TMIN || w == PG_FMIN ? 0xFFFFFFFFu : 0u;
    }
    if (threadIdx.x == 0) {
        gp[s] = ((uint64_t)hs << 32) | 0xFFFFFFFFull;
        near[0] = ((uint64_t)hs << 32) | (uint32_t)s;
    }
}

using PgFn = void (*)(PgArgs);

PgFn pick_pg(int hk)
{
    switch (hk) {
    case DDP_H_ZERO: return ga_piles_kernel<kPgBlock, DDP_H_ZERO>;
    case DDP_H_ARRAY: return ga_piles_kernel<kPgBlock, DDP_H_ARRAY>;
    case DDP_H_MANHATTAN: return ga_piles_kernel<kPgBlock, DDP_H_MANHATTAN>;
    default: return ga_piles_kernel<kPgBlock, DDP_H_EUCLID>;
    }
}

int32_t pg_blocks(const ddp_ctx *ctx, const GaGridPlan &P, int hk)
{
    return pg_workgroups(P.edges, hk == DDP_H_MANHATTAN || hk == DDP_H_EUCLID, ctx->prop.multiProcessorCount);
}

PgSizes ga_pg_sizes(const GaGridPlan &P, int32_t N) { return pg_sizes((uint64_t)P.K * P.cap, N); }

// Workgroup mode: all K <= 1024 queues live in one workgroup, one per lane,
// and an improved node goes to the queue of the lane that relaxed it.  An
// iteration then synchronises through LDS barriers only, where the grid
// mode pays a device-wide barrier and its atomics; searches whose frontier
// holds a few thousand nodes (or whose iteration count is set by a long
// path) are bound by that per-iteration latency, not by bandwidth.
struct WgArgs {
    GraphView g;
    GraphView gr;        // transposed rows (bidirectional mode)
    HeurView h;
    uint64_t *gp;        // N (bidirectional: 2N, forward then backward)
    uint64_t *home;      // heap spill (entry i of queue q at home[i*B + q]), or the piles (two sets: bidirectional)
    int32_t *touched;    // N: nodes whose word left INF (bidirectional: 2N)
    int32_t *path;       // bidirectional mode: the path s..t is walked on the device into path[0..path_cap)
    int32_t path_cap;
    uint32_t *ctrl;
    unsigned long long *stats;
    int32_t N, s, t, lcap, cap, maxit;
    uint32_t ncap, fcap, delta0;  // pile mode: near ring, far buffers, first window
    uint32_t lring;               // pile mode: entries of the LDS near ring (dynamic LDS)
};

enum { WM_HEAPS = 0, WM_PILES = 1, WM_BIDI = 2 };

// WM_HEAPS: lane heaps (slot_search); WM_PILES: near/far piles
// (slot_search_piles); WM_BIDI: piles from both ends (slot_search_bidi)
template <int B, int HK, int WM>
__global__ void __launch_bounds__(B) ga_wg_kernel(WgArgs a)
{
    extern __shared__ uint64_t s_heap[];  // lcap * B (heaps), near rings (piles)
    __shared__ std::conditional_t<WM == WM_BIDI, BidiLds<B>, SlotLds<B, WM == WM_PILES>> S;
    const int lane = threadIdx.x;
    const LaneHeap H{s_heap + lane, a.home + lane, B, a.lcap, (int64_t)B, a.cap};
    ExpandCounters C;
    uint32_t stale = 0;
    if (lane == 0) S.rc = RefillCounts{};
    if constexpr (WM == WM_BIDI) {
        const int32_t N = a.N;
        uint64_t *bh = a.home + (int64_t)a.cap * B;
        const PilePtrs PF{a.home, a.home + a.ncap, a.home + a.ncap + a.fcap, a.ncap, a.fcap, s_heap, a.lring / 2};
        const PilePtrs PB{bh, bh + a.ncap, bh + a.ncap + a.fcap, a.ncap, a.fcap, s_heap + a.lring / 2, a.lring / 2};
        const BidiSide D{{a.g.off, a.gr.off}, {a.g.col, a.gr.col}, {a.g.w, a.gr.w}, {a.gp, a.gp + N},
                         {a.touched, a.touched + N}, {PF, PB}};
        slot_search_bidi<B, HK>(D, a.h, a.g.relax_min != 0, N, a.s, a.t, a.maxit, a.delta0, S, C, stale);
        if (a.path) slot_path_bidi(D, N, a.s, a.t, a.path, a.path_cap, S);
        if (lane == 0) {
            const uint32_t e = S.err;
            a.ctrl[GA_RES_IT] = (uint32_t)S.iters;
            a.ctrl[GA_RES_F] = (uint32_t)(S.meet >> 32);
            a.ctrl[GA_RES_ERR] = ((e & QERR_HEAP) ? ERR_HEAP : 0u) | ((e & QERR_ITERS) ? ERR_ITERS : 0u) |
                                 ((e & QERR_PATH) ? ERR_PATH : 0u);
            a.ctrl[GA_RES_PLEN] = (uint32_t)(a.path ? S.plen : 0);
        }
    } else {
        if constexpr (WM == WM_PILES) {
            const PilePtrs P{a.home, a.home + a.ncap, a.home + a.ncap + a.fcap, a.ncap, a.fcap, s_heap, a.lring};
            slot_search_piles<B, HK, true>(a.g, a.h, a.gp, a.touched, P, a.N, a.s,
                                                                              a.t, a.maxit, a.delta0, S, C, stale);
        } else {
            slot_search<B, HK>(a.g, a.h, a.gp, a.touched, H, s_heap, a.N, a.s, a.t, a.maxit, S, C, stale);
        }
        if (lane == 0) {
            const uint32_t e = S.err;
            a.ctrl[GA_RES_IT] = (uint32_t)S.iters;
            a.ctrl[GA_RES_F] = S.F;
            a.ctrl[GA_RES_ERR] = ((e & QERR_HEAP) ? ERR_HEAP : 0u) | ((e & QERR_ITERS) ? ERR_ITERS : 0u);
        }
    }
    slot_flush_stats(a.stats, C, stale, S.rc);
}

using WgFn = void (*)(WgArgs);

template <int B, int WM>
WgFn pick_wg_b(int hk)
{
    switch (hk) {
    case DDP_H_ZERO: return ga_wg_kernel<B, DDP_H_ZERO, WM>;
    case DDP_H_ARRAY:
        if constexpr (WM == WM_BIDI) return nullptr;  // the potential needs h toward s as well as t
        else return ga_wg_kernel<B, DDP_H_ARRAY, WM>;
    case DDP_H_MANHATTAN: return ga_wg_kernel<B, DDP_H_MANHATTAN, WM>;
    default: return ga_wg_kernel<B, DDP_H_EUCLID, WM>;
    }
}

template <int WM>
WgFn pick_wg_p(int B, int hk)
{
    if constexpr (WM == WM_BIDI) {
        switch (B) {
        case 256: return pick_wg_b<256, WM>(hk);
        case 512: return pick_wg_b<512, WM>(hk);
        case 1024: return pick_wg_b<1024, WM>(hk);
        default: return nullptr;
        }
    }
    switch (B) {
    case 64: return pick_wg_b<64, WM>(hk);
    case 128: return pick_wg_b<128, WM>(hk);
    case 256: return pick_wg_b<256, WM>(hk);
    case 512: return pick_wg_b<512, WM>(hk);
    default: return pick_wg_b<1024, WM>(hk);
    }
}

WgFn pick_wg(int B, int hk, int wm)
{
    return wm == WM_BIDI ? pick_wg_p<WM_BIDI>(B, hk) : wm == WM_PILES ? pick_wg_p<WM_PILES>(B, hk)
                                                                       : pick_wg_p<WM_HEAPS>(B, hk);
}

}  // namespace

int ddp_ga_plan(ddp_ctx *ctx, const ddp_graph *g, const ddp_astar_opts_t *o, GaGridPlan *p, int64_t min_pcap,
                bool allow_wg)
{
    int32_t B = (o && o->block) ? o->block : 0;
    int32_t K = (o && o->K) ? o->K : 1024;
    DDP_CHECK(K >= 1, ctx, DDP_ERR_ARG, "K must be >= 1 (got %d)", K);
    const int32_t mode = (o && allow_wg) ? o->mode : DDP_ASTAR_GRID;
    DDP_CHECK(mode >= DDP_ASTAR_AUTO && mode <= DDP_ASTAR_BIDI, ctx, DDP_ERR_ARG, "unknown mode %d", mode);
    const bool one_wg = mode == DDP_ASTAR_WORKGROUP || mode == DDP_ASTAR_PILES || mode == DDP_ASTAR_BIDI;
    DDP_CHECK(!(one_wg && K > 1024), ctx, DDP_ERR_ARG, "one-workgroup modes hold at most 1024 lanes (K=%d)", K);
    if (one_wg) {
        const bool piles = mode == DDP_ASTAR_PILES || mode == DDP_ASTAR_BIDI;
        int32_t WB = mode == DDP_ASTAR_BIDI ? 256 : 64;  // two directions: half a block each
        while (WB < K) WB *= 2;
        DDP_CHECK(B == 0 || B == WB, ctx, DDP_ERR_ARG,
                  "one-workgroup mode runs K=%d on a block of %d lanes (got block %d)", K, WB, B);
        int32_t lcap = (o && o->lds_cap) ? o->lds_cap : std::max(1, std::min(32, 8192 / WB));
        if (piles) lcap = 0;
        DDP_CHECK((int64_t)lcap * WB * 8 <= 96 * 1024, ctx, DDP_ERR_ARG,
                  "lds_cap %d x block %d exceeds the LDS budget", lcap, WB);
        int64_t cap = (o && o->heap_cap) ? o->heap_cap : (2 * (int64_t)g->N + WB - 1) / WB + 256;
        if (piles && !(o && o->heap_cap))  // room for an exhaustive search: 3N entries
            cap = std::max<int64_t>(2048, (3 * (int64_t)g->N + WB - 1) / WB);
        cap = std::max<int64_t>(cap, std::max(lcap, 16));
        DDP_CHECK(cap < (1 << 30) && cap * WB < (1LL << 32), ctx, DDP_ERR_ARG, "heap_cap too large");
        const int32_t maxit =
            (o && o->max_iters) ? o->max_iters : (int32_t)std::min<int64_t>(4LL * g->N + 1024, 1 << 30);
        *p = GaGridPlan{WB, WB, 1, lcap, (int32_t)cap, 1024, maxit, true};
        if (piles) {
            const uint64_t total = (uint64_t)cap * WB;
            uint64_t nc = 1;
            while (nc * 2 <= total / 4) nc *= 2;
            p->piles = true;
            p->bidi = mode == DDP_ASTAR_BIDI;
            p->ncap = (uint32_t)nc;
            p->fcap = (uint32_t)std::min<uint64_t>((total - nc) / 2, 0xFFFFFFFFull);
            p->delta0 = std::max<uint32_t>(1, g->meanw);
        }
        return DDP_OK;
    }
    // Grid mode's workgroups have 1,024 lanes whatever B is (pg_workgroups): B, given
    // or by these steps, is what K is rounded up to and bounded by, as callers
    // that sized K for lane heaps know it.
    if (B == 0) B = K >= 65536 ? 1024 : K >= 4096 ? 256 : 64;
    DDP_CHECK(B == 64 || B == 256 || B == 1024, ctx, DDP_ERR_ARG,
              "block must be 64, 256 or 1024 (got %d)", B);
    K = ((K + B - 1) / B) * B;
    const int32_t nblocks = K / B;
    int32_t lcap = (o && o->lds_cap) ? o->lds_cap : std::max(1, std::min(32, 8192 / B));
    DDP_CHECK((int64_t)lcap * B * 8 <= 96 * 1024, ctx, DDP_ERR_ARG,
              "lds_cap %d x block %d exceeds the LDS budget", lcap, B);
    int64_t cap = (o && o->heap_cap) ? o->heap_cap : (2 * (int64_t)g->N + K - 1) / K + 256;
    cap = std::max<int64_t>(cap, lcap);
    DDP_CHECK(cap < (1 << 30), ctx, DDP_ERR_ARG, "heap_cap too large");
    // room for a DA* batch's pushes (and, with E close to 2^31, a refusal of its own)
    int64_t pcap = (int64_t)K * std::max(1, g->maxdeg) + K;
    pcap = std::min<int64_t>(pcap, (int64_t)g->E + 2 * (int64_t)K + 64);
    pcap = std::max<int64_t>(pcap, std::max<int64_t>(1024, min_pcap));
    DDP_CHECK(pcap < (1LL << 31), ctx, DDP_ERR_ARG, "push buffer too large");
    int32_t maxit = (o && o->max_iters) ? o->max_iters : (int32_t)std::min<int64_t>(4LL * g->N + 1024, 1 << 30);
    *p = GaGridPlan{K, B, nblocks, lcap, (int32_t)cap, (int32_t)pcap, maxit};
    p->pg = true;
    p->edges = g->E;
    p->hubcap = (uint32_t)((int64_t)g->E / kPgSeg + kPgRound + 64);
    p->delta0 = std::max<uint32_t>(1, g->meanw);
    // The bound on K is part of the interface, not a limit of the piles (which
    // need no LDS per queue): the lane heaps of K queues that the device could
    // hold at once, in workgroups of B lanes, 20 waves a CU at most.
    const size_t lds = (size_t)lcap * B * 8 + 48 * (size_t)B + 392;
    const int per_cu = (int)std::min<size_t>(ctx->prop.maxSharedMemoryPerMultiProcessor / lds, 20 * 64 / B);
    DDP_CHECK((int64_t)per_cu * ctx->prop.multiProcessorCount >= nblocks, ctx, DDP_ERR_ARG,
              "K=%d needs %d co-resident workgroups of %d lanes; the device holds %d", K, nblocks, B,
              per_cu * ctx->prop.multiProcessorCount);
    return DDP_OK;
}

int ddp_ga_alloc(ddp_ctx *ctx, const ddp_graph *g, const GaGridPlan &P, GaGridState *S)
{
    void *p;
    int rc;
    const size_t dirs = P.bidi ? 2 : 1;
    size_t queue = dirs * P.cap * P.K, push = 0;  // 8-byte entries
    if (P.pg) {
        queue = ga_pg_sizes(P, g->N).entries();
        push = 2 * (size_t)P.hubcap;
    }
    if ((rc = ddp_ws(ctx, WS_ASTAR_GP, dirs * g->N * 8, &p))) return rc;
    S->gp = (uint64_t *)p;
    if ((rc = ddp_ws(ctx, WS_ASTAR_HEAP, queue * 8, &p))) return rc;
    S->home = (uint64_t *)p;
    if ((rc = ddp_ws(ctx, WS_ASTAR_PBUF, push * 8 + 64, &p))) return rc;
    S->pbuf = (uint64_t *)p;
    if ((rc = ddp_ws(ctx, WS_ASTAR_CTRL, GA_CTRL_WORDS * 4 + 64, &p))) return rc;
    S->ctrl = (uint32_t *)p;
    S->stats = (unsigned long long *)((char *)p + GA_CTRL_WORDS * 4);
    S->touched = nullptr;
    if (P.wg) {
        if ((rc = ddp_ws(ctx, WS_ASTAR_TOUCH, dirs * g->N * 4, &p))) return rc;
        S->touched = (int32_t *)p;
    }
    S->owned = false;
    return DDP_OK;
}

int ddp_ga_alloc_owned(ddp_ctx *ctx, int32_t N, const GaGridPlan &P, GaGridState *S)
{
    *S = GaGridState{};
    S->owned = true;
    hipError_t e = hipSuccess;
    auto al = [&](void **p, size_t bytes) {
        if (e == hipSuccess) e = hipMalloc(p, std::max<size_t>(bytes, 64));
    };
    DDP_CHECK(P.pg, ctx, DDP_ERR_STATE, "GA*: not a grid plan");
    al((void **)&S->gp, (size_t)N * 8);
    al((void **)&S->home, ga_pg_sizes(P, N).entries() * 8);
    al((void **)&S->pbuf, 16 * (size_t)P.hubcap);
    al((void **)&S->ctrl, GA_CTRL_WORDS * 4 + 64);
    if (e != hipSuccess) {
        ddp_ga_free(S);
        return ddp_hip_err(ctx, e, "GA* state allocation", __FILE__, __LINE__);
    }
    S->stats = (unsigned long long *)((char *)S->ctrl + GA_CTRL_WORDS * 4);
    return DDP_OK;
}

void ddp_ga_free(GaGridState *S)
{
    if (!S->owned) return;
    void *ptrs[] = {S->gp, S->home, S->pbuf, S->ctrl};
    for (void *p : ptrs)
        if (p) hipFree(p);
    *S = GaGridState{};
}

int ddp_ga_reset(ddp_ctx *ctx, int32_t N, const GaGridPlan &P, const GaGridState &S)
{
    hipLaunchKernelGGL(fill_u64_kernel, dim3(1024), dim3(256), 0, ctx->stream, S.gp, (int64_t)N * (P.bidi ? 2 : 1),
                       (uint64_t)DDP_GP_INF);
    DDP_HIP(ctx, hipMemsetAsync(S.stats, 0, 64, ctx->stream));
    DDP_HIP(ctx, hipGetLastError());
    return DDP_OK;
}

int ddp_ga_stats(ddp_ctx *ctx, const GaGridState &S, unsigned long long out[4])
{
    DDP_HIP(ctx, hipMemcpyAsync(out, S.stats, 32, hipMemcpyDeviceToHost, ctx->stream));
    DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return DDP_OK;
}

namespace {

// Seeds s and enqueues the grid search.  Ordinary launch of at most one
// workgroup per CU; those that find room at once are the search's team
// (grid_team.h), and the grid barrier is software with bounded waits (a
// cooperative launch would also reserve the global wave-sync unit, one process
// only).
int pg_enqueue(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P, const GaGridState &S,
               int32_t s, uint32_t hs, int32_t t)
{
    const PgSizes z = ga_pg_sizes(P, gv.N);
    PgArgs a{};
    a.g = gv;
    a.h = hv;
    a.gp = S.gp;
    a.near = S.home;
    a.far0 = S.home + z.ring;
    a.far1 = a.far0 + z.far;
    a.hubs = S.pbuf;
    a.nmask = (uint32_t)(z.ring - 1);
    a.fcap = (uint32_t)z.far;
    a.N = gv.N;
    a.rebuild = z.rebuild;
    a.hubcap = P.hubcap;
    a.ctrl = S.ctrl;
    a.stats = S.stats;
    a.grow = (uint32_t)P.K;
    a.t = t;
    a.maxit = P.maxit;
    a.delta0 = pg_first_window(P.delta0, hv.kind == DDP_H_MANHATTAN);
    a.thr0 = hs > 0xFFFFFFFFu - a.delta0 ? 0xFFFFFFFFu : hs + a.delta0;
    a.barrier_ticks = 100ull * 1000 * 1000 * 20;  // 20 s of the 100 MHz clock
    hipLaunchKernelGGL(pg_seed_kernel, dim3(1), dim3(256), 0, ctx->stream, S.gp, S.home, S.ctrl, s, hs);
    void *args[] = {&a};
    DDP_HIP(ctx, hipLaunchKernel((const void *)pick_pg(hv.kind), dim3(pg_blocks(ctx, P, hv.kind)), dim3(kPgBlock), args,
                                 0, ctx->stream));
    return DDP_OK;
}

// Waits for a grid search (its events recorded) and reads its outcome.
int grid_finish(ddp_ctx *ctx, const GaGridPlan &P, const GaGridState &S, uint32_t *F_out, int32_t *iters_out,
                float *kernel_ms)
{
    uint32_t res[4];
    DDP_HIP(ctx, hipMemcpyAsync(res, S.ctrl + GA_RES_IT, 16, hipMemcpyDeviceToHost, ctx->stream));
    DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    float ms = 0;
    DDP_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    if (kernel_ms) *kernel_ms = ms;
    if (iters_out) *iters_out = (int32_t)res[0];
    if (F_out) *F_out = res[2];
    const uint32_t err = res[3];
    DDP_CHECK(!(err & ERR_BARRIER), ctx, DDP_ERR_TIMEOUT, "GA*: grid barrier wait timed out");
    DDP_CHECK(!(err & ERR_ITERS), ctx, DDP_ERR_TIMEOUT, "GA*: iteration limit %d reached", P.maxit);
    DDP_CHECK(!(err & ERR_HEAP), ctx, DDP_ERR_OVERFLOW,
              "GA*: a queue exceeded heap_cap=%d entries; raise heap_cap", P.cap);
    return DDP_OK;
}

}  // namespace

int ddp_ga_launch(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P,
                  const GaGridState &S, int32_t N, int32_t s, uint32_t hs, int32_t t)
{
    DDP_CHECK(P.pg, ctx, DDP_ERR_STATE, "GA*: not a grid plan");
    int rc;
    if ((rc = ddp_ga_reset(ctx, N, P, S))) return rc;
    return pg_enqueue(ctx, gv, hv, P, S, s, hs, t);
}

// Grid mode on piles: a fresh search (ddp_ga_reset before).
int ddp_ga_run_piles(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P, const GaGridState &S,
                     int32_t s, uint32_t hs, int32_t t, uint32_t *F_out, int32_t *iters_out, float *kernel_ms)
{
    DDP_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    int rc = pg_enqueue(ctx, gv, hv, P, S, s, hs, t);
    if (rc) return rc;
    DDP_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    return grid_finish(ctx, P, S, F_out, iters_out, kernel_ms);
}

int ddp_ga_run_wg(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P,
                  const GaGridState &S, int32_t N, int32_t s, int32_t t, uint32_t *F_out, int32_t *iters_out,
                  float *kernel_ms, const GraphView *gr, int32_t *dpath, int32_t dpath_cap, int32_t *plen)
{
    DDP_CHECK(P.wg && S.touched && P.B == P.K && P.nblocks == 1, ctx, DDP_ERR_STATE, "GA*: not a workgroup plan");
    DDP_CHECK(!P.bidi || gr, ctx, DDP_ERR_STATE, "GA*: the bidirectional plan needs transposed rows");
    WgArgs a{};
    a.g = gv;
    if (gr) a.gr = *gr;
    a.path = dpath;
    a.path_cap = dpath_cap;
    a.h = hv;
    a.gp = S.gp;
    a.home = S.home;  // cap * K entries
    a.touched = S.touched;
    a.ctrl = S.ctrl;
    a.stats = S.stats;
    a.N = N;
    a.s = s;
    a.t = t;
    a.lcap = P.lcap;
    a.cap = P.cap;
    a.maxit = P.maxit;
    a.ncap = P.ncap;
    a.fcap = P.fcap;
    a.delta0 = P.delta0;
    a.lring = P.piles ? 8u * (uint32_t)P.B : 0u;  // LDS near ring
    const size_t lds = P.piles ? (size_t)a.lring * 8 : (size_t)P.lcap * P.B * 8;
    WgFn fn = pick_wg(P.B, hv.kind, P.bidi ? WM_BIDI : P.piles ? WM_PILES : WM_HEAPS);
    DDP_CHECK(fn, ctx, DDP_ERR_ARG, "no workgroup kernel for block %d with this heuristic and mode", P.B);
    DDP_HIP(ctx, hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    DDP_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    hipLaunchKernelGGL(fn, dim3(1), dim3(P.B), lds, ctx->stream, a);
    DDP_HIP(ctx, hipGetLastError());
    DDP_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    uint32_t res[5];
    DDP_HIP(ctx, hipMemcpyAsync(res, S.ctrl + GA_RES_IT, 20, hipMemcpyDeviceToHost, ctx->stream));
    DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    float ms = 0;
    DDP_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    if (kernel_ms) *kernel_ms = ms;
    if (iters_out) *iters_out = (int32_t)res[0];
    if (F_out) *F_out = res[2];
    if (plen) *plen = (int32_t)res[4];
    const uint32_t err = res[3];
    DDP_CHECK(!(err & ERR_ITERS), ctx, DDP_ERR_TIMEOUT, "GA*: iteration limit %d reached", P.maxit);
    DDP_CHECK(!(err & ERR_HEAP), ctx, DDP_ERR_OVERFLOW,
              "GA*: a queue exceeded heap_cap=%d entries; raise heap_cap", P.cap);
    DDP_CHECK(!(err & ERR_PATH), ctx, DDP_ERR_STATE, "GA*: the parent chains through the meeting node are broken");
    return DDP_OK;
}

extern "C" int ddp_astar(ddp_ctx *ctx, const ddp_graph *g, ddp_heur_t h, int32_t s, int32_t t,
                         const ddp_astar_opts_t *opts, int32_t *cost, int32_t *parent_out,
                         int32_t *path_out, int32_t path_cap, int32_t *path_len,
                         ddp_astar_stats_t *stats)
{
    const auto t0 = std::chrono::steady_clock::now();
    if (!ctx || !g || !cost) return ddp_set_err(ctx, DDP_ERR_ARG, "ddp_astar: null argument");
    DDP_CHECK(s >= 0 && s < g->N && t >= 0 && t < g->N, ctx, DDP_ERR_ARG,
              "ddp_astar: s=%d t=%d outside [0,%d)", s, t, g->N);
    DDP_CHECK(!path_out || path_len, ctx, DDP_ERR_ARG, "ddp_astar: path_out needs path_len");
    DDP_HIP(ctx, hipSetDevice(ctx->device));
    s = ddp_to_dev(g, s);
    t = ddp_to_dev(g, t);
    HeurView hv;
    int rc = ddp_make_heur(g, h, t, &hv);
    if (rc) return rc;
    GaGridPlan P;
    if ((rc = ddp_ga_plan(ctx, g, opts, &P, 0, true))) return rc;
    if (P.bidi) {
        DDP_CHECK(g->roff, ctx, DDP_ERR_STATE, "DDP_ASTAR_BIDI needs a graph uploaded with DDP_GRAPH_REVERSE");
        DDP_CHECK(hv.kind != DDP_H_ARRAY, ctx, DDP_ERR_ARG,
                  "DDP_ASTAR_BIDI needs a closed-form heuristic (DDP_H_ZERO, _MANHATTAN or _EUCLID)");
    }
    GaGridState S;
    if ((rc = ddp_ga_alloc(ctx, g, P, &S))) return rc;
    std::vector<int32_t> bpath;  // bidirectional mode: the path walked on the device (device ids)
    int32_t hs = 0;
    if ((rc = ddp_heur_at(g, hv, s, &hs))) return rc;
    if (stats) {
        std::memset(stats, 0, sizeof *stats);
        stats->K = P.K;
        stats->block = P.pg ? kPgBlock : P.B;
        stats->blocks = P.pg ? pg_blocks(ctx, P, hv.kind) : P.nblocks;
    }
    if ((rc = ddp_ga_reset(ctx, g->N, P, S))) return rc;
    if (hv.kind == DDP_H_ARRAY && hs < 0) {
        // h(s) = -1: the heuristic says s cannot reach t.
        *cost = DDP_INF_COST;
        if (path_len) *path_len = 0;
    } else if (s == t) {
        *cost = hs;
        if (path_out && path_cap >= 1) {
            path_out[0] = s;
            *path_len = 1;
        } else if (path_len) {
            *path_len = -1;
        }
    } else {
        uint32_t F = 0;
        int32_t iters = 0;
        float kms = 0;
        if (P.wg && P.bidi) {
            GraphView gv = ddp_view(g);
            gv.relax_min = g->minw >= 1;
            GraphView gr = gv;
            gr.off = g->roff;
            gr.col = g->rcol;
            gr.w = g->rw;
            // the path is walked on the device; a parent array needs all of it
            const int32_t dcap = parent_out ? g->N : (path_out ? std::max(path_cap, 1) : 0);
            int32_t *dpath = nullptr, plen = 0;
            void *p;
            if (dcap > 0) {
                if ((rc = ddp_ws(ctx, WS_PATH, ((size_t)dcap + 64) * 4, &p))) return rc;
                dpath = (int32_t *)p;
            }
            rc = ddp_ga_run_wg(ctx, gv, hv, P, S, g->N, s, t, &F, &iters, &kms, &gr, dpath, dcap, &plen);
            if (!rc && plen != 0) {
                bpath.resize(plen > 0 ? plen : 0);
                if (plen > 0)
                    DDP_HIP(ctx, hipMemcpy(bpath.data(), dpath, (size_t)plen * 4, hipMemcpyDeviceToHost));
                else
                    bpath.assign(1, plen);  // too long for dcap: only the (negative) length is known
            }
        } else if (P.wg) {
            GraphView gv = ddp_view(g);
            gv.relax_min = g->minw >= 1;
            rc = ddp_ga_run_wg(ctx, gv, hv, P, S, g->N, s, t, &F, &iters, &kms);
        } else {
            GraphView gv = ddp_view(g);
            gv.relax_min = g->minw >= 1;
            rc = ddp_ga_run_piles(ctx, gv, hv, P, S, s, (uint32_t)hs, t, &F, &iters, &kms);
        }
        if (rc) return rc;
        *cost = (int32_t)F;
        if (stats) {
            unsigned long long st[4];
            if ((rc = ddp_ga_stats(ctx, S, st))) return rc;
            stats->expansions = (int64_t)st[0];
            stats->edges = (int64_t)st[1];
            stats->improvements = (int64_t)st[2];
            stats->stale_pops = (int64_t)st[3];
            stats->iterations = iters;
            stats->kernel_ms = kms;
        }
        if (path_out && P.bidi) {
            if (F == DDP_INF_F || bpath.empty()) {
                *path_len = 0;
            } else if (bpath.size() == 1 && bpath[0] < 0) {
                *path_len = bpath[0];
            } else if ((int64_t)bpath.size() > path_cap) {
                *path_len = -(int32_t)bpath.size();
            } else {
                std::memcpy(path_out, bpath.data(), bpath.size() * 4);
                *path_len = (int32_t)bpath.size();
            }
        } else if (path_out) {
            if (F == DDP_INF_F) *path_len = 0;
            else if ((rc = ddp_extract_path(ctx, S.gp, g->N, s, t, path_out, path_cap, path_len))) return rc;
        } else if (path_len) {
            *path_len = 0;
        }
    }
    if (parent_out) {
        void *p;
        if ((rc = ddp_ws(ctx, WS_PATH, (size_t)g->N * 4 + 256, &p))) return rc;
        int32_t *dpar = (int32_t *)p;
        hipLaunchKernelGGL(unpack_parent_kernel, dim3(1024), dim3(256), 0, ctx->stream, S.gp, dpar, g->N);
        DDP_HIP(ctx, hipMemcpyAsync(parent_out, dpar, (size_t)g->N * 4, hipMemcpyDeviceToHost, ctx->stream));
        DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
        // bidirectional mode: the forward search's parents, and along the path
        // from the meeting node to t the path's own predecessors, so that the
        // parent chain from t leads back to s
        if (P.bidi && !(bpath.size() == 1 && bpath[0] < 0))
            for (size_t i = 1; i < bpath.size(); ++i) parent_out[bpath[i]] = bpath[i - 1];
        if (!g->iperm.empty()) {  // device ids and order -> caller ids and order
            std::vector<int32_t> tmp(parent_out, parent_out + g->N);
            for (int32_t i = 0; i < g->N; ++i) parent_out[g->iperm[i]] = ddp_to_user(g, tmp[i]);
        }
    }
    if (path_out && path_len && !g->iperm.empty())  // written only when the length is positive
        for (int32_t i = 0; i < *path_len; ++i) path_out[i] = ddp_to_user(g, path_out[i]);
    DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (stats)
        stats->total_ms =
            std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return DDP_OK;
}
