// Host-side interface of the single-query GA* kernels, shared by the entry
// points that run them (ddp_astar, serving, DA*).
#pragma once

#include "ddp_internal.h"

// Control block layout (uint32 words): the result words; grid_piles.h keeps its
// counters behind them.
enum : int {
    GA_RES_IT = 32, GA_RES_F = 34, GA_RES_ERR = 35, GA_RES_PLEN = 36,
    GA_CTRL_WORDS = 1280,
};

// Error bits of GA_RES_ERR.
enum : uint32_t { GA_ERR_HEAP = 1, GA_ERR_ITERS = 4, GA_ERR_BARRIER = 8 };

struct GaGridPlan {
    int32_t K, B, nblocks, lcap, cap, pcap, maxit;
    bool wg = false;     // one workgroup (ddp_astar only): lane heaps, or piles when `piles`
    bool piles = false;
    bool bidi = false;   // piles from both ends: two (f, parent) arrays, touched logs and pile sets
    uint32_t ncap = 0, fcap = 0, delta0 = 1;  // pile mode: near ring, far buffers, first window
    // grid mode (grid_piles.h): the graph's edges and the segments one round's long rows can be cut into
    bool pg = false;
    int64_t edges = 0;
    uint32_t hubcap = 0;
};

// Device buffers of one GA* search state.
struct GaGridState {
    uint64_t *gp = nullptr;      // N packed (f << 32 | parent); bidirectional: 2N, forward then backward
    uint64_t *home = nullptr;    // cap * K queue entries (bidirectional: twice; grid mode: ga_pg_sizes)
    int32_t *touched = nullptr;  // N, workgroup mode only (bidirectional: 2N)
    uint64_t *pbuf = nullptr;    // grid mode: hubcap segments of 2 words
    uint32_t *ctrl = nullptr;    // GA_CTRL_WORDS
    unsigned long long *stats = nullptr;  // 8 counters after ctrl
    bool owned = false;          // allocated by ddp_ga_alloc_owned (freed by ddp_ga_free)
};

// min_pcap: lower bound on pcap, the room for a DA* batch's repair pushes.
// allow_wg: honour opts->mode and plan the workgroup mode when it applies.
int ddp_ga_plan(ddp_ctx *ctx, const ddp_graph *g, const ddp_astar_opts_t *o, GaGridPlan *p,
                int64_t min_pcap = 0, bool allow_wg = false);
// State in the context's reusable scratch (valid until the next ddp_astar on ctx).
int ddp_ga_alloc(ddp_ctx *ctx, const ddp_graph *g, const GaGridPlan &P, GaGridState *S);
// Grid-mode state owned by the caller (serving), freed by ddp_ga_free.
int ddp_ga_alloc_owned(ddp_ctx *ctx, int32_t N, const GaGridPlan &P, GaGridState *S);
void ddp_ga_free(GaGridState *S);
// gp = INF everywhere, queues empty, counters zero.
int ddp_ga_reset(ddp_ctx *ctx, int32_t N, const GaGridPlan &P, const GaGridState &S);
// Grid mode on piles: a fresh search from s to completion (ddp_ga_reset before; no seed needed).
int ddp_ga_run_piles(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P, const GaGridState &S,
                     int32_t s, uint32_t hs, int32_t t, uint32_t *F_out, int32_t *iters_out, float *kernel_ms);
// Grid mode on piles, asynchronous: resets the state, seeds s and enqueues the grid
// kernel on ctx->stream without waiting.  Stream-ordered work after it reads
// the outcome from S.ctrl (GA_RES_F: f of t, DDP_INF_F if unreachable;
// GA_RES_ERR: GA_ERR_* bits).
int ddp_ga_launch(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P,
                  const GaGridState &S, int32_t N, int32_t s, uint32_t hs, int32_t t);
// Workgroup mode: one search from s to completion (no seed needed).  The
// bidirectional plan also needs the transposed rows (gr) and walks the path on
// the device into dpath[0..dpath_cap) (length to *plen: 0 if unreachable,
// -len if dpath_cap is too small) when dpath is given.
int ddp_ga_run_wg(ddp_ctx *ctx, const GraphView &gv, const HeurView &hv, const GaGridPlan &P,
                  const GaGridState &S, int32_t N, int32_t s, int32_t t, uint32_t *F_out, int32_t *iters_out,
                  float *kernel_ms, const GraphView *gr = nullptr, int32_t *dpath = nullptr, int32_t dpath_cap = 0,
                  int32_t *plen = nullptr);
// Reads the four search counters (expanded, edges, improved, stale).
int ddp_ga_stats(ddp_ctx *ctx, const GaGridState &S, unsigned long long out[4]);
