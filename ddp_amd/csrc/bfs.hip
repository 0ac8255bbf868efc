// Reverse-BFS heuristic (bfs_hx).
//
// Reference (GA_star/bfs_hx.cu:11-36, 111-138): one thread per frontier node
// walks its row serially; duplicates are appended when two threads see
// dist = -1 at once; the host launches one kernel per level and copies the
// next frontier size back each time.  Here persistent kernels run the levels:
//   * the queue holds row segments (start, length), not nodes: a row longer
//     than `seg` edges is queued as several, so a hub's edges spread over the
//     whole grid instead of staying with one workgroup, and the row bounds are
//     read by the lane that discovers a node, beside its CAS;
//   * eight lanes walk a segment, eight segments per wave, with no scan or
//     barrier inside a level; a node is queued by the lane whose CAS from -1
//     wins (no duplicates);
//   * a workgroup collects its discoveries in LDS and reserves their places
//     in the queue with one atomic per level (one counter takes about 11 ns
//     per atomic; one per wave made that counter the bound of wide levels);
//   * levels are separated by grid_sync; the size of level L lives in one of
//     three rotating words so no extra barrier is needed to reset it.
// A level is latency-bound until it is thousands of segments wide (about four
// dependent round trips and the barrier), so two grids share the work: the
// narrow one (32 workgroups of 256 lanes, a cheap barrier) runs levels of up
// to kNarrowMax segments, the wide one (a workgroup of 1,024 lanes per CU) the
// others; each returns when the next level is not its own.
// Measured against one grid of 512 workgroups, node queue, fenced barrier (whole
// call, result on the host): random graph of 100,000 nodes 0.87 -> 0.125 ms,
// R-MAT scale 20 (1M nodes, 16.8M edges) 21.8 -> 1.24 ms, 2048 x 2048 maze (4,600
// levels of about 640 nodes) 273 -> 18.9 ms (4.0 us a level).
#include <algorithm>
#include <mutex>

#include "device_common.h"

namespace {

// control words, a line apart where workgroups update them
enum : int {
    BC_CNT = 0,  // three rotating level sizes, 32 words apart
    BC_LEVEL = 96, BC_HEAD = 97, BC_ERR = 98, BC_NEXT = 99, BC_BAR = 128, BC_TEAM = BC_BAR + GRID_SYNC_WORDS,
    BC_WORDS = BC_TEAM + TEAM_WORDS
};

struct BfsArgs {
    const int32_t *off, *col;
    int32_t *dist;
    uint64_t *queue;  // row segments: start | length << 32
    uint32_t cap;     // entries of queue
    uint32_t seg;     // longest segment
    uint32_t lo, hi;  // this grid's levels: lo < segments <= hi
    uint32_t *ctrl;
    uint64_t barrier_ticks;
};

// Row segments of node v in front of the whole wave: the first through
// `first`, the rest of a long row straight into the queue, written by the wave.
__device__ __forceinline__ void bfs_split(const BfsArgs &a, bool is_new, uint32_t b, uint32_t deg, uint32_t base,
                                          uint32_t *ncnt)
{
    uint64_t m = __ballot(is_new && deg > a.seg);
    const uint32_t wl = threadIdx.x & 63;
    while (m) {
        const int src = __builtin_ctzll(m);
        m &= m - 1;
        const uint32_t hb = __builtin_amdgcn_readlane(b, src), hd = __builtin_amdgcn_readlane(deg, src);
        const uint32_t extra = (hd - 1) / a.seg;
        uint32_t at = 0;
        if (wl == 0) at = add_u32(ncnt, extra);
        at = __builtin_amdgcn_readfirstlane(at) + base;
        for (uint32_t k = wl; k < extra; k += 64) {
            const uint32_t o = (k + 1) * a.seg;
            const uint32_t len = hd - o < a.seg ? hd - o : a.seg;
            if (at + k < a.cap) st_u64(a.queue + at + k, (uint64_t)len << 32 | (hb + o));
        }
    }
}

// CHECK: read a target's distance before trying the CAS.  Wide levels meet
// mostly visited nodes, and a load costs less than an atomic (one CU: 0.86
// random loads against 0.59 atomics per ns, 2.4 when they hit L2); a narrow
// level is a chain of round trips and does without that one.
// TEAM: the workgroups that are resident together do the work (grid_team.h);
// the narrow grid, 32 workgroups of four waves, takes up to four CUs and is
// launched as a whole.
template <int B, int U, bool CHECK, bool TEAM>
__global__ void __launch_bounds__(B) bfs_kernel(BfsArgs a)
{
    constexpr uint32_t kLanes = 8, kPerWave = 64 / kLanes, kWaves = B / 64, kLocal = 4 * B;
    __shared__ uint64_t s_q[kLocal];
    __shared__ uint32_t s_n, s_base;
    __shared__ int32_t s_flag;
    __shared__ Team s_team;
    const uint32_t wl = threadIdx.x & 63, sub = wl % kLanes;
    uint32_t *ctrl = a.ctrl;
    const uint32_t rank = TEAM ? grid_arrive(ctrl + BC_TEAM) : 0u;
    uint32_t gen = ld_u32(ctrl + BC_BAR + 32);
    uint32_t level = ctrl[BC_LEVEL], head = ctrl[BC_HEAD];
    uint32_t n = ld_u32(ctrl + BC_CNT + 32 * (level % 3));
    Team tm{blockIdx.x, gridDim.x};
    if constexpr (TEAM) {
        bool timeout;
        tm = grid_team(ctrl + BC_TEAM, rank, a.barrier_ticks, &s_team, timeout, n <= a.lo || n > a.hi);
        if (tm.n == 0) {  // not this grid's level, or the team was complete before this workgroup started
            if (timeout && threadIdx.x == 0) atomicOr(ctrl + BC_ERR, 1u);
            return;
        }
    }
    while (n > a.lo && n <= a.hi) {  // lo >= 0: an empty level ends every grid
        if (tm.me == 0 && threadIdx.x == 0) st_u32(ctrl + BC_CNT + 32 * ((level + 2) % 3), 0);
        uint32_t *ncnt = ctrl + BC_CNT + 32 * ((level + 1) % 3);
        const uint32_t base = head + n;
        const int32_t nl = (int32_t)level + 1;
        if (threadIdx.x == 0) s_n = 0;
        __syncthreads();
        // chunk of kPerWave segments per wave, dealt over the workgroups first
        // so that the segments of one hub go to different CUs
        const uint64_t chunks = ((uint64_t)n + kPerWave - 1) / kPerWave;
        for (uint64_t ch = (threadIdx.x >> 6) * (uint64_t)tm.n + tm.me; ch < chunks;
             ch += (uint64_t)kWaves * tm.n) {
            const uint32_t i = (uint32_t)ch * kPerWave + wl / kLanes;
            uint64_t e = 0;
            if (i < n) e = ld_gp(a.queue + head + i);
            const uint32_t start = (uint32_t)e, len = (uint32_t)(e >> 32);
            for (uint32_t j = 0; __any(j < len); j += kLanes * U) {
                int32_t c[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    c[u] = -1;
                    if (j + u * kLanes + sub < len) c[u] = a.col[start + j + u * kLanes + sub];  // < 0: deleted edge
                }
                if constexpr (CHECK) {
                    int32_t d[U];
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (c[u] >= 0) d[u] = a.dist[c[u]];  // stale copies only miss a visit; the CAS decides
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        if (c[u] >= 0 && d[u] >= 0) c[u] = -1;
                }
                int32_t old[U];
                uint32_t b[U], re[U];
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (c[u] >= 0) old[u] = atomicCAS(a.dist + c[u], -1, nl);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (c[u] >= 0) {
                        b[u] = (uint32_t)a.off[c[u]];
                        re[u] = (uint32_t)a.off[c[u] + 1];
                    }
                bool sel[U];
                uint32_t pos[U];
#pragma unroll
                for (int u = 0; u < U; ++u) sel[u] = c[u] >= 0 && old[u] == -1;
                wave_append<U>(sel, &s_n, pos);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t deg = sel[u] ? re[u] - b[u] : 0;
                    const uint64_t ent = (uint64_t)(deg < a.seg ? deg : a.seg) << 32 | (sel[u] ? b[u] : 0);
                    if (sel[u] && pos[u] < kLocal) s_q[pos[u]] = ent;
                    if (__any(sel[u] && pos[u] >= kLocal)) {  // LDS is full: the wave places these itself
                        const bool far1[1] = {sel[u] && pos[u] >= kLocal};
                        uint32_t fp[1];
                        wave_append<1>(far1, ncnt, fp);
                        if (far1[0] && base + fp[0] < a.cap) st_u64(a.queue + base + fp[0], ent);
                    }
                    bfs_split(a, sel[u], sel[u] ? b[u] : 0, deg, base, ncnt);
                }
            }
        }
        __syncthreads();
        const uint32_t mine = s_n < kLocal ? s_n : kLocal;
        if (threadIdx.x == 0 && mine) s_base = add_u32(ncnt, mine) + base;
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < mine; k += B)
            if (s_base + k < a.cap) st_u64(a.queue + s_base + k, s_q[k]);
        if (!grid_sync(ctrl + BC_BAR, tm, gen, a.barrier_ticks, &s_flag)) {
            if (threadIdx.x == 0) atomicOr(ctrl + BC_ERR, 1u);
            break;
        }
        head = base;
        ++level;
        n = ld_u32(ctrl + BC_CNT + 32 * (level % 3));
    }
    if (tm.me == 0 && threadIdx.x == 0) {
        ctrl[BC_LEVEL] = level;
        ctrl[BC_HEAD] = head;
        ctrl[BC_NEXT] = n;
    }
    if (!TEAM && blockIdx.x == 0)  // for the wide launch behind this one
        for (uint32_t k = threadIdx.x; k < TEAM_WORDS; k += B) st_u32(ctrl + BC_TEAM + k, 0u);
}

// Every distance to -1 but t's, t's row in front of the queue and the control words.
__global__ void bfs_init(const int32_t *off, int32_t *dist, int32_t N, uint64_t *queue, uint32_t cap, uint32_t seg,
                         uint32_t *ctrl, int32_t t)
{
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        dist[i] = i == t ? 0 : -1;
    if (blockIdx.x != 0) return;
    const uint32_t b = (uint32_t)off[t], deg = (uint32_t)off[t + 1] - b;
    const uint32_t parts = deg > seg ? (deg - 1) / seg + 1 : 1;
    for (uint32_t k = threadIdx.x; k < parts && k < cap; k += blockDim.x) {
        const uint32_t o = k * seg;
        queue[k] = (uint64_t)(deg - o < seg ? deg - o : seg) << 32 | (b + o);
    }
    for (int k = threadIdx.x; k < BC_WORDS; k += blockDim.x) ctrl[k] = k == BC_CNT ? parts : 0u;
}

__global__ void bfs_scale(const int32_t *dist, int32_t *out, int32_t N, int32_t scale)
{
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const int32_t d = dist[i];
        out[i] = d < 0 ? -1 : d * scale;
    }
}

// bfs_scale into the caller's numbering: out[iperm[i]] = hops(i) * scale.
__global__ void bfs_scale_perm(const int32_t *dist, const int32_t *iperm, int32_t *out, int32_t N, int32_t scale)
{
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        const int32_t d = dist[i];
        out[iperm[i]] = d < 0 ? -1 : d * scale;
    }
}

// Segments of a row of the default length; a level of one segment per 8 lanes
// fills the narrow grid at 1,024.
constexpr uint32_t kBfsSeg = 64;
constexpr int kNarrowBlocks = 32, kNarrowBlock = 256, kWideBlock = 1024;
constexpr uint32_t kNarrowMax = 4096;

// Queue entries a BFS over N nodes and E edges can need with segments of at
// most seg edges: every node once, and a further entry per seg edges.
uint64_t bfs_entries(int32_t N, int64_t E, uint32_t seg) { return (uint64_t)N + (uint64_t)E / seg + 1; }

// Runs the BFS from device node t into dist (N entries) with queue (cap
// entries, at least bfs_entries for seg) and ctrl (BC_WORDS words) as scratch;
// waits for it and returns the level count.  Allocates nothing.
int bfs_run(ddp_ctx *ctx, const ddp_graph *g, int32_t t, int32_t reverse, int32_t *dist, uint64_t *queue,
            uint32_t cap, uint32_t seg, uint32_t *ctrl, int32_t *levels)
{
    const int32_t N = g->N;
    const int32_t *off = reverse ? g->roff : g->off;
    const int wide_blocks = ctx->prop.multiProcessorCount;
    // the control words are cleared by a kernel, not a memset node
    hipLaunchKernelGGL(bfs_init, dim3(std::min(1024, (N + 255) / 256)), dim3(256), 0, ctx->stream, off, dist, N,
                       queue, cap, seg, ctrl, t);
    BfsArgs a{off, reverse ? g->rcol : g->col, dist, queue, cap, seg, 0, 0, ctrl, 100ull * 1000 * 1000 * 20};
    // Ordinary launches: the grid barrier is software and only needs its
    // workgroups resident at once (a cooperative launch would also reserve the
    // GPU's global wave-sync unit, which only one process may hold).  Every
    // barrier wait is bounded, so a narrow grid without room for its 32
    // workgroups ends with DDP_ERR_TIMEOUT, not a hang.
    const bool wide = bfs_entries(N, reverse ? g->RE : g->E, seg) > kNarrowMax;  // some level may be
    auto run = [&](bool w) {
        a.lo = w ? kNarrowMax / 2 : 0;  // the wide grid keeps a level until it is clearly narrow
        a.hi = w ? 0xFFFFFFFFu : kNarrowMax;
        void *args[] = {&a};
        return w ? hipLaunchKernel((const void *)bfs_kernel<kWideBlock, 2, true, true>, dim3(wide_blocks),
                                   dim3(kWideBlock), args, 0, ctx->stream)
                 : hipLaunchKernel((const void *)bfs_kernel<kNarrowBlock, 1, false, false>, dim3(kNarrowBlocks),
                                   dim3(kNarrowBlock), args, 0, ctx->stream);
    };
    uint32_t res[4];
    for (;;) {
        // narrow, wide, narrow covers a search that grows and dies down once
        DDP_HIP(ctx, run(false));
        if (wide) {
            DDP_HIP(ctx, run(true));
            DDP_HIP(ctx, run(false));
        }
        DDP_HIP(ctx, hipMemcpyAsync(res, ctrl + BC_LEVEL, 16, hipMemcpyDeviceToHost, ctx->stream));
        DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
        DDP_CHECK(res[BC_ERR - BC_LEVEL] == 0, ctx, DDP_ERR_TIMEOUT, "bfs: grid barrier wait timed out");
        if (res[BC_NEXT - BC_LEVEL] == 0) break;
    }
    *levels = (int32_t)res[0];
    return DDP_OK;
}

int bfs_check(ddp_ctx *ctx, const ddp_graph *g, int32_t t, int32_t reverse, int32_t scale, const char *who)
{
    if (!ctx || !g) return ddp_set_err(ctx, DDP_ERR_ARG, "%s: null argument", who);
    DDP_CHECK(t >= 0 && t < g->N, ctx, DDP_ERR_ARG, "%s: t=%d outside [0,%d)", who, t, g->N);
    DDP_CHECK(!reverse || g->roff, ctx, DDP_ERR_STATE, "%s: reverse=1 needs a graph uploaded with DDP_GRAPH_REVERSE",
              who);
    DDP_CHECK(scale >= 1, ctx, DDP_ERR_ARG, "%s: scale must be >= 1", who);
    return DDP_OK;
}

// ------------------------------------------------- allocation-free variant
//
// Device memory of ddp_bfs_hops_noalloc: the queue (an 8-byte entry per node
// and kBfsScratchExtra more for the parts of long rows), the distance array
// and the control words of one BFS over at most kBfsScratchNodes nodes (26 MiB).
// Every GPU the library runs on holds its own copy until the process ends.
// In host code the name is not a device address: kernels get
// scratch_dev(device), the address hipGetSymbolAddress returns for that device.
constexpr int32_t kBfsScratchNodes = 1 << 21, kBfsScratchExtra = 1 << 18;
static __device__ __align__(256)
    int32_t scratch[3 * (size_t)kBfsScratchNodes + 2 * (size_t)kBfsScratchExtra + BC_WORDS];

constexpr int kMaxDevices = 64;
static std::mutex s_scratch_mu;
static int32_t *s_scratch_ptr[kMaxDevices];

// The address of this device's copy of scratch, looked up once per device
// with that device current.
static int scratch_dev(ddp_ctx *ctx, int32_t **out)
{
    DDP_CHECK(ctx->device >= 0 && ctx->device < kMaxDevices, ctx, DDP_ERR_ARG, "device %d out of range",
              ctx->device);
    std::lock_guard<std::mutex> lock(s_scratch_mu);
    if (!s_scratch_ptr[ctx->device]) {
        void *p = nullptr;
        DDP_HIP(ctx, hipSetDevice(ctx->device));
        DDP_HIP(ctx, hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        DDP_CHECK(p != nullptr, ctx, DDP_ERR_HIP, "hipGetSymbolAddress(scratch) returned no address");
        s_scratch_ptr[ctx->device] = (int32_t *)p;
    }
    *out = s_scratch_ptr[ctx->device];
    return DDP_OK;
}

}  // namespace

extern "C" int ddp_bfs_hops(ddp_ctx *ctx, ddp_graph *g, int32_t t, int32_t reverse, int32_t scale,
                            int32_t store_as_h, int32_t *h_out, int32_t *levels_out)
{
    int rc = bfs_check(ctx, g, t, reverse, scale, "ddp_bfs_hops");
    if (rc) return rc;
    DDP_HIP(ctx, hipSetDevice(ctx->device));
    const int32_t N = g->N;
    t = ddp_to_dev(g, t);
    void *p;
    const uint64_t cap = bfs_entries(N, reverse ? g->RE : g->E, kBfsSeg);  // N + E/64 < 2^32
    if ((rc = ddp_ws(ctx, WS_BFS_FRONT, (size_t)cap * 8 + (size_t)N * 4, &p))) return rc;
    uint64_t *queue = (uint64_t *)p;
    int32_t *dist = (int32_t *)(queue + cap);
    if ((rc = ddp_ws(ctx, WS_BFS_CTRL, BC_WORDS * 4, &p))) return rc;
    uint32_t *ctrl = (uint32_t *)p;
    int32_t levels = 0;
    if ((rc = bfs_run(ctx, g, t, reverse, dist, queue, (uint32_t)cap, kBfsSeg, ctrl, &levels))) return rc;
    if (levels_out) *levels_out = levels;
    int32_t *scaled = dist;
    if (scale != 1 || store_as_h) {
        if (store_as_h) {
            if (!g->h) DDP_HIP(ctx, hipMalloc((void **)&g->h, (size_t)N * 4));
            scaled = g->h;
            g->h_target = t;
        } else {
            scaled = (int32_t *)queue;  // free now, and 8N bytes at least
        }
        hipLaunchKernelGGL(bfs_scale, dim3(1024), dim3(256), 0, ctx->stream, dist, scaled, N, scale);
    }
    if (h_out && g->iperm.empty()) {
        DDP_HIP(ctx, hipMemcpyAsync(h_out, scaled, (size_t)N * 4, hipMemcpyDeviceToHost, ctx->stream));
    } else if (h_out) {  // device order -> caller order
        std::vector<int32_t> tmp(N);
        DDP_HIP(ctx, hipMemcpyAsync(tmp.data(), scaled, (size_t)N * 4, hipMemcpyDeviceToHost, ctx->stream));
        DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
        for (int32_t i = 0; i < N; ++i) h_out[g->iperm[i]] = tmp[i];
    }
    DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return DDP_OK;
}

extern "C" int ddp_bfs_hops_noalloc(ddp_ctx *ctx, const ddp_graph *g, int32_t t, int32_t reverse, int32_t scale,
                                    int32_t *h_out_dev, int32_t *levels_out)
{
    int rc = bfs_check(ctx, g, t, reverse, scale, "ddp_bfs_hops_noalloc");
    if (rc) return rc;
    DDP_CHECK(h_out_dev, ctx, DDP_ERR_ARG, "ddp_bfs_hops_noalloc: null output");
    DDP_CHECK(g->N <= kBfsScratchNodes, ctx, DDP_ERR_CAPACITY,
              "ddp_bfs_hops_noalloc: N = %d exceeds the %d nodes its static device memory holds", g->N,
              kBfsScratchNodes);
    DDP_HIP(ctx, hipSetDevice(ctx->device));
    int32_t *base = nullptr;
    if ((rc = scratch_dev(ctx, &base))) return rc;
    const int32_t N = g->N;
    // queue N + kBfsScratchExtra entries, dist N, ctrl BC_WORDS; rows are cut
    // into parts long enough that the extra entries hold them
    const uint32_t cap = (uint32_t)N + kBfsScratchExtra;
    const uint32_t seg = std::max<uint32_t>(kBfsSeg, (uint32_t)((reverse ? g->RE : g->E) / (kBfsScratchExtra - 1)) + 1);
    uint64_t *queue = (uint64_t *)base;
    int32_t *dist = base + 2 * (size_t)cap;
    uint32_t *ctrl = (uint32_t *)(dist + N);
    int32_t levels = 0;
    if ((rc = bfs_run(ctx, g, ddp_to_dev(g, t), reverse, dist, queue, cap, seg, ctrl, &levels))) return rc;
    if (levels_out) *levels_out = levels;
    if (g->d_iperm)
        hipLaunchKernelGGL(bfs_scale_perm, dim3(1024), dim3(256), 0, ctx->stream, dist, (const int32_t *)g->d_iperm,
                           h_out_dev, N, scale);
    else
        hipLaunchKernelGGL(bfs_scale, dim3(1024), dim3(256), 0, ctx->stream, dist, h_out_dev, N, scale);
    DDP_HIP(ctx, hipGetLastError());
    DDP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return DDP_OK;
}
