// The workgroups of a launch that are resident together, found at its start.
//
// A kernel whose workgroups meet at a software barrier needs all of them on
// the GPU at once.  A grid of one 1,024-lane workgroup per CU has that on an idle
// GPU only: beside a serving kernel that holds some of the CUs (another
// context, another process), or beside a second such grid, part of it would
// wait for CUs while the rest waits at the barrier.  So the launch's members
// are the workgroups that have started when the last one does, or when the
// first has waited kTeamWait for the others; a workgroup that starts later
// finds the team closed and leaves at once.  Whatever is resident does the work,
// and no member waits for a workgroup that is not running.
//
// On an idle GPU it costs 2 us a launch (BFS of a random graph of 100,000 nodes
// 123 and 125 us, a grid search on it 417 and 420).  Beside 160 and 224 idle slots
// of a server in another context, searches of 600,000 nodes take 1.0 and 1.6 ms
// (0.9 alone); a whole grid would spin until the server leaves, or fail after 20 s.
//
// Arrivals are counted in eight groups (one word takes about 11 ns per atomic),
// as in grid_sync.  Host-compilable: Mem gives the accesses (add, fetch_or, load,
// store, and a fence after which this thread's stores are seen before its next
// one), a clock in 100 MHz ticks and a pause.
#pragma once

#include <cstdint>

#ifdef __HIPCC__
#define DDP_HOST_DEVICE __host__ __device__
#else
#define DDP_HOST_DEVICE
#endif

constexpr uint32_t kTeamGroups = 8;
constexpr uint32_t kTeamClosed = 0x80000000u;
constexpr uint64_t kTeamWait = 100 * 100;  // 100 us: a grid starts within about 10
// Words of a team, zeroed before the launch, a 128-byte line per counter: full
// groups (and kTeamClosed); the settled team (member count, then the first
// number of each group); arrivals of each group (and kTeamClosed).
constexpr uint32_t TEAM_SIZE = 32, TEAM_GROUP = 64, TEAM_WORDS = TEAM_GROUP + 32 * kTeamGroups;

enum : int { TEAM_MEMBER, TEAM_CLOSED, TEAM_TIMEOUT };

// Workgroup `block` of `grid` arrives (the first thing it does, so that the
// atomic's round trip overlaps what it loads), and then waits for the team to be
// settled.  A member gets its number and the member count (a whole grid keeps its
// own numbers); TEAM_CLOSED: too late, leave; TEAM_TIMEOUT: nobody settled the
// team within limit ticks.
template <class Mem>
DDP_HOST_DEVICE inline uint32_t team_arrive(Mem &m, typename Mem::Word *words, uint32_t block)
{
    return m.add(words + TEAM_GROUP + 32 * (block % kTeamGroups), 1u);
}

template <class Mem>
DDP_HOST_DEVICE inline int team_settle(Mem &m, typename Mem::Word *words, uint32_t rank, uint32_t block, uint32_t grid,
                                       uint64_t limit, uint32_t &me, uint32_t &n)
{
    const uint32_t groups = grid < kTeamGroups ? grid : kTeamGroups, g = block % kTeamGroups;
    const uint32_t most = (grid - g + kTeamGroups - 1) / kTeamGroups;
    me = block;
    n = 0;
    if (rank & kTeamClosed) return TEAM_CLOSED;
    if (rank == most - 1 && m.add(words, 1u) == groups - 1) {  // everybody is here
        n = grid;
        m.store(words + TEAM_SIZE, n);
        return TEAM_MEMBER;
    }
    const uint64_t t0 = m.clock();
    bool may_close = true;
    while ((n = m.load(words + TEAM_SIZE)) == 0) {
        const uint64_t waited = m.clock() - t0;
        if (may_close && waited > kTeamWait) {
            // one member closes, unless the last one has come after all
            may_close = false;
            const uint32_t full = m.fetch_or(words, kTeamClosed);
            if (full != groups && !(full & kTeamClosed)) {
                uint32_t total = 0;
                for (uint32_t k = 0; k < groups; ++k) {
                    m.store(words + TEAM_SIZE + 1 + k, total);
                    total += m.fetch_or(words + TEAM_GROUP + 32 * k, kTeamClosed);
                }
                m.fence();
                m.store(words + TEAM_SIZE, total);
            }
            continue;
        }
        if (waited > limit) return TEAM_TIMEOUT;
        m.pause();
    }
    if (n != grid) me = m.load(words + TEAM_SIZE + 1 + g) + rank;
    return TEAM_MEMBER;
}
