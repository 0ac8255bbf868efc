// Sizes of a grid search's piles (grid_piles.h).  No HIP dependency, so the rule
// is also checked on the CPU.
#pragma once

#include <algorithm>
#include <cstdint>

// Entries of the near ring (a power of two) and of each of the two far buffers,
// for K * heap_cap entries in all.  From 2N on, the ring and each buffer hold at
// least 2N, so they can be rebuilt from the N nodes' words when they overflow
// and no search fails for want of room, and the far buffers share what is left:
// together never more than the larger of K * heap_cap and 8N.  Fewer entries are
// the limit that was asked for: the ring and each buffer hold as many, and a
// search that needs more ends with DDP_ERR_OVERFLOW.  (With K * heap_cap for the
// ring and each buffer whatever its size, a heap_cap chosen to fill the memory
// took three to four times that.)
struct PgSizes {
    uint64_t ring, far;
    bool rebuild;
    uint64_t entries() const { return ring + 2 * far; }
};

inline PgSizes pg_sizes(uint64_t wanted, int32_t N)
{
    const uint64_t total = std::min<uint64_t>(wanted, 1ull << 31), most = 2 * (uint64_t)N, least = 1024;
    PgSizes z{least, std::max(total, least), total >= most};
    while (z.ring < std::min(total, most)) z.ring *= 2;
    if (z.rebuild) z.far = std::max({most, (total - std::min(total, z.ring)) / 2, least});
    return z;
}
