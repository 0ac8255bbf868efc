// The pile sizes of a grid search (ddp_amd/csrc/pile_sizes.h).  Prints "failures 0".
#include <cstdio>

#include "pile_sizes.h"

int main()
{
    int failures = 0;
    auto check = [&](bool ok, const char *what, uint64_t wanted, uint64_t N) {
        if (ok) return;
        std::printf("FAILED: %s (%llu entries, N = %llu)\n", what, (unsigned long long)wanted, (unsigned long long)N);
        ++failures;
    };
    for (uint64_t N : {1ul, 2ul, 511ul, 512ul, 513ul, 1000ul, 30000ul, 65536ul, 1000003ul, 1ul << 24, (1ul << 30) - 1,
                       (1ul << 31) - 1})
        for (uint64_t wanted : {1ul, 1023ul, 1024ul, 60000ul, 2 * N - 1, 2 * N, 2 * N + 1, 2 * N + 262144, 4 * N, 8 * N,
                                8 * N + 1, 100 * N, 1ul << 31, (1ul << 31) + 5, 1ul << 36}) {
            const PgSizes z = pg_sizes(wanted, (int32_t)N);
            const uint64_t total = wanted < (1ull << 31) ? wanted : 1ull << 31, small = 3 * 1024;
            check((z.ring & (z.ring - 1)) == 0 && z.ring >= 1024 && z.ring <= (1ull << 31), "ring is a power of two", wanted, N);
            check(z.far < (1ull << 32), "positions fit 32 bits", wanted, N);
            if (total >= 2 * N) {
                check(z.rebuild && z.ring >= 2 * N && z.far >= 2 * N, "room to rebuild", wanted, N);
                check(z.entries() <= std::max({total, 8 * N, small}), "within what was asked for", wanted, N);
            } else {
                check(!z.rebuild && z.ring >= total && z.far >= total, "as many as the limit", wanted, N);
                check(z.entries() <= std::max<uint64_t>(8 * N, small), "within 8N", wanted, N);
            }
        }
    std::printf("failures %d\n", failures);
    return failures != 0;
}
