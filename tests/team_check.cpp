// The team protocol (ddp_amd/csrc/grid_team.h) on CPU threads: a GPU is a number
// of CUs, each running one workgroup at a time to its end, in launch order.
// Whatever number of workgroups finds room, the members number themselves 0..n-1,
// meet at barriers among themselves, deal out every item once and end; with
// room for all of them the whole grid is the team.  Prints "failures 0".
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "grid_team.h"

using clk = std::chrono::steady_clock;

struct CpuMem {
    using Word = std::atomic<uint32_t>;
    uint32_t add(Word *p, uint32_t v) { return p->fetch_add(v); }
    uint32_t fetch_or(Word *p, uint32_t v) { return p->fetch_or(v); }
    uint32_t load(Word *p) { return p->load(); }
    void store(Word *p, uint32_t v) { p->store(v); }
    void fence() {}
    uint64_t clock()
    {
        return std::chrono::duration_cast<std::chrono::nanoseconds>(clk::now().time_since_epoch()).count() / 10;
    }
    void pause() { std::this_thread::yield(); }
};

static int failures = 0;

static void check(bool ok, const char *what, uint32_t grid, uint32_t cus)
{
    if (ok) return;
    std::printf("FAILED: %s (grid %u, CUs %u)\n", what, grid, cus);
    ++failures;
}

static void launch(uint32_t grid, uint32_t cus, unsigned late_us)
{
    std::vector<CpuMem::Word> words(TEAM_WORDS);
    CpuMem::Word arrived{0}, next{0};
    constexpr uint32_t kItems = 1000, kRounds = 3;
    std::vector<std::atomic<uint32_t>> done(kItems), seen(grid);
    std::atomic<uint32_t> members{0}, size{0}, bad{0}, timeouts{0};
    auto workgroup = [&](uint32_t block) {
        CpuMem m;
        uint32_t me, n;
        const uint32_t rank = team_arrive(m, words.data(), block);
        const int got = team_settle(m, words.data(), rank, block, grid, 100ull * 1000 * 1000 * 10, me, n);
        if (got == TEAM_TIMEOUT) ++timeouts;
        if (got != TEAM_MEMBER) return;
        ++members;
        size = n;
        if (n == 0 || n > grid || me >= n || seen[me].fetch_add(1) != 0) ++bad;
        for (uint32_t r = 0; r < kRounds; ++r) {
            for (uint32_t k = me; k < kItems; k += n) ++done[k];
            // barrier among the members, bounded
            ++arrived;
            const auto t0 = clk::now();
            while (arrived < n * (r + 1)) {
                if (clk::now() - t0 > std::chrono::seconds(10)) {
                    ++timeouts;
                    return;
                }
                std::this_thread::yield();
            }
        }
    };
    std::vector<std::thread> gpu;
    for (uint32_t c = 0; c < cus; ++c)
        gpu.emplace_back([&, c] {
            if (c > 0 && late_us) std::this_thread::sleep_for(std::chrono::microseconds(late_us * c));
            for (uint32_t g; (g = next++) < grid;) workgroup(g);
        });
    for (auto &t : gpu) t.join();
    check(timeouts == 0, "a wait ran out", grid, cus);
    check(bad == 0, "numbers are not 0..n-1", grid, cus);
    check(members == size && members >= 1, "member count", grid, cus);
    for (auto &d : done)
        if (d != kRounds) {
            check(false, "an item was not done once a round", grid, cus);
            break;
        }
    if (cus >= grid && !late_us) check(members <= grid, "more members than workgroups", grid, cus);
}

int main()
{
    const uint32_t shapes[][2] = {{1, 1}, {2, 1}, {2, 2}, {8, 3}, {16, 16}, {64, 1}, {64, 7}, {33, 32}, {40, 39}};
    for (int rep = 0; rep < 10; ++rep)
        for (auto &s : shapes)
            for (unsigned late : {0u, 60u}) launch(s[0], s[1], late);
    std::printf("failures %d\n", failures);
    return failures != 0;
}
