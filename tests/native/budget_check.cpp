// Host check of the launch budget (egt_budget.h): what runs together never exceeds the capacity, per device, from many
// threads; a share goes back at the end of its scope. Prints how many checks failed.
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
#include "egt_budget.h"

int main() {
    int bad = 0;
    egt::TileBudget b;
    {
        egt::TileShare one(b, 0, 1024, 1024);
        bad += !one;
        egt::TileShare two(b, 0, 1, 1024);  // full
        bad += (bool)two;
        egt::TileShare other(b, 1, 1024, 1024);  // another device has its own
        bad += !other;
    }
    {
        egt::TileShare all(b, 0, 1024, 1024);  // everything came back, the refused share gave nothing
        bad += !all;
    }
    egt::TileShare large(b, 0, 1025, 1024);
    bad += (bool)large;
    std::atomic<int> now{0}, most{0}, taken{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&, t] {
            for (int i = 0; i < 2000; ++i) {
                const int tiles = 100 + 97 * t;
                egt::TileShare s(b, 0, tiles, 1024);
                if (!s) continue;
                ++taken;
                const int v = now += tiles;
                int m = most;
                while (v > m && !most.compare_exchange_weak(m, v)) {
                }
                now -= tiles;
            }
        });
    for (auto& t : threads) t.join();
    bad += most > 1024 || taken == 0;
    egt::TileShare end(b, 0, 1024, 1024);
    bad += !end;
    std::printf("%d\n", bad);
    return bad;
}
