// Host check of the launch sizes (egt_limits.h): no launch reaches 2^32 threads at any size; where the work goes out in
// parts these cover it once, in order, and below the limit it is one launch. Prints how many checks failed.
#include <cstdio>
#include "egt_limits.h"

int main() {
    int bad = 0;
    const int64_t limit = (int64_t)1 << 32;
    // items in launches of MAX_GROUPS workgroups of 256 threads, `per` items each
    auto check = [&](int64_t items, int64_t per, bool one) {
        int64_t next = 0, launches = 0;
        egt::in_launches(items, egt::MAX_GROUPS * per, [&](int64_t first, int64_t count) {
            bad += first != next || count < 1;
            bad += (count + per - 1) / per * 256 >= limit;
            next = first + count;
            ++launches;
        });
        bad += next != items;
        bad += (launches == 1) != one;
    };
    // the wave-per-query search: chunks of 64 queries, up to its own and the largest point and query count
    bad += egt::WAVE_MAX_QUERIES < ((int64_t)1 << 30) - 64;
    const int64_t queries[] = {1, 64, 65, 99968, 99969, 300000, 268435391, 268435392, 268435393, 268435456,
                               268435457, 536870912, 1073741760, 1073741761, 1073741824, INT32_MAX};
    for (int64_t q : queries) {
        const int64_t chunks = (q + 63) / 64;
        const int qpw = egt::queries_per_wave(chunks * 64);
        bad += qpw < 1 || 16 % qpw != 0;
        // a chunk's workgroups, of four waves with qpw queries each, serve its 64 queries
        bad += egt::wave_groups_per_chunk(qpw) * 4 * qpw != 64;
        if (chunks * 64 <= egt::WAVE_MAX_QUERIES)
            bad += chunks * egt::wave_groups_per_chunk(qpw) * 256 >= limit;
        else
            bad += (chunks + 3) / 4 * 256 >= limit;  // a lane per query
        check(q, 4 * qpw, q <= egt::MAX_GROUPS * 4 * qpw);  // a list of queries
    }
    // plain splits by workgroups
    check(1, 1, true);
    check(egt::MAX_GROUPS, 1, true);
    check(egt::MAX_GROUPS + 1, 1, false);
    check((int64_t)11 * INT32_MAX / 256, 1, false);  // level inserts: a thread per cell of 11 levels
    check((int64_t)4 * INT32_MAX / 256, 1, false);   // edge list: four threads per row
    egt::in_launches(0, egt::MAX_GROUPS, [&](int64_t, int64_t) { ++bad; });
    // iterations of one launch: none and too many are not for it, and twice the most are an int
    bad += egt::resident_iterations(0) || egt::resident_iterations(-1) || !egt::resident_iterations(1);
    bad += !egt::resident_iterations(1000000) || egt::resident_iterations(1 << 30) || egt::resident_iterations(INT32_MAX);
    bad += 2 * (int64_t)egt::MAX_RESIDENT_ITERATIONS > INT32_MAX;
    std::printf("%d\n", bad);
    return bad;
}
