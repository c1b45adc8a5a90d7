// Launch ranges (randomfield_amd/csrc/rf_ranges.h): every block once, in order,
// every grid below 2^32 work-items.
#include "../../randomfield_amd/csrc/rf_ranges.h"

#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);       \
            std::exit(1);                                     \
        }                                                     \
    } while (0)

int main() {
    for (int threads : {64, 256, 512, 1024}) {
        const int64_t most = rf_max_blocks(threads);
        CHECK(most * threads <= 0xffffffffLL && (most + 1) * threads > 0xffffffffLL);
        for (int64_t n : {(int64_t)0, (int64_t)1, most - 1, most, most + 1, 2 * most, 5 * most + 7}) {
            int64_t next = 0;
            int calls = 0;
            const int e = rf_block_ranges(n, threads, [&](int64_t first, unsigned count) {
                CHECK(first == next && count > 0 && (int64_t)count <= most);
                next += count;
                calls++;
                return 0;
            });
            CHECK(e == 0 && next == n && calls == (int)((n + most - 1) / most));
        }
    }
    // the first failure ends it and is returned
    int calls = 0;
    CHECK(rf_block_ranges(4 * rf_max_blocks(256), 256, [&](int64_t, unsigned) { return ++calls == 2 ? 7 : 0; }) == 7);
    CHECK(calls == 2);
    std::printf("ranges ok\n");
    return 0;
}
