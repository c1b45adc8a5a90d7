// Once per device (randomfield_amd/csrc/rf_per_device.h).
#include "../../randomfield_amd/csrc/rf_per_device.h"

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
    rf_per_device p, other;
    int calls = 0, answer = 0;
    auto ask = [&]() { calls++; return answer; };
    // each device asks for itself, once
    for (int device : {0, 1, 7, 63}) {
        const int before = calls;
        CHECK(p.once(device, ask) == 0 && calls == before + 1);
        CHECK(p.once(device, ask) == 0 && calls == before + 1);
    }
    // another kernel's does not count
    CHECK(other.once(0, ask) == 0 && calls == 5);
    // a failure is returned, asked again and then kept as done
    answer = 9;
    CHECK(p.once(2, ask) == 9 && p.once(2, ask) == 9 && calls == 7);
    answer = 0;
    CHECK(p.once(2, ask) == 0 && p.once(2, ask) == 0 && calls == 8);
    // past the mask: every time
    CHECK(p.once(64, ask) == 0 && p.once(64, ask) == 0 && calls == 10);
    std::printf("per device ok\n");
    return 0;
}
