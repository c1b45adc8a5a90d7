// rf_per_device.h -- what a kernel asks of the runtime once per device (host only).
#pragma once

#include <atomic>
#include <cstdint>

// A function attribute belongs to the function on one device.  once(device, ask)
// calls ask() until it has succeeded (returned zero) for that device, then no
// more; a failure is returned and not kept.  Two threads at once may both ask.
// Devices past 63 ask every time.
struct rf_per_device {
    std::atomic<uint64_t> done{0};

    template <typename F>
    auto once(int device, F ask) -> decltype(ask()) {
        const uint64_t bit = device >= 0 && device < 64 ? (uint64_t)1 << device : 0;
        if (done.load(std::memory_order_acquire) & bit) return {};
        const auto e = ask();
        if (!e) done.fetch_or(bit, std::memory_order_release);
        return e;
    }
};
