// State that belongs to a device and not to the process.
#pragma once

#include <atomic>
#include <cstdint>

// Runs f (0: success) unless it has succeeded for this device before.  A failure
// is returned and not kept; threads that meet at the first call may both run f.
class OncePerDevice {
    std::atomic<uint64_t> done_{0};

public:
    template <typename F>
    int operator()(int device, F f) {
        const uint64_t bit = device >= 0 && device < 64 ? 1ull << device : 0;  // (others: every call)
        if (done_.load(std::memory_order_acquire) & bit) return 0;
        const int e = f();
        if (e == 0) done_.fetch_or(bit, std::memory_order_release);
        return e;
    }
};
