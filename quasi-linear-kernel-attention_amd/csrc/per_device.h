// Host code: something done once for each device.
#pragma once

#include <atomic>
#include <cstdint>

namespace qlka {

// once(device, f) runs f() unless it has succeeded for that device before, and returns its status (0: success, and
// later calls return 0 at once). A failure is not remembered. Threads that come together may each run f.
class PerDevice {
public:
    template <class F>
    int operator()(int device, F f) {
        const bool tracked = device >= 0 && device < 64;
        if (tracked && (done_.load(std::memory_order_acquire) >> device & 1)) return 0;
        if (int e = f()) return e;
        if (tracked) done_.fetch_or(uint64_t(1) << device, std::memory_order_release);
        return 0;
    }

private:
    std::atomic<uint64_t> done_{0};
};

}  // namespace qlka
