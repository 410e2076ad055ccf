// What a process has to do once on every device and not once: hipFuncSetAttribute acts on the device that is current.
#pragma once
#include <atomic>
#include <cstdint>

namespace mimir {

class OnceADevice {
    std::atomic<uint64_t> done_{0};  // a bit a device

public:
    // set(), unless it has succeeded (returned zero) for `device` before. Threads may race here: both then call it. A device past
    // the 63rd is set each time.
    template <typename Set>
    auto operator()(int device, Set set) -> decltype(set()) {
        const uint64_t bit = device >= 0 && device < 64 ? uint64_t(1) << device : 0;
        if ((done_.load(std::memory_order_acquire) & bit) != 0) return decltype(set())(0);
        const auto status = set();
        if (status == decltype(set())(0)) done_.fetch_or(bit, std::memory_order_release);
        return status;
    }
};

}  // namespace mimir
