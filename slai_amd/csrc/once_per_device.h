// A setting that the runtime keeps per device (a kernel's limit of dynamic LDS), made before the first launch on each of them.
#pragma once
#include <atomic>
#include <stdint.h>

namespace slai {

class OncePerDevice {
public:
    // set() unless it has succeeded on this device; its status (0: success).  A failure is not remembered, devices past
    // the 64th are set each time, and threads that meet here set twice at worst.
    template <class F> auto operator()(int device, F &&set) -> decltype(set()) {
        using Status = decltype(set());
        const uint64_t bit = device >= 0 && device < 64 ? 1ull << device : 0;
        if (done_.load(std::memory_order_acquire) & bit) return (Status)0;
        const Status status = set();
        if (status == (Status)0) done_.fetch_or(bit, std::memory_order_release);
        return status;
    }

private:
    std::atomic<uint64_t> done_{0};
};

}  // namespace slai
