// zg_once.h — what has to be done once for every device of the process (host code, no HIP): kernel attributes are kept by device.
#pragma once
#include <atomic>
#include <cstdint>

namespace zg {

class OncePerDevice {
    std::atomic<uint64_t> done_{0};  // a bit per device

   public:
    // f() unless it has succeeded for this device before (0: success).  Threads that come first together may both call it.
    template <typename F>
    int run(int device, F&& f) {
        const bool kept = device >= 0 && device < 64;
        const uint64_t bit = kept ? uint64_t(1) << device : 0;
        if ((done_.load(std::memory_order_acquire) & bit) != 0) return 0;
        const int status = f();
        if (status == 0) done_.fetch_or(bit, std::memory_order_release);
        return status;
    }
};

}  // namespace zg
