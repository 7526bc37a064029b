// What has to happen once on every device before a launch there, such as a
// kernel's dynamic LDS limit (hipFuncSetAttribute holds for the current device
// only).
#pragma once

#include <stdint.h>

#include <atomic>

namespace anelm {

class DeviceOnce {
public:
    // `set` on the first call for device `id` (0 .. 63); its status, kept as
    // done only when it is 0.  Threads that meet on a device's first call may
    // each run `set`: it has to bear repetition.
    template <class F>
    int run(int id, F set) {
        const uint64_t bit = uint64_t(1) << id;
        if (done_.load(std::memory_order_acquire) & bit) return 0;
        const int rc = set();
        if (rc == 0) done_.fetch_or(bit, std::memory_order_release);
        return rc;
    }

private:
    std::atomic<uint64_t> done_{0};
};

}  // namespace anelm
