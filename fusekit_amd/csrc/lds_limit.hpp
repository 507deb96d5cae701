// How much dynamic LDS each kernel has been allowed, for the whole process: the runtime keeps ONE limit per kernel, so a planner that
// sets what its own launch needs would lower what another shape's launch, planned earlier or by another thread, relies on.
// Limits therefore only rise.  (A process uses one device: the device's facts are read once, too.)
#pragma once
#include <stdint.h>

#include <map>
#include <mutex>

namespace fk {

class LdsLimits {
public:
    // set(bytes) asks the runtime, under the lock and only for more than the kernel has; returns its status (0: done).
    template <typename Set>
    int raise(const void* func, uint32_t bytes, Set&& set) {
        std::lock_guard<std::mutex> lk(mu_);
        uint32_t& have = limits_[func];
        if (bytes <= have) return 0;
        const int status = set(bytes);
        if (status == 0) have = bytes;
        return status;
    }

private:
    std::mutex mu_;
    std::map<const void*, uint32_t> limits_;
};

}  // namespace fk
