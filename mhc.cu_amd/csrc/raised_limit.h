// A per-device limit that may only grow, behind a setter that takes any value (host code, no HIP header needed).
#pragma once

#include <algorithm>
#include <atomic>
#include <mutex>

namespace mhc {

class RaisedLimit {
    static constexpr int kDevices = 64;
    std::mutex mu_;
    std::atomic<int> limit_[kDevices + 1] = {};  // the last one: devices beyond, whose limit is set on every call

public:
    // Makes sure that the limit of `device` is at least `want`; set(value) sets it and returns 0 on success.  The setter
    // runs under a lock and never with a smaller value than before: of two threads that ask for different values
    // at the same time, the one that sets last would otherwise take the other's limit back.
    template <class Set> auto raise(int device, int want, Set set) -> decltype(set(0)) {
        const bool known = device >= 0 && device < kDevices;
        std::atomic<int> &limit = limit_[known ? device : kDevices];
        if (known && limit.load(std::memory_order_acquire) >= want) return {};
        std::lock_guard<std::mutex> lock(mu_);
        const int have = limit.load(std::memory_order_relaxed);
        if (known && have >= want) return {};
        const int value = std::max(have, want);
        const auto status = set(value);
        if (status == decltype(set(0)){}) limit.store(value, std::memory_order_release);
        return status;
    }
};

}  // namespace mhc
