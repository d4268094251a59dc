// once.h - an action that has to be taken once on every device.
#pragma once

#include <atomic>
#include <cstdint>

namespace lstk {

// Runs `act` unless it has succeeded on `device` before (`done`: a bit per device; devices past 63 run it every time).
// Returns its result, 0 meaning success. Threads that meet here for the first time may each run it.
template <typename F>
inline auto once_per_device(std::atomic<uint64_t> &done, int device, F &&act) -> decltype(act()) {
    const uint64_t bit = device >= 0 && device < 64 ? uint64_t(1) << device : 0;
    if (done.load(std::memory_order_acquire) & bit) return decltype(act())(0);
    const auto rc = act();
    if (rc == decltype(act())(0)) done.fetch_or(bit, std::memory_order_release);
    return rc;
}

}  // namespace lstk
