// gsd_lds_limit.h -- a kernel's limit of dynamic LDS, raised by its launcher.
// No HIP in here: `set` makes the runtime's call.
#pragma once
#include <atomic>
#include <cstddef>
#include <mutex>

namespace gsd {

// One per kernel (a static of its launcher).  The limit and what is known of
// it change together: threads whose launches need different sizes can neither
// lower it under another's nor take a size for set that is not yet.
class LdsLimit {
    std::mutex m_;
    std::atomic<size_t> have_{0};

public:
    // at least `lds` bytes from here on; set(bytes) returns 0 for success
    template <typename Set>
    auto raise(size_t lds, Set set) -> decltype(set(lds)) {
        if (lds <= have_.load(std::memory_order_acquire)) return {};
        const std::lock_guard<std::mutex> hold(m_);
        if (lds <= have_.load(std::memory_order_relaxed)) return {};
        const auto rc = set(lds);
        if (rc == decltype(rc){}) have_.store(lds, std::memory_order_release);
        return rc;
    }
};

}  // namespace gsd
