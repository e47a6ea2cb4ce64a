// Something that has to be done once on every device of a process (a kernel attribute), by whichever thread comes
// first, and again by the next one where it did not succeed.
#pragma once

#include <atomic>
#include <cstdint>

namespace moe355 {

class OncePerDevice {
    std::atomic<uint64_t> done{0};  // a bit per device; devices past the 64th are asked every time

public:
    template <typename F>
    bool operator()(int device, F step)
    {
        const uint64_t bit = device >= 0 && device < 64 ? 1ull << device : 0;
        if (done.load(std::memory_order_acquire) & bit) return true;
        if (!step()) return false;
        done.fetch_or(bit, std::memory_order_release);
        return true;
    }
};

}  // namespace moe355
