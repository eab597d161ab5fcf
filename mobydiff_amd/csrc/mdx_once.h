// mdx_once.h -- an action that has to run once on every device (host code, no HIP types).
#pragma once

#include <atomic>

namespace mdx {

// Runs `f` (0: success) for device `dev` unless it has succeeded there before; a failure is returned
// and tried again by the next call.  Callable from any thread: two first calls may both run `f`,
// which has to be harmless to repeat.  Devices past the table run it every time.
class OncePerDevice {
    static constexpr int N = 64;
    std::atomic<bool> done_[N] = {};

public:
    template <typename F> auto run(int dev, F f) -> decltype(f()) {
        const bool known = dev >= 0 && dev < N;
        if (known && done_[dev].load(std::memory_order_acquire)) return decltype(f())(0);
        const auto e = f();
        if (known && e == decltype(f())(0)) done_[dev].store(true, std::memory_order_release);
        return e;
    }
};

}  // namespace mdx
