// tp_once.h -- a set-up that is made once for all threads, and tried again by
// the next caller as long as it fails (std::call_once takes any return for
// done, so one failure would be kept for the life of the process).
#pragma once

#include <atomic>
#include <mutex>

namespace tpe {

class OnceDone {
    std::mutex m;
    std::atomic<bool> ready{false};

public:
    // True once f() has returned true, here or before; a throw leaves it undone.
    template <class F> bool run(F &&f)
    {
        if (ready.load(std::memory_order_acquire))
            return true;
        const std::lock_guard<std::mutex> lock(m);
        if (!ready.load(std::memory_order_relaxed) && f())
            ready.store(true, std::memory_order_release);
        return ready.load(std::memory_order_relaxed);
    }
    bool done() const { return ready.load(std::memory_order_acquire); }
};

} // namespace tpe
