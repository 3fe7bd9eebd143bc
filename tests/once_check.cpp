// once_check.cpp -- TEST INFRASTRUCTURE ONLY: the once-per-process set-up of
// the engine's tables (3photons-rust_amd/csrc/tp_once.h) under threads, for
// tests/test_once.py.
//
//   g++ -O2 -std=c++17 -pthread -shared -fPIC -I<csrc> once_check.cpp
#include "tp_once.h"

#include <stdexcept>
#include <thread>
#include <vector>

// `threads` callers at once, `rounds` calls each, of a set-up that fails (every
// other time by a throw) its first `failures` times.  Returns the number of
// times it was made; *ok the calls that returned true, *early those that did so
// before it had been made.
extern "C" int tp_once_check(int threads, int rounds, int failures, int *ok, int *early)
{
    tpe::OnceDone once;
    int tries = 0, made = 0; // under the set-up's own lock
    std::atomic<int> good{0}, bad{0}, value{0};
    std::vector<std::thread> t;
    for (int k = 0; k < threads; ++k)
        t.emplace_back([&] {
            for (int i = 0; i < rounds; ++i) {
                bool done = false;
                try {
                    done = once.run([&] {
                        if (++tries <= failures) {
                            if (tries & 1)
                                throw std::runtime_error("set-up");
                            return false;
                        }
                        ++made;
                        value.store(1, std::memory_order_relaxed);
                        return true;
                    });
                } catch (const std::runtime_error &) {
                }
                if (done)
                    ++(value.load(std::memory_order_relaxed) ? good : bad);
            }
        });
    for (auto &x : t)
        x.join();
    *ok = good;
    *early = bad;
    return once.done() ? made : -made - 1;
}
