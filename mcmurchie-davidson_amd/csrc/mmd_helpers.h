// A few host threads for the length of a scope.
#pragma once
#include <thread>

namespace mmd {

constexpr int HELPERS = 4;

inline int helper_count()
{
    const int cpus = (int)std::thread::hardware_concurrency();
    return cpus <= 2 ? 1 : (cpus - 1 < HELPERS ? cpus - 1 : HELPERS);
}

// Helper threads that run f until it returns; joined on destruction.  n of
// them could be started, none included: a caller that goes on without needs no
// exception, and one that left the constructor would end the process with the
// threads that had been started.
struct Helpers {
    std::thread t[HELPERS];
    int n = 0;
    template <class F>
    explicit Helpers(F f)
    {
        const int want = helper_count();
        try {
            for (; n < want; ++n) t[n] = std::thread(f);
        } catch (...) {   // out of threads or of memory
        }
    }
    ~Helpers() { join(); }
    void join()
    {
        for (int i = 0; i < n; ++i) t[i].join();
        n = 0;
    }
};

}  // namespace mmd
