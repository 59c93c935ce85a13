// Host threads for set-up work.
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace falcon {

// f(0) .. f(n - 1), each on a thread of its own.  Shares for which no thread can be
// started (a thread or memory limit) run on the caller's, one alone too.  Returns
// with every share done and every thread joined; the first share's exception, in
// their order, is rethrown.  (A share on the caller's thread as a rule: the ghost
// tables of 648 blocks 62 -> 68 ms on 8 cores, its allocations being the main
// heap's.)
template <class F>
void run_shares(int n, F &&f) {
    std::vector<std::exception_ptr> err(n);
    std::vector<std::thread> th;
    th.reserve(n);
    auto share = [&](int t) {
        try {
            f(t);
        } catch (...) {
            err[t] = std::current_exception();
        }
    };
    try {
        for (int t = 0; t < n && n > 1; t++) th.emplace_back(share, t);
    } catch (...) {
    }
    for (int t = (int)th.size(); t < n; t++) share(t);
    for (auto &x : th) x.join();
    for (auto &e : err)
        if (e) std::rethrow_exception(e);
}

}  // namespace falcon
