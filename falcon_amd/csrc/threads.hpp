// Host threads for set-up work.
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace falcon {

// f(0) .. f(n - 1), each on a thread of its own, or with caller the first on the
// caller's (a thread less to start; not for shares that allocate: on the main
// heap the ghost tables of 648 blocks took 68 instead of 62 ms on 8 cores).
// Shares for which no thread can be started (a thread or memory limit) run on the
// caller's, one alone too.  Returns with every share done and every thread joined;
// the first share's exception, in their order, is rethrown.
template <class F>
void run_shares(int n, F &&f, bool caller = false) {
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
    const int first = caller ? 1 : 0;
    try {
        for (int t = first; t < n && n > 1; t++) th.emplace_back(share, t);
    } catch (...) {
    }
    for (int t = first + (int)th.size(); t < n; t++) share(t);
    if (caller && n > 0) share(0);
    for (auto &x : th) x.join();
    for (auto &e : err)
        if (e) std::rethrow_exception(e);
}

}  // namespace falcon
