// Host threads for set-up work.
#pragma once
#include <exception>
#include <thread>
#include <vector>

namespace falcon {

// f(0) .. f(n - 1), each on a thread of its own (f(0) on the caller's).  Shares
// for which no thread can be started (a thread or memory limit) run on the
// caller's.  Returns with every share done and every thread joined; the first
// share's exception, in their order, is rethrown.
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
        for (int t = 1; t < n; t++) th.emplace_back(share, t);
    } catch (...) {
    }
    for (int t = (int)th.size() + 1; t < n; t++) share(t);
    if (n > 0) share(0);
    for (auto &x : th) x.join();
    for (auto &e : err)
        if (e) std::rethrow_exception(e);
}

}  // namespace falcon
