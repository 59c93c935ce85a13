"""Host threads of the set-up (threads.hpp): a process that cannot start more
threads, or a share that fails, gets a result or an error, never an abort."""
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "falcon_amd", "csrc")

# pthread_create of the program itself: starts `left` threads, then none
MAIN = r"""
#include <dlfcn.h>
#include <pthread.h>
#include <atomic>
#include <cerrno>
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include "layout.hpp"
#include "threads.hpp"

static std::atomic<int> left{1 << 30};
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *p) {
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static Fn real = (Fn)dlsym(RTLD_NEXT, "pthread_create");
    return left-- > 0 ? real(t, a, f, p) : EAGAIN;
}
using namespace falcon;

static int shares(int n, int threads, int bad, bool caller) {
    left = threads;
    std::vector<std::atomic<int>> done(n);
    int err = -1;
    try {
        run_shares(n, [&](int t) {
            done[t]++;
            if (bad >= 0 && t >= bad) throw std::runtime_error(std::to_string(t));
        }, caller);
    } catch (const std::exception &e) {
        err = std::stoi(e.what());
    }
    for (auto &d : done)
        if (d != 1) return 1;
    return err == (bad < n ? bad : -1) ? 0 : 2;
}

static std::vector<GhostEntry> ghosts(int threads) {
    left = threads;
    Layout lay;
    lay.tree.init(4, 4, 4, 2, 4.9e10, 6.7e10);
    lay.tree.divide_all(1, 2, 6);
    lay.tree.label();
    lay.build(8);
    return lay.ghosts;
}

int main() {
    for (int n : {0, 1, 2, 8})
        for (int threads : {0, 1, 3, 100})
            for (int bad : {-1, 0, 1, 5})
                for (bool caller : {false, true}) {
                    const int e = shares(n, threads, bad, caller);
                    if (e) {
                        std::printf("shares n=%d threads=%d bad=%d caller=%d: %d\n", n, threads, bad, caller, e);
                        return 1;
                    }
                }
    const auto a = ghosts(1 << 30);
    for (int threads : {0, 3}) {
        const auto b = ghosts(threads);
        if (a.size() != b.size() || a.empty()) return 2;
        for (size_t q = 0; q < a.size(); q++)
            if (a[q].recv_block != b[q].recv_block || a[q].donor != b[q].donor || a[q].i0 != b[q].i0 ||
                std::memcmp(a[q].w, b[q].w, sizeof(a[q].w))) return 3;
    }
    std::puts("ok");
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("threads")
    (d / "main.cpp").write_text(MAIN)
    exe = str(d / "main")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(d / "main.cpp"), os.path.join(CSRC, "layout.cpp"),
                    "-o", exe, "-lpthread", "-ldl"], check=True)
    return exe


def test_no_more_threads_and_failing_shares(program):
    r = subprocess.run([program], capture_output=True, text=True, timeout=60)
    assert (r.returncode, r.stdout.strip()) == (0, "ok"), (r.returncode, r.stdout, r.stderr)
