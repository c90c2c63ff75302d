"""How a copy is divided among threads (share.h): compiled with the host compiler and run here."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def compiled(tmp_path, source):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "qip_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    return lambda *args: subprocess.run([str(exe), *map(str, args)], check=True, capture_output=True, text=True, timeout=60).stdout


@pytest.fixture(scope="module")
def shares(tmp_path_factory):
    run = compiled(tmp_path_factory.mktemp("shares"), """
#include "share.h"
#include <cstdio>
#include <cstdlib>
int main(int n, char **v) {
    for (int i = 1; i < n; ++i) {
        const auto s = qipgpu::shares_of(strtoull(v[i], nullptr, 10));
        printf("%d %zu %d\\n", s.count, s.each, qipgpu::kCopyThreads);
    }
}
""")
    return lambda sizes: [tuple(map(int, line.split())) for line in run(*sizes).splitlines()]


def test_shares_cover_a_copy_with_no_more_than_a_thread_each(shares):
    mib = 2 ** 20
    sizes = sorted({max(1, b + d) for m in (0, 1, 4, 8, 12, 15, 16, 17, 20, 32, 63, 64, 4096) for b in (m * mib,)
                    for d in (-4097, -3, -1, 0, 1, 2, 3, 4, 4097, mib // 2)})
    for size, (count, each, threads) in zip(sizes, shares(sizes)):
        assert each % mib == 0
        assert 1 <= count <= threads, (size, count, each)
        assert (count - 1) * each < size <= count * each, (size, count, each)
        assert count == 1 or size >= 8 * mib


def test_a_share_whose_helper_comes_late_is_the_callers(tmp_path):
    """Helpers that begin at once, only after the caller has returned, or not at all: every share is worked on once,
    before the call returns, and nothing of the caller's is touched after it."""
    run = compiled(tmp_path, """
#include "share.h"
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <new>
#include <thread>
#include <vector>

static std::vector<std::function<void()>> later;
static int mode = 0;

struct Helper {     // mode 1: begins at once; 2: after the caller has returned; 3: cannot be started; 4: every other one
    bool runs = false;
    size_t at = 0;
    Helper() = default;
    template <typename F> explicit Helper(F f) : runs(true) {
        const int m = mode < 4 ? mode : later.size() % 2 ? 1 : 2;
        if (m == 3) throw std::bad_alloc();
        if (m == 1) f();
        at = later.size();
        later.push_back(m == 1 ? std::function<void()>() : std::function<void()>(f));
    }
    Helper &operator=(Helper &&o) {
        runs = o.runs;
        at = o.at;
        o.runs = false;
        return *this;
    }
    ~Helper() { if (runs) abort(); }
    bool joinable() const { return runs; }
    void join() { if (!runs || later[at]) abort(); runs = false; }       // would wait for ever
    void detach() { if (!runs) abort(); runs = false; }
};

struct Work {
    int count[qipgpu::kCopyThreads] = {};
    bool over = false;
    void operator()(int i) { if (over) abort(); ++count[i]; }
};

int main() {
    for (mode = 1; mode <= 4; ++mode)
        for (int n = 1; n <= qipgpu::kCopyThreads; ++n) {
            later.clear();
            Work w;
            qipgpu::run_shares<Helper>(n, w);
            w.over = true;
            for (auto &f : later) if (f) f();
            for (int i = 0; i < qipgpu::kCopyThreads; ++i) if (w.count[i] != (i < n)) return 10 * mode + n;
        }
    for (int k = 0; k < 2000; ++k) {
        std::atomic<int> count[qipgpu::kCopyThreads] = {};
        auto w = [&count](int i) { ++count[i]; };
        qipgpu::run_shares<std::thread>(1 + k % qipgpu::kCopyThreads, w);
        for (int i = 0; i < qipgpu::kCopyThreads; ++i) if (count[i] != (i <= k % qipgpu::kCopyThreads)) return 1;
    }
    puts("whole");
}
""")
    assert run() == "whole\n"
