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
