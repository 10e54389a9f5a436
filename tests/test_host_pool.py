"""The bounded host loop (steppe_amd/csrc/host_pool.hpp), compiled on its own: every index once
and in its place for thousands of items, at most 16 threads however many items there are, and
the exception of the smallest index on the calling thread."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <chrono>
#include <cstdio>
#include <set>
#include <stdexcept>
#include <string>
#include "host_pool.hpp"

int main() {
    for (std::size_t n : {0, 1, 2, 15, 16, 17, 5000}) {
        std::vector<int> hits(n, 0);
        std::mutex m;
        std::set<std::thread::id> ids;
        stp::for_each_index(n, [&](std::size_t i) {
            ++hits[i];
            if (n <= 17) std::this_thread::sleep_for(std::chrono::milliseconds(5));
            const std::lock_guard<std::mutex> lock(m);
            ids.insert(std::this_thread::get_id());
        });
        int ok = 1;
        for (int h : hits) ok = ok && h == 1;
        std::printf("%zu %d %zu\n", n, ok, ids.size());
    }
    for (std::size_t bad : {0, 700, 4999}) {
        std::string got = "none";
        try {
            stp::for_each_index(5000, [&](std::size_t i) {
                if (i >= bad) throw std::runtime_error(std::to_string(i));
            });
        } catch (const std::runtime_error& e) {
            got = e.what();
        }
        std::printf("%zu %s\n", bad, got.c_str());
    }
}
"""


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("pool")
    (d / "pool.cpp").write_text(PROGRAM)
    exe = str(d / "pool")
    subprocess.run([gxx, "-std=c++20", "-O2", "-pthread", "-I", os.path.join(ROOT, "steppe_amd", "csrc"),
                    str(d / "pool.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=60).stdout
    return [ln.split() for ln in out.split("\n") if ln]


def test_every_index_once_on_few_threads(lines):
    counts = {int(n): (ok, int(t)) for n, ok, t in lines[:7]}
    assert all(ok == "1" for ok, _ in counts.values())
    assert all(t <= min(16, n) for n, (_, t) in counts.items())


def test_first_exception_reaches_the_caller(lines):
    assert [(int(b), g) for b, g in lines[7:]] == [(0, "0"), (700, "700"), (4999, "4999")]
