"""The chunk loop of the batched fits (steppe_amd/csrc/chunks.hpp), compiled on its own: every
item once and in order within the limits, and smaller chunks where there is no room."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# items of size 1 + i % 3; arguments: n, most items, budget, room
PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include "chunks.hpp"

int main(int, char** v) {
    const std::size_t n = std::atoi(v[1]), most = std::atoi(v[2]), budget = std::atoi(v[3]), room = std::atoi(v[4]);
    auto size = [](std::size_t i) { return 1 + i % 3; };
    try {
        stp::for_chunks(n, most, budget, size,
            [&](std::size_t i0, std::size_t i1) {
                std::size_t total = 0;
                for (std::size_t i = i0; i < i1; ++i) total += size(i);
                if (total <= room) return true;
                if (i1 - i0 == 1) throw std::runtime_error("no room");
                std::printf("cut %zu %zu\n", i0, i1);
                return false;
            },
            [](std::size_t i0, std::size_t i1) { std::printf("run %zu %zu\n", i0, i1); });
    } catch (const std::runtime_error& e) {
        std::printf("%s\n", e.what());
    }
}
"""


@pytest.fixture(scope="module")
def chunks(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("chunks")
    (d / "chunks.cpp").write_text(PROGRAM)
    exe = str(d / "chunks")
    subprocess.run([gxx, "-std=c++20", "-I", os.path.join(ROOT, "steppe_amd", "csrc"), str(d / "chunks.cpp"), "-o",
                    exe], check=True)

    def run(n, most=1000, budget=1000, room=1000):
        out = subprocess.run([exe, *map(str, (n, most, budget, room))], check=True, capture_output=True, text=True,
                             timeout=20).stdout
        lines = [ln.split() for ln in out.split("\n") if ln]
        return ([(int(a), int(b)) for w, a, b in (x for x in lines if len(x) == 3) if w == "run"],
                sum(x[0] == "cut" for x in lines), ["no", "room"] in lines)
    return run


def _size(a, b):
    return sum(1 + i % 3 for i in range(a, b))


@pytest.mark.parametrize("n,most,budget", [(0, 5, 10), (1, 5, 10), (10, 1000, 1000), (10, 3, 1000), (100, 1000, 7),
                                           (100, 2, 7), (9, 1000, 1)])
def test_limits(chunks, n, most, budget):
    run, cut, full = chunks(n, most, budget)
    assert [i for a, b in run for i in range(a, b)] == list(range(n)) and not cut and not full
    for a, b in run:
        assert b - a <= most and (b - a == 1 or _size(a, b) <= budget)
        # and no smaller than they need be
        assert b == n or b - a == most or _size(a, b + 1) > budget


@pytest.mark.parametrize("room", [200, 100, 50, 13, 5, 3])
def test_less_room_than_the_budget(chunks, room):
    run, cut, full = chunks(100, room=room)
    assert [i for a, b in run for i in range(a, b)] == list(range(100)) and not full
    assert all(_size(a, b) <= room for a, b in run)
    assert cut == 0 if room >= _size(0, 100) else 1 <= cut <= 8


def test_an_item_without_room(chunks):
    run, cut, full = chunks(100, room=2)
    assert full and run == [(0, 1), (1, 2)]
