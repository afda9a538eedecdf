"""The step-wise path's working buffers (csrc/buffer_set.hpp) under a memory limit: compiled for the host with
an allocator that counts and refuses."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = r"""
#include <stdio.h>
#include <stdlib.h>
#include <map>
#include "buffer_set.hpp"
static size_t limit, used;
static int allocs, frees;
static std::map<void*, size_t> live;
static void* take(size_t b) {
    if (used + b > limit) return nullptr;
    void* q = malloc(1);
    live[q] = b; used += b; ++allocs;
    return q;
}
static void give(void* q) {
    if (!live.count(q)) { printf("free of a foreign pointer\n"); exit(1); }
    used -= live[q]; live.erase(q); free(q); ++frees;
}
int main(int argc, char** argv) {
    limit = (size_t)atol(argv[1]);
    pa::BufferSet s;
    for (int i = 2; i + 2 < argc; i += 3) {
        allocs = frees = 0;
        const int got = s.get((size_t)atol(argv[i]), atoi(argv[i + 1]), atoi(argv[i + 2]), take, give);
        for (int k = 0; k < got; ++k)
            if (!live.count(s.p[k]) || live[s.p[k]] < (size_t)atol(argv[i])) { printf("buffer %d is not held\n", k); return 1; }
        printf("%d %d %d %zu\n", got, allocs, frees, live.size());
    }
    s.clear(give);
    printf("%zu\n", used);
    return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("buffers")
    (d / "driver.cpp").write_text(SOURCE)
    inc = os.path.join(os.path.dirname(HERE), "parament_amd", "csrc")
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", inc, "-o", str(d / "driver"), str(d / "driver.cpp")], check=True)

    def run(limit, *calls):
        """(got, allocations, frees, held) of each call (bytes, need, want)."""
        args = [str(limit)] + [str(v) for c in calls for v in c]
        out = subprocess.run([str(d / "driver"), *args], check=True, capture_output=True, text=True).stdout.split("\n")
        assert out[len(calls)] == "0"   # everything is given back at the end
        return [tuple(int(v) for v in line.split()) for line in out[:len(calls)]]
    return run


@pytest.mark.parametrize("need, want", [(3, 4), (3, 5), (4, 5)])
def test_repeated_call_without_room_allocates_nothing(driver, need, want):
    """Memory for need buffers but not for want: the first call takes need, later ones the same buffers."""
    for fits in range(need, want):
        first, *later = driver(100 * fits + 50, *[(100, need, want)] * 4)
        assert first[0] == need and first[3] == need
        assert later == [(need, 0, 0, need)] * 3


def test_held_buffers_survive_a_failed_extension(driver):
    """Three buffers held from a call that needed no more: a call that wants five keeps them and adds none."""
    assert driver(450, (100, 3, 3), (100, 3, 5), (100, 3, 5), (100, 3, 3)) == [
        (3, 3, 0, 3), (3, 1, 1, 3), (3, 0, 0, 3), (3, 0, 0, 3)]
    # four fitted: a call that wants four gets them
    assert driver(450, (100, 3, 5), (100, 3, 4), (100, 3, 5)) == [(3, 4, 1, 3), (4, 1, 0, 4), (3, 0, 0, 4)]


def test_growth_and_failure(driver):
    assert driver(10000, (100, 3, 5), (200, 3, 4), (200, 3, 5), (150, 4, 4)) == [
        (5, 5, 0, 5), (4, 4, 5, 4), (5, 1, 0, 5), (4, 0, 0, 5)]
    # not even need: nothing is held, and a smaller call takes its own
    assert driver(250, (100, 3, 5), (50, 3, 4)) == [(0, 2, 2, 0), (4, 4, 0, 4)]
    # buffers larger than asked for, of which need do not fit, make way for smaller ones
    assert driver(1000, (300, 3, 3), (200, 4, 5)) == [(3, 3, 0, 3), (5, 5, 3, 5)]
