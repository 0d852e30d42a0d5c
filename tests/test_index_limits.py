"""Index arithmetic at the limits that the library accepts (pair counts below
2^31, cubes of up to 2^21 cells), on the CPU: the functions that the kernels
use, compiled for the host."""

import subprocess

import pytest

from martini_amd import build_native

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "mi_internal.h"
#include "mi_tile.h"

using namespace mi;

// Chunks of item q of n, or -1 if the walk leaves the cell or does not end.
static long walk(long start, long end, int q, int n) {
    ItemWalk w((uint32_t)start, (uint32_t)end, Item{0, q, n, -1}, KC);
    long seen = 0;
    for (; w.more(); w.next(), ++seen)
        if (w.at() != start + (q + seen * n) * KC || w.at() >= end || seen > (1 << 20)) return -1;
    return seen;
}

int main(int argc, char** argv) {
    const long start = atol(argv[1]), end = atol(argv[2]);
    const int n = (int)((end - start + ITEM_MAX - 1) / ITEM_MAX);
    long chunks = 0;
    for (int q = 0; q < n; ++q) {
        const long seen = walk(start, end, q, n);
        if (seen < 0) return printf("item %d of %d\n", q, n), 1;
        chunks += seen;
    }
    if (chunks != (end - start + KC - 1) / KC) return printf("%ld chunks\n", chunks), 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def walk_items(tmp_path_factory):
    d = tmp_path_factory.mktemp("walk")
    src, exe = d / "walk.hip", d / "walk"
    src.write_text(PROGRAM)
    subprocess.run([build_native.HIPCC, "--offload-host-only", "-O1", "-std=c++17",
                    "-I", build_native.CSRC, str(src), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("start,end", [
    (0, 2**31 - 1),                    # every pair in one cell
    (0, 2**31 - 2**24), (0, 2130000000),
    (2**31 - 100, 2**31 - 1), (2**31 - 1000000, 2**31 - 1), (2**30, 2**31 - 7),
    (5, 6), (0, 32), (7, 4103), (7, 4104), (1000, 50000),
])
def test_items_visit_each_chunk_of_their_cell_once(walk_items, start, end):
    r = subprocess.run([str(walk_items), str(start), str(end)], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout
