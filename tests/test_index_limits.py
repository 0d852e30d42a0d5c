"""Index arithmetic at the limits that the library accepts (pair counts below
2^31, cubes of up to 2^21 cells) and of loops whose ends matter, on the CPU: the
functions that the kernels use, compiled for the host."""

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

// Total of `n` counts of `each` pairs, as a wave sums them (32 bits a part).
static unsigned long long total(int n, uint32_t each) {
    PairSum sum;
    for (int k = 0; k < n; ++k) {
        const PairSum one(each);
        sum.upper += one.upper;
        sum.lower += one.lower;
    }
    return sum.total();
}

// Whether the steps of a beam pass take every row of the cube that feeds an output
// of [l0, l0 + 32), and at most two steps more than those rows need.
static bool line_steps(int l0, int L, int k) {
    const int S = (k + 15 + 3) / 4, all = S + 4;
    const LineSteps s(l0, L, k, all);
    int lowest = L, highest = -1;
    for (int l = l0; l < l0 + 32 && l < L; ++l)
        for (int a = 0; a < k; ++a) {
            const int m = l + k / 2 - a;
            if (m < 0 || m >= L) continue;
            lowest = m < lowest ? m : lowest;
            highest = m > highest ? m : highest;
        }
    return s.first >= 0 && s.last <= all && s.m0 + 4 * s.first <= lowest &&
           s.m0 + 4 * s.last > highest && s.last - s.first <= (highest - lowest) / 4 + 10 &&
           s.last - s.first <= L / 4 + 2;
}

// The most partial tiles that `pairs` pairs in `cells` cells can need: k cells of one
// pair more than an item, the rest of the pairs in whole items of the last of them.
static long worst_tiles(long pairs, long cells, int len) {
    long most = 0;
    for (long k = 1; k <= cells && k * (len + 1) <= pairs; ++k) {
        const long rest = pairs - (k - 1) * (len + 1);
        const long tiles = 2 * (k - 1) + (rest + len - 1) / len;
        most = tiles > most ? tiles : most;
    }
    return most;
}

int main(int argc, char** argv) {
    if (argc == 3 && argv[1][0] == 'F') {
        const long tiles = atol(argv[2]);
        for (int ny = 1; ny <= 32767; ++ny) {
            const int rows = fits_rows(tiles, ny);
            const long groups = tiles * ((ny + rows - 1) / rows);
            if (rows < 1 || rows > FITS_MAX_ROWS) return printf("%d rows\n", rows), 1;
            // one more for each tile's remainder
            if (rows < FITS_MAX_ROWS && groups > FITS_GROUPS + tiles) return printf("%d: %ld groups\n", ny, groups), 1;
        }
        return 0;
    }
    if (argc == 3 && argv[1][0] == 'T') {
        const long cells = atol(argv[2]);
        for (long pairs = 0; pairs < 40000000; pairs = pairs * 21 / 20 + 1) {
            const int len = item_length(pairs);
            const long most = worst_tiles(pairs, cells, len), room = partial_tiles_max(pairs, len, cells);
            if (room < most || room > most + 1) return printf("%ld pairs: %ld, room %ld\n", pairs, most, room), 1;
        }
        return 0;
    }
    if (argc == 3 && argv[1][0] == 'L') {
        const int L = atoi(argv[2]);
        for (int k = 1; k < 4096; k = k < 130 ? k + 2 : k * 3 / 2 | 1)
            for (int l0 = 0; l0 < L; l0 += 32)
                if (!line_steps(l0, L, k)) return printf("%d taps, output %d\n", k, l0), 1;
        return 0;
    }
    if (argc == 2) return printf("%llu %llu\n", total(16, atol(argv[1])), total(64, atol(argv[1]))), 0;
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
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("index")
    src, exe = d / "index.hip", d / "index"
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
def test_items_visit_each_chunk_of_their_cell_once(program, start, end):
    r = subprocess.run([str(program), str(start), str(end)], capture_output=True, text=True,
                       timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("each", [0, 1, 64, 64 * 4096, 2**26 - 1, 2**26, 64 * (2**21 - 1)])
def test_group_pair_totals_do_not_wrap(program, each):
    """A wave's 64 particles make up to 64 (2^21 - 1) pairs; groups of 16 waves, and of 16 in 4 rounds."""
    r = subprocess.run([str(program), str(each)], capture_output=True, text=True, check=True)
    assert [int(v) for v in r.stdout.split()] == [16 * each, 64 * each]


@pytest.mark.parametrize("tiles", [1, 2, 3, 10, 100, 1000])
def test_fits_work_groups(program, tiles):
    r = subprocess.run([str(program), "F", str(tiles)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("cells", [1, 2, 7, 100, 512, 4096, 100000])
def test_room_for_partial_tiles(program, cells):
    """What the worst split of the pairs over the cells needs, and one more at most."""
    r = subprocess.run([str(program), "T", str(cells)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.parametrize("length", [1, 2, 3, 4, 5, 15, 16, 31, 32, 33, 64, 65, 97, 300])
def test_beam_steps_reach_the_cube(program, length):
    r = subprocess.run([str(program), "L", str(length)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4096, 2**19, 2**19 + 4096])
def test_an_undercounted_capacity_is_refused(n):
    """Particles that each cover a whole 16384 x 16384 map, 2^20 cells: from 2^19
    particles on, a group of 4096 makes 2^32 pairs.  Nothing is written past the
    workspace and the overflow is reported."""
    import numpy as np
    import torch

    from martini_amd import _lib

    desc = _lib.make_desc(16384, 16384, 64, _lib.SPECTRUM_GAUSS)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"] = rec["iy"] = 8192
    rec["h"], rec["r_kind"] = 20000.0, (16384 << 8) | _lib.KERNEL_CUBIC
    rec["c_hi"], rec["s"], rec["amp"] = 63, 0.1, 1.0
    assert _lib.count_pairs(rec[:2], desc) == 2 << 20
    for cap in (0, 1000):
        need = _lib.workspace_bytes(desc, n, cap)
        whole = torch.full((need + (1 << 20),), 0xA5, dtype=torch.uint8, device="cuda")
        ws = whole[:need]
        d = torch.from_numpy(rec.view(np.uint8)).cuda()
        _lib.bin(d, n, cap, desc, ws)
        pairs, overflow, items, _ = _lib.status(desc, n, cap, ws)
        assert (pairs, overflow, items) == ((n << 20) & 0xFFFFFFFF, 1, 0)
        assert bool((whole[need:] == 0xA5).all())
