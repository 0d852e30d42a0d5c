"""Binning at the edges of its launch shapes: the emit groups (256 x 1, 1024 x 1
and 1024 x 4 particles), the radix tiles (1024, 4096 and 8192 pairs), one to
three radix passes, cells cut into many items, and pair capacities above and
below the count.

Records of the Dirac kernel and the Dirac line put `amp` into one pixel of one
channel, so with amp = 1 the cube is a histogram: whole numbers below 2^24,
exact in FP32 and in the split products, and equal to numpy's bincount.  A
particle misplaced, lost or taken twice by any stage changes it."""

import numpy as np
import pytest

from martini_amd import _lib

pytestmark = pytest.mark.gpu

# nx, ny, nc; cells of 16 x 16 x 64, or 8 x 16 x 128 from 128 channels on
CUBES = {"one_cell": (16, 16, 8), "few": (40, 33, 70), "wide": (70, 50, 300),
         "three_passes": (4096, 2304, 2)}


def _records(n, shape, spread, seed):
    """n point particles, the fraction 1 - spread of them in one pixel; every
    thirteenth has no channel and makes no pair."""
    rng = np.random.default_rng(seed)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    one = rng.random(n) >= spread
    for f, m in (("ix", shape[0]), ("iy", shape[1])):
        rec[f] = np.where(one, m // 2, rng.integers(0, m, n))
    c = np.where(one, shape[2] - 1, rng.integers(0, shape[2], n))
    rec["c_lo"] = rec["c_hi"] = c
    rec["c_lo"][::13], rec["c_hi"][::13] = 1, 0
    rec["r_kind"] = _lib.KERNEL_DIRAC
    rec["amp"] = 1.0
    flat = (rec["ix"].astype(np.int64) * shape[1] + rec["iy"]) * shape[2] + c
    return rec, np.bincount(flat[np.arange(n) % 13 != 0], minlength=int(np.prod(shape)))


def _insert(rec, shape, n_pairs, method, layout=False):
    import torch

    from martini_amd.insertion import layout_records

    desc = _lib.make_desc(*shape, _lib.SPECTRUM_DIRAC)
    d = torch.from_numpy(rec.view(np.uint8)).cuda()
    if layout:
        d = layout_records(d, method, shape[2])
    cube = torch.zeros(int(np.prod(shape)), dtype=torch.float32, device="cuda")
    ws = torch.full((_lib.workspace_bytes(desc, rec.size, n_pairs),), 255, dtype=torch.uint8,
                    device="cuda")
    _lib.insert(d, rec.size, n_pairs, desc, cube, ws, method=method)
    return cube.cpu().numpy(), _lib.status(desc, rec.size, n_pairs, ws)


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("cube", CUBES)
@pytest.mark.parametrize("n,spread", [
    (1, 1.0), (255, 0.5), (257, 1.0), (1112, 0.9), (65535, 1.0), (65537, 0.1), (141990, 1.0),
    (142000, 0.5), (524287, 0.02), (524289, 1.0), (1136000, 1.0),
])
def test_point_particles_are_counted(method, cube, n, spread):
    shape = CUBES[cube]
    if cube == "three_passes" and n < 65535:
        pytest.skip("the large cube at the larger sizes only")
    rec, want = _records(n, shape, spread, n + len(cube))
    pairs = int(want.sum())
    for cap, layout in ((pairs, False), (pairs + 5000, True)):
        got, (n_pairs, overflow, items, _) = _insert(rec, shape, cap, method, layout)
        assert n_pairs == pairs and not overflow and (items > 0) == (pairs > 0)
        assert np.array_equal(got, want)


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("n", [1000, 100_000, 600_000])
def test_too_small_a_capacity_leaves_the_cube(method, n):
    import torch

    shape = CUBES["few"]
    rec, want = _records(n, shape, 1.0, n)
    pairs = int(want.sum())
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_DIRAC)
    for cap in (pairs - 1, pairs // 2, 1, 0):
        d = torch.from_numpy(rec.view(np.uint8)).cuda()
        cube = torch.full((int(np.prod(shape)),), 3.0, device="cuda")
        ws = torch.empty(_lib.workspace_bytes(desc, n, cap), dtype=torch.uint8, device="cuda")
        with pytest.raises(_lib.MartiniLibError):
            _lib.insert(d, n, cap, desc, cube, ws, method=method)
        assert bool((cube == 3.0).all())
        assert _lib.status(desc, n, cap, ws)[:2] == (pairs, 1)


@pytest.mark.parametrize("method", ["plain", "mfma"])
def test_wide_footprints_are_counted(method):
    """Particles over many cells (written by a whole wave each) beside narrow
    ones: table weights of one make every pixel of a footprint count."""
    import torch

    shape, n = (120, 90, 130), 3000
    rng = np.random.default_rng(4)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = rng.integers(0, shape[0], n), rng.integers(0, shape[1], n)
    r = np.where(rng.random(n) < 0.1, rng.integers(10, 60, n), rng.integers(0, 3, n))
    rec["r_kind"] = (r << 8) | _lib.KERNEL_TABLE
    rec["c_lo"] = rng.integers(0, 100, n)
    rec["c_hi"] = rec["c_lo"] + rng.integers(0, 60, n)
    rec["amp"] = 1.0
    want = np.zeros(shape)
    offs, at = np.zeros(n, np.uint32), 0
    for k in range(n):
        i0, i1 = max(rec["ix"][k] - r[k], 0), min(rec["ix"][k] + r[k], shape[0] - 1)
        j0, j1 = max(rec["iy"][k] - r[k], 0), min(rec["iy"][k] + r[k], shape[1] - 1)
        offs[k] = at
        at += (i1 - i0 + 1) * (j1 - j0 + 1)
        want[i0:i1 + 1, j0:j1 + 1, rec["c_lo"][k]:min(rec["c_hi"][k], shape[2] - 1) + 1] += 1
    rec["h"] = offs.view(np.float32)
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_DIRAC)
    weights = torch.ones(at, dtype=torch.float32, device="cuda")
    desc.weights, desc.weights_n = weights.data_ptr(), at
    got, _ = _insert_desc(rec, shape, desc, method)
    assert np.array_equal(got.reshape(shape), want)


def _insert_desc(rec, shape, desc, method):
    import torch

    pairs = _lib.count_pairs(rec, desc)
    d = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(int(np.prod(shape)), dtype=torch.float32, device="cuda")
    ws = torch.empty(_lib.workspace_bytes(desc, rec.size, pairs), dtype=torch.uint8, device="cuda")
    _lib.insert(d, rec.size, pairs, desc, cube, ws, method=method)
    return cube.cpu().numpy(), pairs
