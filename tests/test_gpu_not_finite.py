"""Infinite and NaN amplitudes and spectra stay, in the FP32 form, in the footprint
and the channel window of their particle: every other voxel has the value it has
without them.

Whole-number weights and amplitudes (sums below 2^24) make the finite part exact; what is not finite is w * s by IEEE rules (an infinity at a
zero weight of the footprint is a NaN), the same in any order of the sum."""

import numpy as np
import pytest

from martini_amd import _lib

pytestmark = pytest.mark.gpu

ODD = np.array([np.inf, -np.inf, np.nan], np.float32)
SHAPES = [(16, 16, 64), (8, 16, 128), (33, 47, 70), (21, 40, 200)]


def _insert(rec, desc):
    import torch

    pairs = _lib.count_pairs(rec, desc)
    d = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(desc.nx * desc.ny * desc.nc, dtype=torch.float32, device="cuda")
    ws = torch.full((_lib.workspace_bytes(desc, rec.size, pairs),), 255, dtype=torch.uint8,
                    device="cuda")
    _lib.insert(d, rec.size, pairs, desc, cube, ws, method="plain")
    return cube.cpu().numpy().reshape(desc.nx, desc.ny, desc.nc)


def _records(n, shape, rng, kind):
    nx, ny, nc = shape
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = rng.integers(-1, nx + 1, n), rng.integers(-1, ny + 1, n)
    r = rng.choice([0, 1, 2, 5], n, p=[0.4, 0.3, 0.2, 0.1])
    rec["r_kind"] = (r << 8) | kind
    rec["c_lo"] = rng.integers(0, nc, n)
    rec["c_hi"] = np.minimum(rec["c_lo"] + rng.integers(0, 30, n), nc - 1)
    rec["k0"] = np.arange(n)
    return rec, r


def _box(rec, r, k, shape):
    i0, i1 = max(rec["ix"][k] - r[k], 0), min(rec["ix"][k] + r[k], shape[0] - 1)
    j0, j1 = max(rec["iy"][k] - r[k], 0), min(rec["iy"][k] + r[k], shape[1] - 1)
    return slice(i0, i1 + 1), slice(j0, j1 + 1), slice(rec["c_lo"][k], rec["c_hi"][k] + 1)


@pytest.mark.parametrize("spectrum", [_lib.SPECTRUM_DIRAC, _lib.SPECTRUM_TABLE])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n", [1, 31, 70, 1000, 30000])
def test_whole_numbers(spectrum, shape, n):
    import torch

    rng = np.random.default_rng(n + shape[2])
    rec, r = _records(n, shape, rng, _lib.KERNEL_TABLE)
    bad = np.arange(n) % max(n // 7, 1) == n // 2 % max(n // 7, 1)  # some eight particles
    if spectrum == _lib.SPECTRUM_DIRAC:
        rec["amp"] = rng.integers(-8, 9, n)
        rec["amp"][bad] = rng.choice(ODD, bad.sum())
        spectra = np.repeat(rec["amp"][:, None], shape[2], 1)
    else:
        rec["amp"] = 1.0
        spectra = rng.integers(-8, 9, (n, shape[2])).astype(np.float32)
        hit = bad[:, None] & (rng.random(spectra.shape) < 0.3)
        spectra[hit] = rng.choice(ODD, hit.sum())
    want, offs, weights, at = np.zeros(shape), np.zeros(n, np.uint32), [np.zeros(1, np.float32)], 1
    with np.errstate(invalid="ignore"):
        for k in range(n):
            box = _box(rec, r, k, shape)
            size = [max(b.stop - b.start, 0) for b in box[:2]]
            offs[k] = at
            w = rng.integers(-4, 5, size).astype(np.float32)
            weights.append(w.ravel())
            at += w.size
            if w.size:
                want[box] += w.astype(float)[:, :, None] * spectra[k, box[2]]
    rec["h"] = offs.view(np.float32)
    weights = np.concatenate(weights)
    d_w, d_s = torch.from_numpy(weights).cuda(), torch.from_numpy(spectra).cuda()
    table = dict(spectra=d_s, spectra_ld=shape[2]) if spectrum == _lib.SPECTRUM_TABLE else {}
    desc = _lib.make_desc(*shape, spectrum, **table)
    desc.weights, desc.weights_n = d_w.data_ptr(), weights.size
    assert np.array_equal(_insert(rec, desc), want, equal_nan=True)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kind", [_lib.KERNEL_CUBIC, _lib.KERNEL_GAUSS, _lib.KERNEL_DIRAC])
@pytest.mark.parametrize("n", [40, 1000])
def test_gaussian_lines(shape, kind, n):
    """Against the same particles with the odd ones' amplitude zero, bit for bit."""
    rng = np.random.default_rng(n + kind)
    rec, r = _records(n, shape, rng, kind)
    rec["h"] = np.maximum(r, 0.5) + 0.3
    if kind != _lib.KERNEL_DIRAC:
        rec["fx"], rec["fy"] = rng.random(n), rng.random(n)
    rec["k0"] = (rec["c_lo"] + rec["c_hi"]) // 2
    rec["fu"], rec["s"] = rng.random(n), np.exp(rng.uniform(-3, 1.5, n))
    rec["amp"] = rng.uniform(0.5, 2.0, n)
    bad = rng.choice(n, 5, replace=False)
    without = rec.copy()
    without["amp"][bad] = 0.0
    rec["amp"][bad[:3]] = ODD
    rec["s"][bad[3]] = np.nan
    rec["fu"][bad[4]] = np.nan
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_GAUSS, ((3.0, 0.97),))
    inside = np.zeros(shape, bool)
    for k in bad:
        i, j, c = _box(rec, r, k, shape)
        inside[i.start + int(rec["fx"][k] > 0 and rec["ix"][k] - r[k] >= 0):i.stop,
               j.start + int(rec["fy"][k] > 0 and rec["iy"][k] - r[k] >= 0):j.stop, c] = True
    got = _insert(rec, desc)
    assert np.array_equal(got[~inside], _insert(without, desc)[~inside])
    assert np.all(np.isfinite(got[~inside]))
    # the particle's own pixel, if it lies in the cube (a footprint of half width zero
    # about a position off the pixel's centre is empty)
    for k in bad[(r[bad] > 0) | (kind == _lib.KERNEL_DIRAC)]:
        i, j = rec["ix"][k], rec["iy"][k]
        if 0 <= i < shape[0] and 0 <= j < shape[1]:
            assert not np.any(np.isfinite(got[i, j, rec["c_lo"][k]:rec["c_hi"][k] + 1]))
