"""The gather's products against an FP64 sum, both forms, at the edges of its
chunks (32 particles), pairs of chunks and tiles.

Table kernels and table spectra give every (particle, pixel, channel) product
freely chosen factors, so what is tested is the contraction alone: operand
slots, the skips by row, block and group of four particles, and the clearing
between chunks.  With whole-number factors (exact in BF16, sums below 2^24)
both forms are exact; with real ones an FP32 sum of m terms of magnitude sum A
is off by at most (m + 1) 2^-24 A."""

import numpy as np
import pytest

from martini_amd import _lib

pytestmark = pytest.mark.gpu


def _case(n, shape, spread, seed, whole):
    rng = np.random.default_rng(seed)
    nx, ny, nc = shape
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"] = nx // 2 + rng.integers(-spread, spread + 1, n)
    rec["iy"] = ny // 2 + rng.integers(-spread, spread + 1, n)
    r = rng.choice([0, 1, 3, 9], n, p=[0.3, 0.3, 0.3, 0.1])
    rec["r_kind"] = (r << 8) | _lib.KERNEL_TABLE
    rec["c_lo"] = rng.integers(0, nc, n)
    rec["c_hi"] = np.minimum(rec["c_lo"] + rng.integers(0, 40, n), nc - 1)
    rec["k0"] = np.arange(n)
    rec["amp"] = 1.0
    if whole:
        spectra = rng.integers(-100, 101, (n, nc)).astype(np.float32)
    else:
        spectra = (rng.normal(size=(n, nc)) * 10.0 ** rng.uniform(-3, 3, (n, 1))).astype(np.float32)
    want, mag, terms = np.zeros(shape), np.zeros(shape), np.zeros(shape)
    offs, weights, at = np.zeros(n, np.uint32), [], 0
    for k in range(n):
        i0, i1 = max(rec["ix"][k] - r[k], 0), min(rec["ix"][k] + r[k], nx - 1)
        j0, j1 = max(rec["iy"][k] - r[k], 0), min(rec["iy"][k] + r[k], ny - 1)
        offs[k] = at
        if i0 > i1 or j0 > j1:
            continue
        size = (i1 - i0 + 1, j1 - j0 + 1)
        w = (rng.integers(-16, 17, size) if whole else rng.normal(size=size)).astype(np.float32)
        weights.append(w.ravel())
        at += w.size
        c = slice(rec["c_lo"][k], rec["c_hi"][k] + 1)
        term = w.astype(float)[:, :, None] * spectra[k, c].astype(float)
        box = (slice(i0, i1 + 1), slice(j0, j1 + 1), c)
        want[box] += term
        mag[box] += np.abs(term)
        terms[box] += 1
    rec["h"] = offs.view(np.float32)
    return rec, spectra, np.concatenate(weights), want, mag, terms


@pytest.mark.parametrize("method,whole", [("plain", False), ("plain", True), ("mfma", True)])
@pytest.mark.parametrize("shape,spread", [((16, 16, 64), 6), ((33, 47, 70), 15),
                                          ((8, 16, 128), 5), ((21, 40, 200), 12)])
@pytest.mark.parametrize("n", [1, 3, 31, 32, 33, 63, 64, 65, 97, 129, 1000])
def test_products(method, whole, shape, spread, n):
    import torch

    rec, spectra, weights, want, mag, terms = _case(n, shape, spread, n + shape[2], whole)
    d_s, d_w = torch.from_numpy(spectra).cuda(), torch.from_numpy(weights).cuda()
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_TABLE, spectra=d_s, spectra_ld=shape[2])
    desc.weights, desc.weights_n = d_w.data_ptr(), weights.size
    pairs = _lib.count_pairs(rec, desc)
    d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(want.size, dtype=torch.float32, device="cuda")
    ws = torch.full((_lib.workspace_bytes(desc, n, pairs),), 255, dtype=torch.uint8, device="cuda")
    _lib.insert(d_rec, n, pairs, desc, cube, ws, method=method)
    got = cube.cpu().numpy().reshape(shape).astype(float)
    if whole:
        assert np.array_equal(got, want)
        return
    assert np.all(got[terms == 0] == 0.0)
    worst = np.max(np.abs(got - want) - (terms + 1) * 2.0**-24 * mag)
    assert worst <= 0.0, worst


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("shape", [(16, 16, 64), (8, 16, 128)])
@pytest.mark.parametrize("n", [24577, 50001, 74015, 99000, 124033, 172800, 600001])
def test_long_items(method, shape, n):
    """One cell whose work items hold 2 to 9 chunks, over the edges of the chunks
    staged together: one pixel and one of 64 spectra per particle, whole numbers, so
    the cube is exact (sums below 2^24)."""
    import torch

    rng = np.random.default_rng(n)
    nx, ny, nc = shape
    rows = 64
    spectra = rng.integers(-8, 9, (rows, nc)).astype(np.float32)
    lo = rng.integers(0, nc, rows)
    hi = np.minimum(lo + rng.integers(0, 40, rows), nc - 1)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = rng.integers(0, nx, n), rng.integers(0, ny, n)
    rec["r_kind"] = _lib.KERNEL_TABLE
    rec["h"] = np.arange(n, dtype=np.uint32).view(np.float32)
    rec["k0"] = rng.integers(0, rows, n)
    rec["c_lo"], rec["c_hi"] = lo[rec["k0"]], hi[rec["k0"]]
    rec["amp"] = 1.0
    weights = rng.integers(-4, 5, n).astype(np.float32)
    sums = np.zeros((nx * ny, rows))
    np.add.at(sums, (rec["ix"] * ny + rec["iy"], rec["k0"]), weights)
    c = np.arange(nc)
    inside = (c >= lo[:, None]) & (c <= hi[:, None])
    want = (sums @ (spectra * inside)).reshape(shape)
    d_s, d_w = torch.from_numpy(spectra).cuda(), torch.from_numpy(weights).cuda()
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_TABLE, spectra=d_s, spectra_ld=nc)
    desc.weights, desc.weights_n = d_w.data_ptr(), n
    pairs = _lib.count_pairs(rec, desc)
    assert pairs == n
    d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(want.size, dtype=torch.float32, device="cuda")
    ws = torch.full((_lib.workspace_bytes(desc, n, pairs),), 255, dtype=torch.uint8, device="cuda")
    _lib.insert(d_rec, n, pairs, desc, cube, ws, method=method)
    assert np.array_equal(cube.cpu().numpy().reshape(shape), want)


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("shape", [(16, 16, 64), (8, 16, 128)])
@pytest.mark.parametrize("widths", [(0.2, 0.5), (0.50001, 1.0), (1.0, 40.0), (0.2, 8.0)])
def test_lines(method, shape, widths):
    """Gaussian lines from narrow to far wider channels than lines, a pixel and a
    particle each (weight 1), against FP64.

    Per edge x of a wide channel (s > 1/2) erf or erfc, whichever is the smaller,
    has a relative error of at most 10 * 2^-24 (9 Horner steps, a reciprocal, an
    exponential and products) and x one of 2.5 * 2^-24, whose effect is at most
    max(x exp(-x^2)) * 2 / sqrt(pi) * 2.5 * 2^-24 = 1.3 * 2^-24.  A narrow one has 5e-7
    of the line's peak, and its offset, below 128 channels, 2^-18 channels.  The split
    form adds 2^-16 of the value."""
    import torch
    from scipy.special import erf, erfc

    rng = np.random.default_rng(shape[2])
    nx, ny, nc = shape
    n = nx * ny
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    order = rng.permutation(n)
    rec["ix"], rec["iy"] = order // ny, order % ny
    rec["r_kind"] = _lib.KERNEL_TABLE
    rec["h"] = np.arange(n, dtype=np.uint32).view(np.float32)
    rec["s"] = np.exp(rng.uniform(*np.log(widths), n))
    rec["fu"] = rng.uniform(0, 1, n)
    rec["k0"] = rng.integers(0, nc, n)
    half = np.ceil(5.0 / rec["s"]).astype(int) + 1
    rec["c_lo"] = np.maximum(rec["k0"] - half, 0)
    rec["c_hi"] = np.minimum(rec["k0"] + half, nc - 1)
    rec["amp"] = rng.uniform(0.5, 2.0, n)
    c = np.arange(nc)
    s, amp = rec["s"].astype(float)[:, None], rec["amp"].astype(float)[:, None]
    b = s * (rec["k0"][:, None] - c + rec["fu"].astype(float)[:, None])
    a = b - s
    across = (a < 0) & (b > 0)
    pa, pb = (np.where(across, erf(abs(x)), erfc(abs(x))) for x in (a, b))
    want = 0.5 * amp * np.where(across, pa + pb, abs(pa - pb))
    wide = 0.5 * amp * (10.0 * (pa + pb) + 2 * 1.3 + 2.0) * 2.0**-24
    narrow = 0.5642 * amp * s * (5e-7 + 0.86 * s * 2.0**-18)
    tol = np.where(s > 0.5, wide, narrow) + (2.0**-16 * want if method == "mfma" else 0.0)
    inside = (c >= rec["c_lo"][:, None]) & (c <= rec["c_hi"][:, None])
    d_w = torch.ones(n, dtype=torch.float32, device="cuda")
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_GAUSS)
    desc.weights, desc.weights_n = d_w.data_ptr(), n
    pairs = _lib.count_pairs(rec, desc)
    d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(n * nc, dtype=torch.float32, device="cuda")
    ws = torch.full((_lib.workspace_bytes(desc, n, pairs),), 255, dtype=torch.uint8, device="cuda")
    _lib.insert(d_rec, n, pairs, desc, cube, ws, method=method)
    got = cube.cpu().numpy().reshape(n, nc)[rec["ix"] * ny + rec["iy"]].astype(float)
    assert np.all(got[~inside] == 0.0)
    worst = np.max(np.where(inside, np.abs(got - want) / tol, 0.0))
    assert worst <= 1.0, worst


def test_line_centres_have_no_bias():
    """The channel that holds a line's centre, both edges within 0.85 of it: over many
    lines the mean relative error is that of the fit of erf, below 1.6e-8, and five
    standard errors of roundings of at most 2^-22 each."""
    from scipy.special import erf

    n, nc = 1 << 16, 8
    rng = np.random.default_rng(0)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["s"], rec["fu"] = rng.uniform(0.55, 0.84, n), rng.uniform(0, 1, n)
    rec["k0"], rec["c_hi"], rec["amp"] = 4, nc - 1, rng.uniform(0.5, 2.0, n)
    got = _lib.spectra(rec, _lib.make_desc(1, 1, nc, _lib.SPECTRUM_GAUSS))[:, 4].astype(float)
    s, fu, amp = (rec[k].astype(float) for k in ("s", "fu", "amp"))
    want = 0.5 * amp * (erf(s * fu) + erf(s * (1.0 - fu)))
    bias = np.mean(got / want - 1.0)
    assert abs(bias) <= 1.6e-8 + 5 * 2.0**-22 / np.sqrt(n), bias


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("shape", [(16, 16, 64), (8, 16, 128)])
@pytest.mark.parametrize("widths", [(1.0, 1.4999), (0.2, 1.4999), (0.5001, 1.4999), (1.4, 1.6)])
def test_lines_of_the_longer_series(method, shape, widths):
    """Channels of up to 3/2, where a wave whose lines are all that narrow takes a
    series, and chunks with lines on both sides of it."""
    test_lines(method, shape, widths)


def test_last_channels_of_wide_lines():
    """The last channels of lines of 1.45 to 1.5 per channel, at 1e-7 of the peak: over
    many their mean relative error is at most the first term that a series to D^16 leaves
    out and five standard errors of a rounding of the exponent (up to 21, two roundings of
    2^-24 of it, twice that in the square) and eight more."""
    import torch
    from scipy.special import erfc, eval_hermite, factorial

    shape = (64, 64, 64)
    n, nc = 4096, shape[2]
    rng = np.random.default_rng(1)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = np.arange(n) // 64, np.arange(n) % 64
    rec["r_kind"], rec["amp"], rec["h"] = _lib.KERNEL_DIRAC, 1.0, 1.0
    rec["s"], rec["fu"] = rng.uniform(1.45, 1.4999, n), rng.uniform(0, 1, n)
    rec["k0"], rec["c_lo"], rec["c_hi"] = 32, 20, 44
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_GAUSS)
    pairs = _lib.count_pairs(rec, desc)
    d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(n * nc, dtype=torch.float32, device="cuda")
    ws = torch.zeros(_lib.workspace_bytes(desc, n, pairs), dtype=torch.uint8, device="cuda")
    _lib.insert(d_rec, n, pairs, desc, cube, ws, method="plain")
    got = cube.cpu().numpy().reshape(n, nc).astype(float)
    s = rec["s"].astype(float)[:, None]
    b = s * (32 - np.arange(nc) + rec["fu"].astype(float)[:, None])
    m = np.abs(b - 0.5 * s)
    with np.errstate(over="ignore", invalid="ignore"):
        want = 0.5 * (erfc(m - 0.5 * s) - erfc(m + 0.5 * s))
    last = (m > 4.2) & (m < 4.5)
    S, M = np.broadcast_to(s, m.shape)[last], m[last]
    left_out = (S / np.sqrt(np.pi) * np.exp(-M**2) * S**18 * np.abs(eval_hermite(18, M))
                / (4.0**9 * factorial(19)))
    rel = got[last] / want[last] - 1.0
    bound = np.mean(left_out / want[last]) + 5 * (4 * 21 + 8) * 2.0**-24 / np.sqrt(rel.size)
    assert rel.size > 1000 and abs(rel.mean()) <= bound, (rel.mean(), bound)


def _one_voxel_column(w, spectra, shape, method):
    """Particles whose weight is w[k] in every pixel of one cell, in record order in
    one work item (the pair capacity of a long list makes items that long)."""
    import torch

    n, (nx, ny, nc) = w.size, shape
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["r_kind"], rec["c_hi"], rec["k0"], rec["amp"] = (40 << 8) | _lib.KERNEL_TABLE, nc - 1, np.arange(n), 1.0
    rec["h"] = (np.arange(n, dtype=np.uint32) * (nx * ny)).view(np.float32)
    weights = np.repeat(w, nx * ny)
    d_s, d_w = torch.from_numpy(spectra).cuda(), torch.from_numpy(weights).cuda()
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_TABLE, spectra=d_s, spectra_ld=nc)
    desc.weights, desc.weights_n = d_w.data_ptr(), weights.size
    cap = 6_000_000
    d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(nx * ny * nc, dtype=torch.float32, device="cuda")
    ws = torch.empty(_lib.workspace_bytes(desc, n, cap), dtype=torch.uint8, device="cuda")
    _lib.insert(d_rec, n, cap, desc, cube, ws, method=method)
    assert _lib.status(desc, n, cap, ws)[2] == 1
    got = cube.cpu().numpy().reshape(nx * ny, nc)
    assert np.array_equal(got, np.broadcast_to(got[0], got.shape))
    return got[0]


@pytest.mark.parametrize("shape", [(16, 16, 64), (8, 16, 128)])
@pytest.mark.parametrize("n", [1, 2, 5, 31, 32, 33, 64, 100, 500])
def test_fp32_sums_are_ieee_chains(shape, n):
    """The FP32 form's sum of a voxel, bit for bit: a chunk of 32 particles as a chain
    of multiply-adds from zero, the chunks' sums added in order.  (A product of two
    FP32 values is exact in FP64; the sum there is rounded once more to FP32.)"""
    rng = np.random.default_rng(n)
    w = rng.normal(size=n).astype(np.float32)
    spectra = (rng.normal(size=(n, shape[2])) * 10.0 ** rng.uniform(-2, 2, (n, 1))).astype(np.float32)
    want = np.zeros(shape[2], np.float32)
    for k in range(0, n, 32):
        chunk = np.zeros(shape[2], np.float32)
        for i in range(k, min(k + 32, n)):
            chunk = (chunk.astype(float) + w[i].astype(float) * spectra[i].astype(float)).astype(np.float32)
        want = want + chunk
    assert np.array_equal(_one_voxel_column(w, spectra, shape, "plain"), want)


@pytest.mark.parametrize("shape", [(16, 16, 64), (8, 16, 128)])
@pytest.mark.parametrize("n", [641, 1600])
def test_small_terms_are_not_lost(shape, n):
    """A bright particle and terms of 2^-26 of it, below half an ulp each: a sum of
    sums of 32 is off by at most 32 + n / 32 roundings of 2^-24."""
    w = np.full(n, 2.0**-26, np.float32)
    w[0] = 1.0
    got = _one_voxel_column(w, np.ones((n, shape[2]), np.float32), shape, "plain").astype(float)
    want = w.astype(float).sum()
    assert np.max(np.abs(got - want)) <= (32 + n / 32 + 1) * 2.0**-24 * want


def _narrow_lines(widths, n, seed):
    rng = np.random.default_rng(seed)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = np.arange(n) // 64, np.arange(n) % 64
    rec["r_kind"], rec["amp"], rec["h"] = _lib.KERNEL_DIRAC, rng.uniform(0.5, 2.0, n), 1.0
    rec["s"], rec["fu"] = rng.uniform(*widths, n), rng.uniform(0, 1, n)
    rec["k0"], rec["c_lo"], rec["c_hi"] = 64, 62, 66
    s, fu, amp = (rec[k].astype(float)[:, None] for k in ("s", "fu", "amp"))
    b = s * (64 - np.arange(62, 67) + fu)
    from scipy.special import erf

    return rec, 0.5 * amp * (erf(b) - erf(b - s))


def test_narrow_lines_have_no_bias():
    """Channels about the centre of narrow lines, one particle a pixel: their mean
    relative error is that of the constant, below 1e-8, and five standard errors of
    roundings of 2^-21 at most.  The same where lines of other widths in every chunk of
    32 send it another way.  (FP32; the split form's residuals hide it.)"""
    import torch

    n, shape = 4096, (64, 64, 128)
    rec, want = _narrow_lines((0.1, 0.3), n, 3)
    mixed = rec.copy()
    wide = np.arange(n) % 16 == 0  # two in every chunk of a tile row's 16 pixels or more
    mixed["s"][wide] = 0.9
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_GAUSS)
    bound = 1e-8 + 5 * 2.0**-21 / np.sqrt(want.size)
    for r, use in ((rec, np.ones(n, bool)), (mixed, ~wide)):
        pairs = _lib.count_pairs(r, desc)
        d_rec = torch.from_numpy(r.view(np.uint8)).cuda()
        cube = torch.zeros(n * shape[2], dtype=torch.float32, device="cuda")
        ws = torch.empty(_lib.workspace_bytes(desc, n, pairs), dtype=torch.uint8, device="cuda")
        _lib.insert(d_rec, n, pairs, desc, cube, ws, method="plain")
        got = cube.cpu().numpy().reshape(n, shape[2])[use, 62:67].astype(float)
        bias = np.mean(got / want[use] - 1.0)
        assert abs(bias) <= bound, (bias, bound)


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("widths", [(0.05, 0.5), (0.5001, 1.4999), (1.5001, 30.0)])
def test_windows_over_all_channels(method, widths):
    """Windows that take in every channel, thousands from the line: zero there, and
    1e-6 of the amplitude right elsewhere."""
    import torch
    from scipy.special import erf

    shape = (8, 8, 4096)
    n, nc = 64, shape[2]
    rng = np.random.default_rng(2)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = np.arange(n) // 8, np.arange(n) % 8
    rec["r_kind"], rec["amp"], rec["h"] = _lib.KERNEL_DIRAC, 100.0, 1.0
    rec["s"], rec["fu"] = np.exp(rng.uniform(*np.log(widths), n)), rng.uniform(0, 1, n)
    rec["k0"], rec["c_hi"] = rng.choice([0, 5, 2000, nc - 1], n), nc - 1
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_GAUSS)
    pairs = _lib.count_pairs(rec, desc)
    d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
    cube = torch.zeros(n * nc, dtype=torch.float32, device="cuda")
    ws = torch.zeros(_lib.workspace_bytes(desc, n, pairs), dtype=torch.uint8, device="cuda")
    _lib.insert(d_rec, n, pairs, desc, cube, ws, method=method)
    got = cube.cpu().numpy().reshape(n, nc).astype(float)
    b = rec["s"].astype(float)[:, None] * (rec["k0"][:, None] - np.arange(nc) + rec["fu"].astype(float)[:, None])
    a = b - rec["s"].astype(float)[:, None]
    want = 50.0 * (erf(b) - erf(a))
    assert np.all(np.isfinite(got))
    assert np.max(np.abs(got - want)) <= 100.0 * (1e-6 if method == "plain" else 2.0**-16)
    assert np.all(got[(a > 20.0) | (b < -20.0)] == 0.0)


@pytest.mark.parametrize("method", ["plain", "mfma"])
@pytest.mark.parametrize("shape", [(16, 16, 64), (8, 16, 128)])
@pytest.mark.parametrize("widths", [(0.2, 0.5), (0.5001, 1.0), (1.4, 1.4999), (2.0, 8.0)])
def test_bright_lines(method, shape, widths):
    """Lines of the largest amplitudes, a particle a pixel: 2^k times the cube of
    amplitudes near 1, bit for bit where that is far from FP32's smallest numbers (a power
    of two changes no rounding there; a split value's second part is 2^-17 of it)."""
    import torch

    nx, ny, nc = shape
    n = nx * ny
    rng = np.random.default_rng(nc)
    rec = np.zeros(n, _lib.PARTICLE_DTYPE)
    rec["ix"], rec["iy"] = np.arange(n) // ny, np.arange(n) % ny
    rec["r_kind"], rec["h"] = _lib.KERNEL_DIRAC, 1.0
    rec["s"], rec["fu"], rec["k0"] = rng.uniform(*widths, n), rng.uniform(0, 1, n), rng.integers(0, nc, n)
    half = np.ceil(4.0 / rec["s"]).astype(int) + 1
    rec["c_lo"], rec["c_hi"] = np.maximum(rec["k0"] - half, 0), np.minimum(rec["k0"] + half, nc - 1)
    amp = rng.uniform(0.5, 1.0, n).astype(np.float32)
    desc = _lib.make_desc(*shape, _lib.SPECTRUM_GAUSS)
    pairs = _lib.count_pairs(rec, desc)
    cubes = []
    for k in (0, 127):
        rec["amp"] = amp * np.float32(2.0**k)
        d_rec = torch.from_numpy(rec.view(np.uint8)).cuda()
        cube = torch.zeros(n * nc, dtype=torch.float32, device="cuda")
        ws = torch.empty(_lib.workspace_bytes(desc, n, pairs), dtype=torch.uint8, device="cuda")
        _lib.insert(d_rec, n, pairs, desc, cube, ws, method=method)
        cubes.append(cube.cpu().numpy().astype(float))
    assert np.all(np.isfinite(cubes[1])) and np.max(cubes[0]) > 0.1
    normal = cubes[0] > 2.0**-100
    assert np.array_equal(cubes[1][normal], cubes[0][normal] * 2.0**127)
    assert np.all(cubes[1][~normal] <= 2.0**27)
