"""The native packing (mi_pack_records) gives the bytes of the NumPy evaluation."""

from types import SimpleNamespace as NS

import numpy as np
import pytest

from martini_amd import DataCube, _lib, _pack
from martini_amd.spectral_models import DiracDeltaSpectrum, GaussianSpectrum
from martini_amd.sph_kernels import (CubicSplineKernel, DiracDeltaKernel, GaussianKernel,
                                     WendlandC2Kernel, _QuarticSplineKernel)

N = 4000


def _inputs(kernel, spectrum, seed, freq):
    rng = np.random.default_rng(seed)
    dc = DataCube(n_px_x=40, n_px_y=33, n_channels=21, px_size=10.0, channel_width=5.0,
                  spectral_centre=300.0)
    e = np.asarray(dc.velocity_channel_edges, float)
    if freq:  # edges falling instead of rising
        e = e[::-1].copy()
    shape = (40, 33, 21)
    x, y = rng.uniform(-12, 55, N), rng.uniform(-12, 55, N)
    x[::7], y[::11] = np.floor(x[::7]), np.floor(y[::11]) + 0.5  # on pixel centres and edges
    r = np.ceil(rng.exponential(3.0, N))
    v = rng.uniform(e.min() - 3e4, e.max() + 3e4, N) / 1e3
    v[::5] = rng.choice(e, v[::5].size) / 1e3  # on channel edges
    for k, bad in enumerate((np.nan, np.inf, -np.inf, -0.0, 1e300, -1e300, 3e6, -3e6)):
        x[20 + k], y[40 + k], v[60 + k], r[80 + k % 4] = bad, bad, bad, (np.nan, -1.0, 0.0, 1e9)[k % 4]
    x[26] = y[46] = 5.0  # 3e6 with a footprint in the cube is refused: another test
    x[100:108], r[100:108] = -5.0, 5.0  # on the cube's border
    sigma = rng.uniform(0.5, 20.0, N)
    sigma[:6] = 0.0, np.inf, np.nan, 1e-300, 1e300, 7.0
    n_k = len(kernel.kernels) if hasattr(kernel, "kernels") else 1
    which = rng.integers(0, n_k, N)
    ker = NS(_device_kernels=lambda: (kernel.kernels if n_k > 1 else (kernel,), which),
             sm_lengths=rng.exponential(3.0, N), sm_ranges=r, _rescale=rng.uniform(0.5, 2.0, N))
    src = NS(pixcoords=np.vstack((x, y, np.zeros(N))), npart=N, mHI_g=rng.uniform(0, 1e5, N),
             skycoords=NS(radial_velocity=v, distance=rng.uniform(1, 9, N)))
    cube = NS(velocity_channel_edges=e, n_channels=21, _array=np.zeros(shape))
    model = NS(_mi_kind=spectrum._mi_kind, _sigma_kms=lambda s: sigma)
    return src, ker, model, cube


def _numpy(src, ker, model, cube, out_scale):
    ix, iy, fx, fy, h, r_kind, gauss, _ = _pack.kernel_fields(ker, src.pixcoords, 40, 33)
    f = _pack.spectral_fields(src.skycoords.radial_velocity, model._sigma_kms(src), src.mHI_g,
                              src.skycoords.distance, cube, model._mi_kind, out_scale)
    k0, fu, s, amp, c_lo, c_hi = f
    return _pack.make_records(N, ix, iy, fx, fy, h, r_kind, k0, fu, s, amp, c_lo, c_hi), gauss


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
@pytest.mark.parametrize("freq", [False, True])
@pytest.mark.parametrize("spectrum", [GaussianSpectrum(), DiracDeltaSpectrum()])
@pytest.mark.parametrize("kernel", [CubicSplineKernel(), WendlandC2Kernel(), DiracDeltaKernel(),
                                    GaussianKernel(truncate=3.0), _QuarticSplineKernel()])
def test_same_bytes(kernel, spectrum, freq):
    src, ker, model, cube = _inputs(kernel, spectrum, 5, freq)
    want, gauss = _numpy(src, ker, model, cube, 0.01)
    got, gauss2 = _pack._native_records(src, ker, model, cube, 0.01)
    assert gauss == gauss2
    for f in want.dtype.names:
        a, b = (np.ascontiguousarray(w[f]).view(np.uint32) for w in (want, got))
        nan = np.isnan(want[f]) & np.isnan(got[f]) if want[f].dtype.kind == "f" else False
        assert np.all((a == b) | nan), f
    # one width for all particles
    model._sigma_kms = lambda s: 7.0
    assert np.array_equal(_numpy(src, ker, model, cube, 1.0)[0]["s"],
                          _pack._native_records(src, ker, model, cube, 1.0)[0]["s"])


@pytest.mark.filterwarnings("ignore::RuntimeWarning")
def test_far_coordinates_are_refused():
    src, ker, model, cube = _inputs(CubicSplineKernel(), GaussianSpectrum(), 6, False)
    src.pixcoords[0, 26], ker.sm_ranges[26] = 3e6, 4e6
    for f in (lambda: _numpy(src, ker, model, cube, 1.0),
              lambda: _pack._native_records(src, ker, model, cube, 1.0)):
        with pytest.raises(ValueError, match="beyond 2\\^21"):
            f()


def test_lengths_are_checked():
    one, two = np.ones(1), np.ones(2)
    with pytest.raises(ValueError, match="different lengths"):
        _lib.pack_records(two, two, two, two, np.zeros(2), one, 1.0, two, np.arange(4.0), 1.0,
                          (4, 4, 3), _lib.SPECTRUM_GAUSS)
