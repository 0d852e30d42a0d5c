"""Device FP64 setup (mi_prepare) against the host setup and packer.

The same raw particle arrays go through Martini's host setup
(SPHSource -> Martini.__init__ -> _pack.pack_particles) and through
mi_prepare on the GPU; the records must agree field by field (integers
exactly, FP32 fields to rounding), and the cubes inserted from them must
agree to 1e-6 of the peak.
"""

import dataclasses

import numpy as np
import pytest

from martini_amd import Martini, _lib, synthetic
from martini_amd.device_setup import DeviceSource, observation, prepare
from martini_amd.sph_kernels import CubicSplineKernel, WendlandC2Kernel, _CubicSplineKernel
from martini_amd.spectral_models import DiracDeltaSpectrum, GaussianSpectrum

pytestmark = pytest.mark.gpu

INT_FIELDS = ("ix", "iy", "r_kind", "c_lo", "c_hi", "k0")
FLOAT_FIELDS = ("fx", "fy", "h", "fu", "s", "amp")


def _case(name):
    w1 = synthetic.WORKLOADS["disc1e4_64px"]
    w2 = synthetic.WORKLOADS["disc1e6_256px"]
    if name == "cubic":
        return w1, None, CubicSplineKernel, lambda: GaussianSpectrum(sigma="thermal")
    if name == "wc2_2e5":
        return w2, 200_000, WendlandC2Kernel, lambda: GaussianSpectrum(sigma="thermal")
    if name == "pruned_cube":  # a cube smaller than the disc: spatial pruning and edge clipping
        return (dataclasses.replace(w1, n_px=24, n_channels=12), None, CubicSplineKernel,
                lambda: GaussianSpectrum(sigma="thermal"))
    if name == "fixed_sigma":
        return w1, None, CubicSplineKernel, lambda: GaussianSpectrum(sigma=7.0)
    if name == "dirac_spectrum":
        return w1, None, CubicSplineKernel, DiracDeltaSpectrum
    if name == "fixed_kernel":
        return w1, None, _CubicSplineKernel, lambda: GaussianSpectrum(sigma="thermal")
    raise KeyError(name)


def _host(w, n, make_k, make_s):
    src, dc, k, s = synthetic.build(w, n, kernel=make_k(), spectrum=make_s())
    m = Martini(source=src, datacube=dc, sph_kernel=k, spectral_model=s, quiet=True)
    from martini_amd import _pack

    rec, desc = _pack.pack_particles(m.source, m.sph_kernel, m.spectral_model, dc,
                                     out_scale=1.0 / dc.px_size**2)
    return rec, desc, dc, m


def _mask_pixels(m):
    """Pixels of the reference's square masks inside the padded cube."""
    nx, ny = m.datacube._array.shape[:2]
    x, y = m.source.pixcoords[0], m.source.pixcoords[1]
    r = np.asarray(m.sph_kernel.sm_ranges, float)
    nxp = np.clip(np.minimum(nx - 1, np.floor(x + r)) - np.maximum(0, np.ceil(x - r)) + 1, 0, None)
    nyp = np.clip(np.minimum(ny - 1, np.floor(y + r)) - np.maximum(0, np.ceil(y - r)) + 1, 0, None)
    return int(np.sum(nxp * nyp))


def _device(w, n, make_k, make_s, dc):
    import torch

    a = w.arrays(n)
    src = DeviceSource(a.xyz, a.vxyz, a.mHI, a.hsm, a.T)
    obs, desc = observation(distance=w.distance, datacube=dc, sph_kernel=make_k(),
                            spectral_model=make_s(), rotation=w.rotation, h=0.7)
    out, counts = prepare(src, obs, datacube=dc)
    torch.cuda.synchronize()
    kept, pairs, flags, mask_px = (int(v) for v in counts.cpu())
    rec = out[: kept * 48].cpu().numpy().view(_lib.PARTICLE_DTYPE)
    return rec, desc, pairs, flags, out, mask_px


@pytest.mark.parametrize("name", ["cubic", "wc2_2e5", "pruned_cube", "fixed_sigma",
                                  "dirac_spectrum", "fixed_kernel"])
def test_prepare_matches_host(name):
    w, n, make_k, make_s = _case(name)
    hrec, hdesc, dc, m = _host(w, n, make_k, make_s)
    drec, ddesc, pairs, flags, _, mask_px = _device(w, n, make_k, make_s, dc)
    print(f"{name}: host {hrec.size} device {drec.size} pairs {pairs} flags {flags}")
    assert drec.size == hrec.size
    assert pairs == _lib.count_pairs(hrec, hdesc)
    assert mask_px == _mask_pixels(m)
    for f in INT_FIELDS:
        bad = np.count_nonzero(drec[f] != hrec[f])
        assert bad == 0, (f, bad)
    for f in FLOAT_FIELDS:
        a, b = drec[f].astype(float), hrec[f].astype(float)
        tol = 2.0**-21 * np.maximum(np.abs(b), 1.0 if f in ("fx", "fy", "fu") else 0.0)
        worst = np.max(np.abs(a - b) - tol)
        assert worst <= 0.0, (f, float(np.max(np.abs(a - b))))
    assert tuple(ddesc.gauss_t) == tuple(hdesc.gauss_t)
    assert (ddesc.nx, ddesc.ny, ddesc.nc, ddesc.spectrum) == (hdesc.nx, hdesc.ny, hdesc.nc,
                                                              hdesc.spectrum)


def test_prepared_records_insert_like_host_records():
    import torch

    from martini_amd.insertion import Inserter

    w, n, make_k, make_s = _case("wc2_2e5")
    hrec, hdesc, dc, _ = _host(w, n, make_k, make_s)
    drec, ddesc, pairs, flags, d_out, _ = _device(w, n, make_k, make_s, dc)
    ins = Inserter()
    host_cube = ins.insert(hrec, hdesc, method="plain").cpu().numpy()
    cube = torch.zeros(ddesc.nx * ddesc.ny * ddesc.nc, dtype=torch.float32, device=d_out.device)
    ins.insert_device(d_out, drec.size, pairs, ddesc, cube, method="plain")
    dev_cube = cube.cpu().numpy()
    diff = np.abs(dev_cube - host_cube).max() / np.abs(host_cube).max()
    print(f"device-setup cube vs host-setup cube: {diff:.3e}")
    assert diff <= 1e-6


@pytest.mark.parametrize("n", [1, 255, 256, 511, 512, 513, 65 * 512 + 3])
@pytest.mark.parametrize("massless", ["none", "some", "all"])
def test_prepare_is_the_sum_of_its_parts(n, massless):
    """The look-back over work groups of 512 particles: one call gives the
    records and counts of separate calls on slices of at most 512 (one group
    each), back to back, byte for byte, for groups that keep all, some (in
    whole groups too) or none of their particles."""
    import torch

    w, _, make_k, make_s = _case("pruned_cube")
    _, dc, k, s = synthetic.build(w, 16, kernel=make_k(), spectrum=make_s())
    obs, _ = observation(distance=w.distance, datacube=dc, sph_kernel=k, spectral_model=s,
                         rotation=w.rotation, h=0.7)
    a = w.arrays(n)
    m = a.mHI.copy()
    if massless == "all":
        m[:] = 0.0
    elif massless == "some":
        m[np.arange(n) % 7 < 3] = 0.0
        m[(np.arange(n) // 512) % 3 == 1] = 0.0

    def run(sl):
        src = DeviceSource(a.xyz[sl], a.vxyz[sl], m[sl], a.hsm[sl], a.T[sl])
        out, counts = prepare(src, obs)
        counts = counts.cpu()
        return out[: int(counts[0]) * 48].cpu(), counts

    rec, counts = run(slice(0, n))
    parts = [run(slice(b, min(b + 512, n))) for b in range(0, n, 512)]
    assert torch.equal(rec, torch.cat([p[0] for p in parts]))
    total = torch.stack([p[1] for p in parts]).sum(0)
    assert torch.equal(counts[[0, 1, 3]], total[[0, 1, 3]])
    if massless == "all":
        assert counts.tolist() == [0, 0, 0, 0]


def test_prepare_directions_match_host():
    """Keep flags and sky pixels where the direction is degenerate: the
    observer itself, the far hemisphere, infinite and NaN positions."""
    inf, nan, D = np.inf, np.nan, 3000.0  # kpc
    xyz = np.array([[0, 0, 0], [-D, 0, 0], [-2 * D, 1, 1], [inf, 0, 0], [0, inf, 0], [0, 0, -inf],
                    [inf, 1, inf], [-inf, 2, 0], [nan, 0, 0], [0, 0, nan], [1, 2, 3]], float)
    w = dataclasses.replace(synthetic.WORKLOADS["disc1e4_64px"], n=len(xyz))
    n = len(xyz)
    from martini_amd import DataCube, SPHSource

    for ra, dec in ((0.0, 0.0), (30.0, -20.0)):
        kw = dict(n_px_x=33, n_px_y=20, n_channels=16, px_size=16.0, channel_width=8.0,
                  spectral_centre=w.vsys, ra=ra, dec=dec)
        src = SPHSource(distance=w.distance, h=0.7, T_g=np.full(n, 1e4), mHI_g=np.full(n, 1e4),
                        xyz_g=xyz, vxyz_g=np.zeros((n, 3)), hsm_g=np.full(n, 0.5))
        with np.errstate(all="ignore"):
            m = Martini(source=src, datacube=DataCube(**kw), sph_kernel=CubicSplineKernel(),
                        spectral_model=GaussianSpectrum(sigma="thermal"), quiet=True)
            from martini_amd import _pack

            hrec, _ = _pack.pack_particles(m.source, m.sph_kernel, m.spectral_model, m.datacube)
        obs, _ = observation(distance=w.distance, datacube=DataCube(**kw),
                             sph_kernel=CubicSplineKernel(),
                             spectral_model=GaussianSpectrum(sigma="thermal"))
        out, counts = prepare(DeviceSource(xyz, np.zeros((n, 3)), np.full(n, 1e4), np.full(n, 0.5),
                                           np.full(n, 1e4)), obs)
        drec = out[: int(counts.cpu()[0]) * 48].cpu().numpy().view(_lib.PARTICLE_DTYPE)
        assert drec.size == hrec.size
        for f in ("ix", "iy", "c_lo", "c_hi"):
            assert np.array_equal(drec[f], hrec[f]), (f, drec[f], hrec[f])


def test_prepare_directions_out_of_range_match_host():
    """The same for positions whose squares overflow or underflow, and with
    several infinite components."""
    inf, D, c = np.inf, 3000.0, np.sqrt(0.5)  # kpc
    xyz = np.array([[1e200, 1e197, 0], [1e160, -1e157, 2e157], [-1e200, 1, 1], [1e200, 1e200, 0],
                    [-D, 1e-190, 0], [-D, 0, -1e-200], [inf, 1, inf], [inf, inf, inf],
                    [inf, 1, 1e200], [1, inf, -inf], [1, 2, 3],
                    # and one in the middle of each map below
                    [0.5 * D - D, 0.5 * D, c * D], [c * D - D, 0, c * D]], float)
    w = dataclasses.replace(synthetic.WORKLOADS["disc1e4_64px"], n=len(xyz))
    n = len(xyz)
    from martini_amd import DataCube, SPHSource, _pack

    for ra, dec in ((0.0, 0.0), (45.0, 45.0), (0.0, 45.0)):
        kw = dict(n_px_x=65, n_px_y=64, n_channels=16, px_size=16.0, channel_width=8.0,
                  spectral_centre=w.vsys, ra=ra, dec=dec)
        src = SPHSource(distance=w.distance, h=0.7, T_g=np.full(n, 1e4), mHI_g=np.full(n, 1e4),
                        xyz_g=xyz, vxyz_g=np.zeros((n, 3)), hsm_g=np.full(n, 0.5))
        with np.errstate(all="ignore"):
            m = Martini(source=src, datacube=DataCube(**kw), sph_kernel=CubicSplineKernel(),
                        spectral_model=GaussianSpectrum(sigma="thermal"), quiet=True)
            hrec, _ = _pack.pack_particles(m.source, m.sph_kernel, m.spectral_model, m.datacube)
        obs, _ = observation(distance=w.distance, datacube=DataCube(**kw),
                             sph_kernel=CubicSplineKernel(),
                             spectral_model=GaussianSpectrum(sigma="thermal"))
        out, counts = prepare(DeviceSource(xyz, np.zeros((n, 3)), np.full(n, 1e4), np.full(n, 0.5),
                                           np.full(n, 1e4)), obs)
        drec = out[: int(counts.cpu()[0]) * 48].cpu().numpy().view(_lib.PARTICLE_DTYPE)
        assert drec.size == hrec.size > 0
        for i, f in (("ix", "fx"), ("iy", "fy")):  # a position may lie on a pixel's edge
            at = [r[i] + r[f].astype(float) for r in (drec, hrec)]
            assert np.allclose(*at, rtol=1e-9, atol=1e-6), (i, at)
        for f in ("c_lo", "c_hi"):
            assert np.array_equal(drec[f], hrec[f]), (f, drec[f], hrec[f])
