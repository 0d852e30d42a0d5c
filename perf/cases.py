"""Performance cases of the insertion framework.

Each case is one call (or one short sequence of calls) that a program using
martini_amd makes, on inputs with the distributions it meets in earnest:

* ``insert``: one insertion of records that are already in HBM into a zeroed
  cube (``Inserter.insert_device``), both gather forms, from the smallest mock
  to the 1e7-particle one, square and ragged cubes;
* ``prepare``: the FP64 setup of raw particle arrays on the device
  (``device_setup.prepare``) and the read of its counters;
* ``beam``: the beam convolution of a padded cube, as two one-dimensional
  passes (circular beam) or with the whole image (rotated elliptical beam);
* ``fits``: the FITS data unit of a cube;
* ``serve``: a burst of small requests through the serving loop;
* ``martini``: ``Martini.insert_source_in_cube`` on a host source.

The discs follow the recipe of ``martini_amd.synthetic`` (exponential disc,
tanh rotation curve, lognormal smoothing lengths), drawn on the GPU from the
seed.  ``exact`` restates the whole chain in FP64 with plain torch.
"""

import math

import numpy as np
import torch

ASEC = 180.0 / math.pi * 3600.0
SIG = 1.0 / (2.0 * math.sqrt(2.0 * math.log(2.0)))  # Gaussian kernel sigma for FWHM 1
BAND_KMS = 600.0


def _fit_arcsec(mpc, npx):
    """Pixel size at which npx pixels span 1.1 times a 15 kpc disc."""
    return 2.2 * math.atan(15.0 / (mpc * 1000.0)) * ASEC / npx


def _scene(n, nx, ny, nc, kms, arcsec, mpc, incl, kernel, hkpc, hetero=False, sigma=0.0):
    """One observation; sigma = 0 is the thermal line width.  hetero: smoothing
    lengths lognormal about 1 px (sigma_ln 1.5, 0.05 to 50 px) and half the
    particles at T = 1e2 K."""
    return dict(n=n, nx=nx, ny=ny, nc=nc, kms=kms, arcsec=arcsec, mpc=mpc, incl=incl,
                kernel=kernel, hkpc=hkpc, hetero=hetero, sigma=sigma)


def listed():
    c2 = _scene(1_000_000, 256, 256, 128, 4.0, 6.0, 10.0, 60.0, "wc2", 0.3)
    return [
        # the smallest mock: a dwarf sampled by 1e4 particles; launches and latency
        dict(name="insert_1e4_64px_plain", kind="insert", method="plain",
             **_scene(10_000, 64, 64, 32, 4.0, 16.0, 3.0, 60.0, "cubic", 0.8)),
        # the ordinary mock, WendlandC2 with its Gaussian fallback, both forms
        dict(name="insert_1e6_256px_plain", kind="insert", method="plain", **c2),
        dict(name="insert_1e6_256px_mfma", kind="insert", method="mfma", **c2),
        # the largest: a zoom simulation's 1e7 particles, the headline workload
        dict(name="insert_1e7_512px_mfma", kind="insert", method="mfma",
             **_scene(10_000_000, 512, 512, 256, 2.0, 1.5, 10.0, 60.0, "cubic", 0.15)),
        # tiny and huge kernels together, cold and warm gas, many pixels
        dict(name="insert_hetero_1024px_plain", kind="insert", method="plain",
             **_scene(3_000_000, 1024, 1024, 64, 8.0, 0.7, 10.0, 60.0, "cubic", 0.0, hetero=True)),
        # odd sizes: no side a multiple of a tile; fixed line width, quartic kernel
        dict(name="insert_3e5_ragged_mfma", kind="insert", method="mfma",
             **_scene(300_001, 211, 173, 75, 8.0, 3.3, 10.0, 35.0, "quartic", 0.35, sigma=7.0)),
        # device setup of an ordinary source
        dict(name="prepare_1e6", kind="prepare", **c2),
        # a circular beam on the largest cube (padded by half the beam image)
        dict(name="beam_circular_538px", kind="beam", nx=538, ny=538, nc=256, fwhm=3.0, ratio=1.0),
        # a rotated elliptical beam on the ordinary cube
        dict(name="beam_elliptical_282px", kind="beam", nx=282, ny=282, nc=128, fwhm=3.0, ratio=0.7),
        # writing the largest cube, FP64 as the host holds it and write_fits writes it
        dict(name="fits_512px_f64", kind="fits", nx=512, ny=512, nc=256, bits=64, bitpix=-64),
        # a burst of 24 small requests, served with fusion
        dict(name="serve_24_small", kind="serve", requests=24, n_lo=10_000, n_hi=300_000),
        # the reference's own call on a host source
        dict(name="martini_1e5_128px", kind="martini", method="plain",
             **_scene(100_000, 128, 128, 64, 8.0, 6.0, 10.0, 60.0, "cubic", 0.5)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_scene(rng, n_hi, npx_hi=512, nc_hi=256):
    n = _log_int(rng, 1e4, n_hi)
    mpc = rng.uniform(3.0, 30.0)
    if rng.random() < 0.4:
        nx, nc = rng.choice([s for s in ((64, 32), (128, 64), (256, 128), (512, 256))
                             if s[0] <= npx_hi and s[1] <= nc_hi])
        ny = nx
    else:
        nx, ny, nc = _log_int(rng, 48, npx_hi), _log_int(rng, 48, npx_hi), _log_int(rng, 24, nc_hi)
    return _scene(n, nx, ny, nc, BAND_KMS / nc, _fit_arcsec(mpc, min(nx, ny)), mpc,
                  rng.uniform(0.0, 90.0), rng.choice(["cubic", "wc2", "quartic"]),
                  0.8 * (n / 1e4) ** -0.24, hetero=rng.random() < 0.15,
                  sigma=rng.choice([0.0, 0.0, 7.0]))


def draw(rng):
    kind = rng.choice(["insert"] * 9 + ["prepare"] * 2 + ["beam"] * 3 + ["fits"] * 2
                      + ["serve", "martini"])
    if kind == "insert":
        return dict(kind=kind, method=rng.choice(["plain", "mfma"]), **_draw_scene(rng, 3e6))
    if kind == "prepare":
        return dict(kind=kind, **_draw_scene(rng, 5e6))
    if kind == "martini":
        return dict(kind=kind, method=rng.choice(["plain", "mfma"]),
                    **_draw_scene(rng, 1e5, npx_hi=128, nc_hi=64))
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(4, 24), n_lo=10_000,
                    n_hi=_log_int(rng, 5e4, 3e5))
    nx, ny, nc = _log_int(rng, 64, 512), _log_int(rng, 64, 512), _log_int(rng, 24, 256)
    if kind == "fits":
        return dict(kind=kind, nx=nx, ny=ny, nc=nc, bits=rng.choice([32, 64]),
                    bitpix=rng.choice([-32, -64]))
    round_beam = rng.random() < 0.5
    if not round_beam:
        nx, ny, nc = min(nx, 256), min(ny, 256), min(nc, 128)
    return dict(kind=kind, nx=nx, ny=ny, nc=nc, fwhm=rng.uniform(2.0, 3.0 if not round_beam else 5.0),
                ratio=1.0 if round_beam else rng.uniform(0.5, 0.9))


# ------------------------------------------------------------------ inputs
def _disc(s, seed):
    """xyz (kpc, face-on), vxyz (km/s), mHI (Msun), hsm (kpc), T (K) on the GPU, FP64."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    n, f = s["n"], dict(dtype=torch.float64, device="cuda")
    R = torch.empty(0, **f)
    while R.numel() < n:
        m = int((n - R.numel()) * 1.05) + 64
        u = torch.rand((2, m), generator=g, **f).clamp_min_(1e-300)
        t = -3.0 * torch.log(u[0] * u[1])
        R = torch.cat((R, t[t <= 15.0]))
    R = R[:n]
    phi = torch.rand(n, generator=g, **f) * (2.0 * math.pi)
    z = torch.randn(n, generator=g, **f) * 0.3
    noise = torch.randn((n, 3), generator=g, **f) * 10.0
    vc = 200.0 * torch.tanh(R / 2.0)
    xyz = torch.stack((z, R * torch.cos(phi), R * torch.sin(phi)), dim=1)
    vxyz = torch.stack((noise[:, 0], -vc * torch.sin(phi) + noise[:, 1],
                        vc * torch.cos(phi) + noise[:, 2]), dim=1)
    mHI = (0.5 + torch.rand(n, generator=g, **f)) * (1e9 / n)
    e = torch.randn(n, generator=g, **f)
    T = torch.full((n,), 1e4, **f)
    if s["hetero"]:
        hpx = torch.exp(1.5 * e).clamp(0.05, 50.0)
        hsm = torch.tan(hpx * s["arcsec"] / ASEC) * s["mpc"] * 1000.0
        T[::2] = 1e2
    else:
        hsm = s["hkpc"] * torch.exp(0.5 * e)
    return xyz, vxyz, mHI, hsm, T


def _objects(s):
    """DataCube, kernel, spectral model and rotation of a scene."""
    from scipy.spatial.transform import Rotation

    from martini_amd import DataCube, spectral_models, sph_kernels

    dc = DataCube(n_px_x=s["nx"], n_px_y=s["ny"], n_channels=s["nc"], px_size=s["arcsec"],
                     channel_width=s["kms"], spectral_centre=70.0 * s["mpc"])
    k = {"cubic": sph_kernels.CubicSplineKernel, "wc2": sph_kernels.WendlandC2Kernel,
         "quartic": sph_kernels.QuarticSplineKernel}[s["kernel"]]()
    sp = spectral_models.GaussianSpectrum(sigma=s["sigma"] or "thermal")
    return dc, k, sp, Rotation.from_euler("y", math.radians(s["incl"]))


def _device_source(s, seed):
    from martini_amd import device_setup

    dc, k, sp, rot = _objects(s)
    src = device_setup.DeviceSource(*_disc(s, seed))
    obs, desc = device_setup.observation(distance=s["mpc"], datacube=dc, sph_kernel=k,
                                         spectral_model=sp, rotation=rot)
    return src, obs, desc


def _requests(case):
    """Shapes, kernels and observing geometry of a burst of small requests (the
    case's own; the seed draws the discs)."""
    rng = np.random.default_rng(case["requests"] + case["n_hi"])
    lo, hi = math.log(case["n_lo"]), math.log(case["n_hi"])
    out = []
    for _ in range(case["requests"]):
        npx, nc = ((64, 32), (128, 64))[rng.integers(2)]
        n, mpc = int(math.exp(rng.uniform(lo, hi))), float(rng.uniform(3.0, 30.0))
        out.append(_scene(n, npx, npx, nc, BAND_KMS / nc, _fit_arcsec(mpc, npx), mpc,
                          float(rng.uniform(0.0, 90.0)), ("cubic", "wc2")[rng.integers(2)],
                          0.8 * (n / 1e4) ** -0.24))
    return out


def _beam_image(case, seed):
    """A normalised Gaussian beam image out to 4 FWHM (FP64); ratio < 1 is a
    rotated ellipse, whose image is no outer product."""
    fwhm = case["fwhm"] * (1.0 + 0.002 * (seed % 16))
    h = int(math.ceil(4.0 * case["fwhm"])) + 1
    sa = fwhm * SIG
    sb, th = sa * case["ratio"], math.radians(30.0)
    a = np.arange(-h, h + 1)
    x, y = a[:, None], a[None, :]
    u, v = x * math.cos(th) + y * math.sin(th), -x * math.sin(th) + y * math.cos(th)
    K = np.exp(-0.5 * ((u / sa) ** 2 + (v / sb) ** 2))
    line = np.exp(-0.5 * (a / sa) ** 2)
    return np.float32(K / K.sum()), np.float32(line / line.sum())


def _cube(case, seed, dtype=torch.float32):
    """A line cube as insertion leaves it: positive, a large range, empty sky around it."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    v = torch.randn((case["nx"], case["ny"], case["nc"]), generator=g, device="cuda")
    return torch.where(v > -0.5, torch.exp(2.0 * v) * 1e-6, 0.0).to(dtype)


def prepare(case, seed):
    from martini_amd import _lib, device_setup, insertion

    kind = case["kind"]
    if kind == "insert":
        src, obs, desc = _device_source(case, seed)
        rec, counts = device_setup.prepare(src, obs)
        kept, pairs = (int(v) for v in counts[:2].cpu())
        rec = insertion.layout_records(rec[:48 * kept], case["method"], desc.nc)
        cube = torch.empty(desc.nx * desc.ny * desc.nc, dtype=torch.float32, device="cuda")
        return dict(case=case, rec=rec, kept=kept, pairs=pairs, desc=desc, cube=cube,
                    inserter=insertion.Inserter())
    if kind == "prepare":
        src, obs, _ = _device_source(case, seed)
        return dict(case=case, src=src, obs=obs)
    if kind == "beam":
        K, line = _beam_image(case, seed)
        d_in = _cube(case, seed)
        taps = torch.from_numpy(line if case["ratio"] == 1.0 else K).cuda()
        return dict(case=case, d_in=d_in, tmp=torch.empty_like(d_in), out=torch.empty_like(d_in),
                    taps=taps)
    if kind == "fits":
        cube = _cube(case, seed, torch.float64 if case["bits"] == 64 else torch.float32)
        return dict(case=case, cube=cube,
                    out=torch.empty(cube.numel() * (-case["bitpix"] // 8), dtype=torch.uint8,
                                    device="cuda"),
                    rng=torch.empty(2, dtype=torch.float64, device="cuda"))
    if kind == "serve":
        from martini_amd import serving

        scenes = _requests(case)
        specs = [serving.RequestSpec(rid=i, n=s["n"], seed=i, incl=s["incl"], distance=s["mpc"],
                                     n_px=s["nx"], n_channels=s["nc"], kernel=s["kernel"])
                 for i, s in enumerate(scenes)]
        srcs = [device_setup.DeviceSource(*_disc(s, seed * 64 + i)) for i, s in enumerate(scenes)]
        svc = serving.Service(slots=4, method="mfma")
        svc.warm(((64, 32), (128, 64)))
        return dict(case=case, service=svc, specs=specs, srcs=srcs)
    from martini_amd import Martini, SPHSource

    dc, k, sp, rot = _objects(case)
    xyz, vxyz, mHI, hsm, T = (a.cpu().numpy() for a in _disc(case, seed))
    src = SPHSource(distance=case["mpc"], rotation=rot, h=0.7, T_g=T, mHI_g=mHI, xyz_g=xyz,
                    vxyz_g=vxyz, hsm_g=hsm)
    return dict(case=case, martini=Martini(source=src, datacube=dc, sph_kernel=k,
                                           spectral_model=sp, quiet=True))


# -------------------------------------------------------------------- one pass
# the 32-bit words of a record (mi_particle)
INT_FIELDS = {"ix": 0, "iy": 1, "r_kind": 5, "c_lo": 6, "c_hi": 7, "k0": 8}
FLOAT_FIELDS = {"fx": 2, "fy": 3, "h": 4, "fu": 9, "s": 10, "amp": 11}


def run(state):
    from martini_amd import _lib, device_setup

    case = state["case"]
    kind = case["kind"]
    if kind == "insert":
        state["cube"].zero_()
        state["inserter"].insert_device(state["rec"], state["kept"], state["pairs"],
                                        state["desc"], state["cube"], method=case["method"])
        return state["cube"]
    if kind == "prepare":
        rec, counts = device_setup.prepare(state["src"], state["obs"])
        counts = counts.cpu()  # a program needs the counts to size what follows
        words = rec.view(torch.int32).view(-1, 12)[: int(counts[0])]
        reals = rec.view(torch.float32).view(-1, 12)[: int(counts[0])]
        return dict(counts=counts, **{k: words[:, c] for k, c in INT_FIELDS.items()},
                    **{k: reals[:, c] for k, c in FLOAT_FIELDS.items()})
    if kind == "beam":
        nx, ny, nc = case["nx"], case["ny"], case["nc"]
        t = state["taps"]
        if case["ratio"] == 1.0:  # as Martini.convolve_beam does for a separable image
            _lib.convolve_beam(state["d_in"], state["tmp"], nx, ny, nc, t, t.numel(), 1)
            _lib.convolve_beam(state["tmp"], state["out"], nx, ny, nc, t, 1, t.numel())
        else:
            _lib.convolve_beam(state["d_in"], state["out"], nx, ny, nc, t, *t.shape)
        return state["out"]
    if kind == "fits":
        _lib.cube_to_fits(state["cube"], case["nx"], case["ny"], case["nc"], 0, 0,
                          case["bitpix"], state["out"], state["rng"])
        return dict(data=state["out"], range=state["rng"])
    if kind == "serve":
        return [r.cube for r in state["service"].run(state["specs"], state["srcs"])]
    m = state["martini"]
    m.reset()
    m.insert_source_in_cube(method=case["method"])
    return np.asarray(m.datacube._array, np.float32)  # kept in single precision, as a file would


# ------------------------------------------------------------ necessary work
_FWHM = {}


def _radial(kernel, q):
    """The 3D kernels, up to a factor."""
    if kernel == "wc2":
        return (1 - q) ** 4 * (4 * q + 1)
    if kernel == "cubic":
        return 1 - 6 * q**2 + 6 * q**3 if q < 0.5 else 2 * (1 - q) ** 3
    return ((1 - q) ** 4 - 5 * max(0.6 - q, 0.0) ** 4 + 10 * max(0.2 - q, 0.0) ** 4)


def _fwhm(kernel):
    if kernel not in _FWHM:
        lo, hi, half = 0.0, 1.0, 0.5 * _radial(kernel, 0.0)
        for _ in range(200):
            mid = 0.5 * (lo + hi)
            lo, hi = (mid, hi) if _radial(kernel, mid) > half else (lo, mid)
        _FWHM[kernel] = 2.0 * lo
    return _FWHM[kernel]


MIN_PX = {"wc2": 1.51, "cubic": 1.16, "quartic": 1.2385}


def _insert_work(s):
    """Records read once, cube written once; one multiply-add per pixel of a
    particle's support and channel of its line (8 sigma and one channel)."""
    kpc_px = s["mpc"] * 1000.0 * math.tan(s["arcsec"] / ASEC)
    h2 = math.exp(2 * 1.5**2) if s["hetero"] else (s["hkpc"] / kpc_px) ** 2 * math.exp(0.5)
    px = max(1.0, math.pi * h2 / _fwhm(s["kernel"]) ** 2)
    line = min(s["nc"], 8.0 * (s["sigma"] or 9.1) / s["kms"] + 1.0)
    return dict(bytes=48.0 * s["n"] + 4.0 * s["nx"] * s["ny"] * s["nc"], flops=2.0 * s["n"] * px * line)


def work(case):
    kind = case["kind"]
    if kind in ("insert", "martini"):
        return _insert_work(case)
    if kind == "prepare":  # ten FP64 values read, one record written
        return dict(bytes=128.0 * case["n"], flops=500.0 * case["n"])
    if kind == "serve":  # setup and insertion of each request, of the mean size
        n = (case["n_hi"] - case["n_lo"]) / math.log(case["n_hi"] / case["n_lo"]) * case["requests"]
        vox = case["requests"] * 0.5 * (64 * 64 * 32 + 128 * 128 * 64)
        return dict(bytes=176.0 * n + 8.0 * vox, flops=1e4 * n)
    vox = float(case["nx"]) * case["ny"] * case["nc"]
    if kind == "fits":
        return dict(bytes=vox * (case["bits"] - case["bitpix"]) / 8, flops=vox)
    k = 2 * (int(math.ceil(4.0 * case["fwhm"])) + 1) + 1
    if case["ratio"] == 1.0:  # two passes through the public call
        return dict(bytes=16.0 * vox, flops=4.0 * k * vox)
    return dict(bytes=8.0 * vox, flops=2.0 * k * k * vox)


# --------------------------------------------------------------- 64-bit values
def _setup64(s, seed):
    """Pixel positions, kernel tier, ranges and line parameters in FP64."""
    xyz, vxyz, m, hsm, T = _disc(s, seed)
    c, q = math.cos(math.radians(s["incl"])), math.sin(math.radians(s["incl"]))
    rot = torch.tensor([[c, 0.0, q], [0.0, 1.0, 0.0], [-q, 0.0, c]], dtype=torch.float64,
                       device="cuda")

    def turned(v):  # elementwise, so that no matrix unit rounds
        return torch.stack([(v * rot[i]).sum(1) for i in range(3)], dim=1)

    pos, vel = turned(xyz) / 1000.0, turned(vxyz)
    pos[:, 0] += s["mpc"]
    vel = vel + 70.0 * pos
    dist = pos.square().sum(1).sqrt()
    v = (pos * vel).sum(1) / dist * 1e3
    px_deg = s["arcsec"] / 3600.0
    x = s["nx"] / 2.0 - 0.5 - torch.rad2deg(pos[:, 1] / pos[:, 0]) / px_deg
    y = s["ny"] / 2.0 - 0.5 + torch.rad2deg(pos[:, 2] / pos[:, 0]) / px_deg
    hpx = torch.atan(hsm / (dist * 1000.0)) * ASEC / s["arcsec"]
    f = _fwhm(s["kernel"])
    tier = torch.where(hpx / f >= MIN_PX[s["kernel"]], 0, torch.where(hpx <= 0.5, 1, 2))
    size = torch.tensor([1.0 / f, 1.0, 6.0 * SIG], dtype=torch.float64, device="cuda")[tier]
    w = s["kms"] * 1e3
    u = (v - (70.0 * s["mpc"] * 1e3 + 0.5 * w * s["nc"])) / -w
    sig = torch.sqrt(1.380649e-23 * T / 1.67262192369e-27) if not s["sigma"] else \
        torch.full_like(T, s["sigma"] * 1e3)
    r = torch.ceil(hpx * size)
    hw = sig / w
    keep = ~((x + r < 0) | (y + r < 0) | (x - r > s["nx"]) | (y - r > s["ny"])
             | (u - 0.5 + 4 * hw < 0) | (u - 0.5 - 4 * hw > s["nc"]))
    amp = m / dist**2 / s["kms"] / 2.36e5 / s["arcsec"] ** 2
    h = torch.where(tier == 0, hpx / f, hpx)
    cols = dict(x=x, y=y, tier=tier, r=r, h=h, u=u, s=w / (math.sqrt(2.0) * sig), amp=amp)
    return {k: a[keep] for k, a in cols.items()}


def _weight64(kernel, tier, dx, dy, h):
    """The kernel's line-of-sight integral at a pixel, per unit pixel area."""
    if tier == 1:
        return ((dx.abs() < 0.5) & (dy.abs() < 0.5)).double()
    if tier == 2:
        hs, t = h * SIG, 6.0
        b = 1.0 / (hs * math.sqrt(2.0))
        ex = torch.erf((dx + 0.5) * b) - torch.erf((dx - 0.5) * b)
        ey = torch.erf((dy + 0.5) * b) - torch.erf((dy - 0.5) * b)
        d2 = dx * dx + dy * dy
        zmax = (t * t - d2 / (hs * hs)).clamp_min(0.0).sqrt()
        norm = math.erf(t / math.sqrt(2.0)) - 2 * t / math.sqrt(2 * math.pi) * math.exp(-t * t / 2)
        w = 0.25 * torch.erf(zmax / math.sqrt(2.0)) * ex * ey / norm
        return torch.where(d2 <= (t * hs + math.sqrt(0.5)) ** 2, w, 0.0)
    R2 = ((dx * dx + dy * dy) / (h * h)).clamp_min(1e-24)
    if kernel == "wc2":
        A = (1.0 - R2).clamp_min(0.0).sqrt()
        G = 5.0 * R2**2 * (0.5 * R2 + 3.0) * torch.log((1.0 + A) / R2.sqrt()) + A * (
            -13.5 * R2**2 - 14.0 / 3.0 * R2 + 2.0 / 3.0)
        return torch.where(R2 < 1.0, G, 0.0) * (21.0 / (2.0 * math.pi)) / (h * h)
    if kernel == "cubic":
        R2 = 4.0 * R2
        A, B = (1.0 - R2).clamp_min(0.0).sqrt(), (4.0 - R2).clamp_min(0.0).sqrt()
        inner = (A - 0.5 * A**3 - 1.5 * R2 * A + 3.0 / 32.0 * A * (3.0 * R2 + 2.0)
                 + 9.0 / 32.0 * R2**2 * torch.log((1.0 + A) / R2.sqrt()))
        tail = (-B * (3.0 * R2 + 56.0) / 4.0 + A * (4.0 * R2 + 50.0) / 8.0
                - 0.375 * R2 * (R2 + 16.0) * torch.log((2.0 + B) / (1.0 + A))
                + 2.0 * (3.0 * R2 + 4.0) * (B - A) + 2.0 * (B**3 - A**3))
        outer = (-B * (3.0 * R2 + 56.0) / 4.0
                 - 0.375 * R2 * (R2 + 16.0) * torch.log((2.0 + B) / R2.sqrt())
                 + 2.0 * (3.0 * R2 + 4.0) * B + 2.0 * B**3)
        F = torch.where(R2 <= 1.0, inner + 0.25 * tail, torch.where(R2 <= 4.0, 0.25 * outer, 0.0))
        return F * (4.0 / 1.59689476201133) / (h * h)
    R = R2.sqrt()

    def part(a):  # integral over z of (a - sqrt(R^2 + z^2))^4 up to the shell q = a
        z = (a * a - R2).clamp_min(0.0).sqrt()
        g = (z * z + R2).sqrt()
        v = (a**4 * z - 2 * a**3 * z * g + 2 * a * a * z * (3 * R2 + z * z)
             - 0.5 * a * R2 * (4 * a * a + 3 * R2) * torch.asinh(z / R)
             - 0.5 * a * z * g * (5 * R2 + 2 * z * z) + R2 * R2 * z + 2.0 / 3.0 * R2 * z**3
             + 0.2 * z**5)
        return torch.where(R < a, v, 0.0)

    return (part(1.0) - 5.0 * part(0.6) + 10.0 * part(0.2)) * (15625.0 / (256.0 * math.pi)) / (h * h)


def _cube64(s, seed):
    """The inserted cube in Jy/arcsec^2: every particle's line times its pixel weights."""
    P = _setup64(s, seed)
    nx, ny, nc = s["nx"], s["ny"], s["nc"]
    cube = torch.zeros((nx * ny, nc), dtype=torch.float64, device="cuda")
    chan = torch.arange(nc, dtype=torch.float64, device="cuda")
    group = P["tier"] * 4096 + P["r"].long()
    order = torch.argsort(group)
    values, lengths = torch.unique_consecutive(group[order], return_counts=True)
    at = 0
    for value, length in zip(values.tolist(), lengths.tolist()):
        tier, r = value // 4096, value % 4096
        off = torch.arange(-r, r + 1, device="cuda")
        if tier == 1:
            off = torch.arange(0, 1, device="cuda")  # the nearest pixel alone
        oi, oj = off.repeat_interleave(off.numel()), off.repeat(off.numel())
        step = max(1, int(4e8 // (nc * oi.numel())))
        for a in range(at, at + length, step):
            p = {k: v[order[a:min(a + step, at + length)]] for k, v in P.items()}
            x, y = p["x"], p["y"]
            if tier == 1:
                i0, j0 = torch.floor(x + 0.5).long(), torch.floor(y + 0.5).long()
            else:  # |i - x| <= r is i = ceil(x - r) .. floor(x + r)
                i0, j0 = torch.floor(x).long(), torch.floor(y).long()
            i, j = i0[:, None] + oi, j0[:, None] + oj
            dx, dy = x[:, None] - i, y[:, None] - j
            w = _weight64(s["kernel"], tier, dx, dy, p["h"][:, None])
            ok = (i >= 0) & (i < nx) & (j >= 0) & (j < ny) & (w != 0.0)
            ok &= (dx.abs() <= r) & (dy.abs() <= r)
            d = p["u"][:, None] - chan
            b = p["s"][:, None]
            hi, lo = b * d, b * (d - 1.0)  # erf(hi) - erf(lo) on the side where neither cancels
            neg = hi + lo < 0.0
            hi, lo = torch.where(neg, -lo, hi), torch.where(neg, -hi, lo)
            line = 0.5 * p["amp"][:, None] * (torch.erfc(lo) - torch.erfc(hi))
            k, e = ok.nonzero(as_tuple=True)
            cube.index_add_(0, i[k, e] * ny + j[k, e], w[k, e][:, None] * line[k])
        at += length
    return cube


def exact(case, seed):
    kind = case["kind"]
    if kind in ("insert", "martini"):
        cube = _cube64(case, seed)
        return cube.view(-1) if kind == "insert" else cube.view(case["nx"], case["ny"], case["nc"])
    if kind == "serve":
        return [_cube64(s, seed * 64 + i).view(s["nx"], s["ny"], s["nc"]).cpu()
                for i, s in enumerate(_requests(case))]
    if kind == "prepare":
        P = _setup64(case, seed)
        real = {k: P[k] for k in ("h", "s", "amp")}
        real["fu"] = P["u"] - P["u"].floor()
        for k in ("x", "y"):  # a point-like particle's record holds its pixel's centre
            real["f" + k] = torch.where(P["tier"] == 1, 0.0, P[k] - P[k].floor())
        return dict(counts=None, **{k: None for k in INT_FIELDS}, **real)
    if kind == "fits":
        c = _cube(case, seed, torch.float64 if case["bits"] == 64 else torch.float32).double()
        return dict(data=None, range=torch.stack((c.min(), c.max())))
    K, line = _beam_image(case, seed)
    out = _cube(case, seed).double()
    images = [K] if case["ratio"] != 1.0 else [line[:, None], line[None, :]]
    for image in images:
        kx, ky = image.shape
        pad = torch.zeros((case["nx"] + kx - 1, case["ny"] + ky - 1, case["nc"]),
                          dtype=torch.float64, device="cuda")
        pad[kx // 2:kx // 2 + case["nx"], ky // 2:ky // 2 + case["ny"]] = out
        out = torch.zeros_like(out)
        for a in range(kx):
            for b in range(ky):
                out.add_(pad[kx - 1 - a:kx - 1 - a + case["nx"], ky - 1 - b:ky - 1 - b + case["ny"]],
                         alpha=float(image[a, b]))
    return out
