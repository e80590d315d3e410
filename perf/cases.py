"""The work a program built on pdspy_amd has the GPU do, as plain cases.

A fit or a forward model runs, per parameter set: the thermal Monte Carlo
(``DeviceModel.thermal`` + ``temperature``), an image at one wavelength -- with
RADMC-3D's recursive sub-pixeling and the scattering source, as ``run_image``
calls it, or plain with its adjoint in gradient-based fits --, the visibilities
at the data's (u, v) points, exact or by galario's gridded method, and their
transpose; a sampler does all of it for a batch of walkers in one step.  The
sizes are those of ``pdspy_amd.configs``, of the tests and of the benchmark.

``listed`` are fixed sizes, ``draw`` gives others of the same ranges,
``prepare`` the inputs and handles such a program holds, ``run`` one pass,
``work`` the bytes and operations a pass cannot do without and ``exact`` the
outputs in 64 bits by plain torch, without this package's kernels.
"""
import math

import numpy as np
import torch

from pdspy_amd import configs, rt
from pdspy_amd.inputs import AU, arcsec

DPC = 140.0
FIELD = 2.0          # arcsec
H_PL, C_L, K_B = 6.6260755e-27, 2.99792458e10, 1.380658e-16


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # a first look at a model: few packets, plain walk; one long random
        # walk after another in the thick midplane (latency)
        dict(name="thermal_disk_1e4", kind="thermal", model="disk", nr=64, nt=64, nphi=1,
             nphot=10000, mrw=0, max_events=200000),
        # the benchmark's disk + envelope with the modified random walk, at the
        # photon count a sampler gives a walker
        dict(name="thermal_env_1e6_mrw", kind="thermal", model="env", nr=256, nt=128, nphi=1,
             nphot=1000000, mrw=1, max_events=100000),
        # 3-D spiral, Henyey-Greenstein scattering
        dict(name="thermal_spiral_2e6_hg", kind="thermal", model="spiral", nr=64, nt=32, nphi=32,
             nphot=2000000, mrw=1, max_events=200000),
        # one channel map of the disk + envelope, one ray per pixel
        dict(name="image_256", kind="image", model="env", nr=256, nt=128, nphi=1, npix=256,
             incl=60.0, pa=0.0, phi=0.0, lam=1300.0, nrefine=0),
        # the same image as run_image makes it: RADMC-3D's sub-pixeling
        dict(name="image_256_refined", kind="image", model="env", nr=256, nt=128, nphi=1, npix=256,
             incl=60.0, pa=0.0, phi=0.0, lam=1300.0, nrefine=100),
        # image and its gradient to the cells' densities and temperatures
        dict(name="image_256_grad", kind="image_grad", model="env", nr=256, nt=128, nphi=1,
             npix=256, incl=60.0, pa=0.0, phi=0.0, lam=1300.0),
        # 3-D model, turned camera, with the scattering source before the image
        dict(name="scat_image_512_3d", kind="scat_image", model="spiral", nr=128, nt=64, nphi=64,
             npix=512, incl=40.0, pa=25.0, phi=30.0, lam=870.0, nphot=100000),
        # a small image at a few baselines: the smallest call
        dict(name="vis_64_k500", kind="vis", npix=64, K=500),
        # a fit's data set: visibilities and their transpose
        dict(name="vis_256_k5e4_adj", kind="vis_adj", npix=256, K=50000),
        # a large data set
        dict(name="vis_256_k1e6", kind="vis", npix=256, K=1000000),
        # galario's gridded method on a large image, a large data set
        dict(name="grid_1024_k1e6", kind="grid", npix=1024, K=1000000),
        # one step of a sampler: every walker's thermal run, scattering source,
        # image, visibilities, chi^2 and gradient
        dict(name="sampler_step_6", kind="sampler", walkers=6, npix=128, K=2000, nphot=20000,
             nphot_scat=20000, mrw=1, max_events=100000),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["thermal", "thermal", "image", "image", "image_grad", "scat_image", "vis",
                       "vis", "vis_adj", "vis_adj", "grid", "sampler"])
    if kind in ("vis", "vis_adj"):
        npix = _log(rng, 48, 512)
        return dict(kind=kind, npix=npix, K=_log(rng, 300, 1000000 * (200 / max(npix, 200)) ** 2))
    if kind == "grid":
        return dict(kind=kind, npix=_log(rng, 64, 1024), K=_log(rng, 300, 1000000))
    if kind == "sampler":
        return dict(kind=kind, walkers=rng.randint(1, 6), npix=_log(rng, 32, 128),
                    K=_log(rng, 300, 2000), nphot=_log(rng, 2000, 20000),
                    nphot_scat=rng.choice([0, 20000]), mrw=rng.choice([0, 1]), max_events=50000)
    model = rng.choice(["disk", "env", "spiral"])
    nr, nt = _log(rng, 32, 256), 2 * _log(rng, 12, 64)
    nphi = 1
    if model == "spiral":
        nr, nt, nphi = _log(rng, 32, 128), 2 * _log(rng, 8, 32), _log(rng, 8, 64)
    c = dict(kind=kind, model=model, nr=nr, nt=nt, nphi=nphi)
    if kind == "thermal":
        c.update(nphot=_log(rng, 1000, 300000), mrw=1 if model == "env" else rng.choice([0, 1]),
                 max_events=50000)
        return c
    c.update(npix=_log(rng, 40, 256), incl=round(rng.uniform(3.0, 87.0), 3),
             pa=round(rng.uniform(0.0, 180.0), 3), phi=round(rng.uniform(1.0, 359.0), 3),
             lam=round(math.exp(rng.uniform(math.log(2.0), math.log(3000.0))), 3))
    if kind == "image":
        c.update(nrefine=rng.choice([0, 0, 100]))
        if c["nrefine"]:
            c.update(npix=min(c["npix"], 128))
    if kind == "scat_image":
        c.update(nphot=_log(rng, 10000, 200000))
    return c


# ---------------------------------------------------------------- inputs
def _model(case, seed):
    """Model arrays of one parameter set drawn by the seed (host, FP64)."""
    rng = np.random.default_rng([seed, 1])
    if case["model"] == "disk":
        m = configs.disk_c1(case["nr"], case["nt"], case["nphi"])
    elif case["model"] == "env":
        m = configs.disk_envelope(case["nr"], case["nt"], case["nphi"],
                                  mdisk=1e-3 * 10 ** rng.uniform(-0.15, 0.15),
                                  plrho=1.75 + rng.uniform(-0.05, 0.05),
                                  menv=0.1 * 10 ** rng.uniform(-0.15, 0.15))
    else:
        m = configs.spiral_3d(case["nr"], case["nt"], case["nphi"],
                              pitch_deg=rng.uniform(12.0, 18.0), amp=rng.uniform(0.2, 0.4))
    return rt.model_arrays(m.grid, hg=case["model"] == "spiral")


def _temperature(arr, seed):
    """A smooth temperature with Monte Carlo noise, as a thermal run leaves it."""
    rng = np.random.default_rng([seed, 2])
    nr, nt, nphi = len(arr["rw"]) - 1, len(arr["tw"]) - 1, len(arr["pw"]) - 1
    r = np.sqrt(arr["rw"][1:] * arr["rw"][:-1]) / AU
    th = 0.5 * (arr["tw"][1:] + arr["tw"][:-1])
    T = 180.0 * r[None, None, :] ** -0.45 * (0.6 + 0.4 * np.cos(th) ** 2)[None, :, None]
    T = np.broadcast_to(T, (nphi, nt, nr)) * (1.0 + 0.03 * rng.standard_normal((nphi, nt, nr)))
    return np.ascontiguousarray(T.reshape(-1).astype(np.float32))


def _sky(npix, seed):
    """An inclined ring with a compact core and pixel noise, Jy per pixel."""
    rng = np.random.default_rng([seed, 3])
    x = (np.arange(npix) - npix // 2) / npix
    X, Y = np.meshgrid(x, x)
    R = np.hypot(X, Y / rng.uniform(0.4, 0.9))
    img = np.exp(-0.5 * ((R - rng.uniform(0.15, 0.25)) / 0.04) ** 2)
    img += 5.0 * np.exp(-0.5 * (R / 0.03) ** 2)
    img *= 1.0 + 0.01 * rng.standard_normal(img.shape)
    return np.ascontiguousarray((img / img.sum()).astype(np.float32))


def _camera(case, pix_cm, **kw):
    return rt.DeviceModel.camera(case["npix"], pix_cm, case["lam"], incl=case["incl"],
                                 pa=case["pa"], phi=case["phi"], **kw)


def _uv(case, seed):
    # 15 - 2000 m baselines at 1.3 mm; the gridded method needs them on the
    # image's uv grid, which they are for these pixels
    u, v = configs.uv_points(case["K"], seed=seed)
    if case["kind"] == "grid":
        lim = 0.98 * (case["npix"] // 2 - 1) / (FIELD * arcsec)
        s = min(1.0, lim / max(np.abs(u).max(), np.abs(v).max()))
        u, v = u * s, v * s
    return u, v


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case, seed=seed)
    dev = "cuda"
    if kind == "thermal":
        st["dm"] = rt.DeviceModel(_model(case, seed))
    elif kind in ("image", "image_grad", "scat_image"):
        arr = _model(case, seed)
        pix = FIELD / case["npix"] * DPC * AU
        st["dm"] = rt.DeviceModel(arr)
        st["pix"] = pix
        st["T"] = torch.tensor(_temperature(arr, seed), device=dev)
        st["cam"] = _camera(case, pix, nrefine=case.get("nrefine", 0))
        if kind == "image_grad":
            rho = arr["rho"].reshape(arr["rho"].shape[0], -1)
            st["logrho"] = torch.tensor(np.log(np.maximum(rho, 1e-36)).astype(np.float32),
                                        device=dev, requires_grad=True)
            st["T"].requires_grad_(True)
            st["gimg"] = torch.tensor(_cotangent(case, seed), device=dev)
    elif kind in ("vis", "vis_adj", "grid"):
        u, v = _uv(case, seed)
        st["img"] = torch.tensor(_sky(case["npix"], seed), device=dev)
        st["dxy"] = FIELD / case["npix"] * arcsec
        st["u"] = torch.tensor(u, dtype=torch.float64, device=dev)
        st["v"] = torch.tensor(v, dtype=torch.float64, device=dev)
        if kind == "vis_adj":
            st["gre"], st["gim"] = (torch.tensor(g, device=dev) for g in _residuals(case, seed))
    else:
        st.update(_walkers(case, seed))
    return st


def _cotangent(case, seed):
    rng = np.random.default_rng([seed, 4])
    n = case["npix"]
    return rng.standard_normal((n, n)).astype(np.float32)


def _residuals(case, seed):
    rng = np.random.default_rng([seed, 5])
    return (rng.standard_normal(case["K"]).astype(np.float32),
            rng.standard_normal(case["K"]).astype(np.float32))


def _walkers(case, seed):
    """A batch of models, their data and the step's buffers, as a sampler keeps them."""
    rng = np.random.default_rng([seed, 6])
    n, npix, K = case["walkers"], case["npix"], case["K"]
    pixel = FIELD / npix
    u, v = (torch.tensor(x, dtype=torch.float64, device="cuda")
            for x in configs.uv_points(K, seed=seed))
    models, items, img, chi2, glr, gT, keep = [], [], [], [], [], [], []
    f32 = dict(dtype=torch.float32, device="cuda")
    for i in range(n):
        arr = rt.model_arrays(configs.disk_envelope(
            nr=(64, 48, 64)[i % 3], nt=(64, 32, 32)[i % 3],
            mdisk=10 ** rng.uniform(-4.5, -3), menv=10 ** rng.uniform(-3, -1.5)).grid)
        m = rt.DeviceModel(arr)
        cam = rt.DeviceModel.camera(npix, pixel * DPC * AU, 1300.0,
                                    incl=float(rng.uniform(5.0, 85.0)))
        re = torch.tensor(0.5 + 0.2 * rng.standard_normal(K), **f32)
        im = torch.tensor(0.2 * rng.standard_normal(K), **f32)
        w = torch.full((K,), 1.0 / 0.04, **f32)
        models.append(m)
        img.append(torch.zeros((npix, npix), **f32))
        chi2.append(torch.zeros(1, dtype=torch.float64, device="cuda"))
        glr.append(torch.zeros((m.nspec, m.ncell), **f32))
        gT.append(torch.zeros(m.ncell, **f32))
        items.append(rt.Batch.item(cam, pixel * arcsec, u, v, re, im, w, img[i], chi2[i], glr[i],
                                   gT[i], scale=(pixel * arcsec) ** 2 / 1e-23,
                                   nphot_scat=case["nphot_scat"]))
        keep.append((u, v, re, im, w))
    nphot = np.array([case["nphot"] * (1 + i % 3) // 2 for i in range(n)], dtype=np.uint64)
    return dict(batch=rt.Batch(models), items=items, img=img, chi2=chi2, glr=glr, gT=gT,
                keep=keep, nphot=nphot, seeds=np.arange(n, dtype=np.uint64) + np.uint64(seed),
                opts=dict(max_events=case["max_events"], mrw=case["mrw"]))


# ---------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "thermal":
        dm = st["dm"]
        dm.thermal(case["nphot"], st["seed"], mrw=case["mrw"], max_events=case["max_events"])
        return dm.temperature()
    if kind == "image":
        return st["dm"].image(st["cam"], st["T"])
    if kind == "image_grad":
        from pdspy_amd import autograd
        img = autograd.image(st["logrho"], st["T"], st["dm"], st["cam"])
        g = torch.autograd.grad(img, (st["logrho"], st["T"]), grad_outputs=st["gimg"])
        return [img.detach(), g[0], g[1]]
    if kind == "scat_image":
        dm = st["dm"]
        J, _ = dm.scattering_source(case["lam"], case["nphot"], st["T"], seed=st["seed"])
        return [J, dm.image(_camera(case, st["pix"], jscat=J), st["T"])]
    if kind == "vis":
        return list(rt.vis_dft(st["img"], st["dxy"], st["u"], st["v"], 1e-7, -2e-7))
    if kind == "vis_adj":
        n = case["npix"]
        re, im = rt.vis_dft(st["img"], st["dxy"], st["u"], st["v"], 1e-7, -2e-7)
        g = rt.vis_dft_adjoint(st["gre"], st["gim"], n, n, st["dxy"], st["u"], st["v"], 1e-7, -2e-7)
        return [re, im, g]
    if kind == "grid":
        return list(rt.vis_grid(st["img"], st["dxy"], st["u"], st["v"], 1e-7, -2e-7,
                                conv="galario"))
    st["batch"].step(st["items"], st["nphot"], st["seeds"], **st["opts"])
    # chi^2 is a sum over FP32 visibilities: its FP64 word carries FP32 accuracy
    return [st["img"], [c.float() for c in st["chi2"]], st["glr"], st["gT"]]


# ---------------------------------------------------------------- least work
def work(case):
    kind = case["kind"]
    if kind in ("vis", "vis_adj", "grid"):
        n, K = case["npix"], case["K"]
        px = n * n
        # a transform of the image and its value at every point; the points
        # are read (u, v in FP64) and the visibilities written once
        fl = 5.0 * px * math.log2(px) + 30.0 * K
        by = 4.0 * px + 24.0 * K
        if kind == "vis_adj":
            fl, by = 2 * fl, 2 * by
        return dict(bytes=by, flops=fl)
    if kind == "thermal":
        nc = case["nr"] * case["nt"] * case["nphi"]
        S = 2 if case["model"] == "env" else 1
        # a packet crosses a grid's radial walls once on its way out, with one
        # wall distance and one tally per crossing
        steps = case["nphot"] * case["nr"]
        return dict(bytes=12.0 * S * nc, flops=60.0 * steps)
    if kind == "sampler":
        nc, n, w = 64 * 64, case["npix"], case["walkers"]
        return dict(bytes=w * (40.0 * nc + 8.0 * n * n + 36.0 * case["K"]),
                    flops=w * (case["nphot"] * 64 * 60.0 + n * n * 128 * 40.0))
    nc = case["nr"] * case["nt"] * case["nphi"]
    S = 2 if case["model"] == "env" else 1
    n = case["npix"]
    # per ray one radial wall in and out, a wall distance and one attenuation
    # per crossing
    fl = n * n * 2.0 * case["nr"] * 20.0
    by = 4.0 * (S + 1) * nc + 4.0 * n * n
    if kind == "image_grad":
        fl, by = 3 * fl, 2 * by
    if kind == "scat_image":
        by += 8.0 * nc
        fl += case["nphot"] * case["nr"] * 60.0
    return dict(bytes=by, flops=fl)


# ---------------------------------------------------------------- 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind == "image":
        return _exact_image(case, seed)
    if kind == "image_grad":
        return _exact_image(case, seed, _cotangent(case, seed))
    if kind in ("vis", "vis_adj"):
        return _exact_vis(case, seed)
    if kind == "grid":
        return _exact_grid(case, seed)
    return None     # Monte Carlo


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _exact_vis(case, seed):
    dev, n = _dev(), case["npix"]
    img = torch.tensor(_sky(n, seed), device=dev).double()
    u, v = (torch.tensor(a, dtype=torch.float64, device=dev) for a in _uv(case, seed))
    x = (torch.arange(n, device=dev, dtype=torch.float64) - n // 2) * (FIELD / n * arcsec)
    res = [torch.tensor(g, device=dev).double() for g in _residuals(case, seed)] \
        if case["kind"] == "vis_adj" else None
    out, g = [], torch.zeros((n, n), dtype=torch.float64, device=dev)
    for i in range(0, case["K"], 20000):
        uu, vv = u[i:i + 20000, None], v[i:i + 20000, None]
        au, av = -2 * math.pi * uu * x[None], -2 * math.pi * vv * x[None]
        ar, ai, br, bi = torch.cos(au), torch.sin(au), torch.cos(av), torch.sin(av)
        ph = -2 * math.pi * (uu * 1e-7 - vv * 2e-7)
        c, s = torch.cos(ph), torch.sin(ph)
        rr, ri = ar @ img.T, ai @ img.T
        vr = (rr * br - ri * bi).sum(1, keepdim=True)
        vi = (rr * bi + ri * br).sum(1, keepdim=True)
        out.append(torch.cat([vr * c - vi * s, vr * s + vi * c], 1))
        if res is not None:
            gr, gi = res[0][i:i + 20000, None], res[1][i:i + 20000, None]
            hr, hi = gr * c + gi * s, gr * s - gi * c
            g += (br * hr - bi * hi).T @ ar - (br * hi + bi * hr).T @ ai
    o = torch.cat(out)
    return [o[:, 0].contiguous(), o[:, 1].contiguous()] + ([g] if res is not None else [])


def _exact_grid(case, seed):
    n = case["npix"]
    img = _sky(n, seed).astype(np.float64)[::-1]
    F = np.fft.fftshift(np.fft.fft2(np.fft.ifftshift(img)))
    u, v = _uv(case, seed)
    s = n * (FIELD / n * arcsec)
    fa, fb = -u * s + n // 2, -v * s + n // 2
    a, b = np.floor(fa).astype(int), np.floor(fb).astype(int)
    ta, tb = fa - a, fb - b
    V = ((1 - ta) * (1 - tb) * F[b, a] + ta * (1 - tb) * F[b, a + 1] +
         (1 - ta) * tb * F[b + 1, a] + ta * tb * F[b + 1, a + 1])
    V = V * np.exp(-2j * math.pi * (u * 1e-7 - v * 2e-7))
    return [np.ascontiguousarray(V.real), np.ascontiguousarray(V.imag)]


def _exact_image(case, seed, gimg=None):
    """Formal solution: every ray is cut at all its intersections with the
    spheres, cones and planes of the grid, each piece lies in the cell its
    middle is in, and the pieces are summed in order."""
    dev, dt = _dev(), torch.float64
    arr = _model(case, seed)
    t = lambda a: torch.tensor(np.asarray(a, dtype=float), dtype=dt, device=dev)
    nr, nt, nphi = case["nr"], case["nt"], case["nphi"]
    rw, tw, pw = t(arr["rw"] / AU), t(arr["tw"]), t(arr["pw"])
    mirror = abs(float(arr["tw"][-1]) - math.pi / 2) < 1e-6
    S = arr["rho"].shape[0]
    kap = [math.exp(np.interp(math.log(case["lam"]), np.log(arr["lam_um"]), np.log(k)))
           for k in arr["kabs"]]
    rho = arr["rho"].reshape(S, -1)
    T = t(_temperature(arr, seed))
    if gimg is not None:
        logrho = torch.tensor(np.log(np.maximum(rho, 1e-36)).astype(np.float32), device=dev)
        logrho = logrho.double().requires_grad_(True)
        T.requires_grad_(True)
        alpha = sum(torch.exp(logrho[s]) * kap[s] for s in range(S)) * AU
    else:
        alpha = sum(t(rho[s]) * kap[s] for s in range(S)) * AU
    nu = C_L / (case["lam"] * 1e-4)
    src = 2 * H_PL * nu ** 3 / C_L ** 2 / torch.expm1(H_PL * nu / (K_B * T))
    i, ph, pa = (math.radians(case[k]) for k in ("incl", "phi", "pa"))
    nv = np.array([math.sin(i) * math.sin(ph), -math.sin(i) * math.cos(ph), math.cos(i)])
    ex = np.array([math.cos(ph), math.sin(ph), 0.0])
    ey = np.cross(nv, ex)
    npix = case["npix"]
    pix = FIELD / npix * DPC
    ct2 = torch.cos(tw[1:-1]) ** 2
    rc = 0.5 * (rw[1:] + rw[:-1])
    size = torch.minimum(rw[1:] - rw[:-1], rc * (tw[1:] - tw[:-1])[:, None])[None].repeat(nphi, 1, 1)
    if nphi > 1:
        sm = torch.sin(0.5 * (tw[1:] + tw[:-1]))
        size = torch.minimum(size, (rc * sm[:, None])[None] * (pw[1:] - pw[:-1])[:, None, None])
    size = size.reshape(-1)

    def trace(X, Y):
        xp, yp = X * math.cos(pa) + Y * math.sin(pa), -X * math.sin(pa) + Y * math.cos(pa)
        p0 = [(xp * ex[k] + yp * ey[k])[:, None] for k in range(3)]
        d = -nv
        b2 = p0[0] ** 2 + p0[1] ** 2 + p0[2] ** 2
        # a wall that a ray misses becomes a cut at its nearest point, which
        # does no harm
        sr = torch.sqrt(torch.clamp(rw[None] ** 2 - b2, min=0.0))
        # z^2 = ct2 r^2 along the ray
        A = d[2] ** 2 - ct2[None]
        B = p0[2] * d[2]
        Cq = p0[2] ** 2 - ct2[None] * b2
        sq = torch.sqrt(torch.clamp(B * B - A * Cq, min=0.0))
        q = -(B + torch.where(B >= 0, sq, -sq))
        r1, r2 = q / A, Cq / torch.where(q == 0, torch.full_like(q, 1e-300), q)
        parts = [-sr, sr, r1, r2, (-p0[2] / d[2])]
        if nphi > 1:
            cp, sp = torch.cos(pw[:-1])[None], torch.sin(pw[:-1])[None]
            parts.append((p0[0] * sp - p0[1] * cp) / (d[1] * cp - d[0] * sp))
        so = sr[:, -1:]
        s = torch.cat([torch.minimum(torch.maximum(torch.nan_to_num(x, nan=0.0), -so), so)
                       for x in parts], 1)
        s, _ = torch.sort(s, 1)
        ds, sm_ = s[:, 1:] - s[:, :-1], 0.5 * (s[:, 1:] + s[:, :-1])
        x, y, z = (p0[k] + sm_ * d[k] for k in range(3))
        r = torch.sqrt(x * x + y * y + z * z)
        th = torch.atan2(torch.sqrt(x * x + y * y), z.abs() if mirror else z)
        ir = torch.searchsorted(rw, r.contiguous(), right=True) - 1
        it = (torch.searchsorted(tw, th.contiguous(), right=True) - 1).clamp(0, nt - 1)
        ip = 0
        if nphi > 1:
            fi = torch.atan2(y, x)
            fi = torch.where(fi < 0, fi + 2 * math.pi, fi)
            ip = (torch.searchsorted(pw, fi.contiguous(), right=True) - 1).clamp(0, nphi - 1)
        inside = (ir >= 0) & (ir < nr) & (ds > 0)
        c = ir.clamp(0, nr - 1) + nr * (it + nt * ip)
        dtau = torch.where(inside, alpha[c] * ds, torch.zeros_like(ds))
        tau0 = torch.cumsum(dtau, 1) - dtau
        I = (torch.exp(-tau0) * -torch.expm1(-dtau) * src[c]).sum(1)
        lmin = torch.where(inside & (tau0 <= 40.0), size[c], torch.full_like(ds, 3e38)).amin(1)
        return I, lmin

    def render(X, Y, level):
        out = []
        step = 4096 if dev == "cpu" else 16384
        for k in range(0, X.numel(), step):
            I, lmin = trace(X[k:k + step], Y[k:k + step])
            side = pix * 0.5 ** level
            split = (side > lmin) if level < min(case.get("nrefine", 0), 24) else \
                torch.zeros_like(lmin, dtype=torch.bool)
            if split.any():
                xs, ys, h = X[k:k + step][split], Y[k:k + step][split], 0.25 * side
                sub = render(torch.cat([xs - h, xs + h, xs - h, xs + h]),
                             torch.cat([ys - h, ys - h, ys + h, ys + h]), level + 1)
                I = I.clone()
                I[split] = sub.reshape(4, -1).mean(0)
            out.append(I)
        return torch.cat(out)

    g = (torch.arange(npix, dtype=dt, device=dev) - npix // 2) * pix
    Y, X = (a.reshape(-1) for a in torch.meshgrid(g, g, indexing="ij"))
    # the star sits at the origin: its ray runs up one column of cells
    th_n = math.acos(abs(nv[2])) if mirror else math.acos(nv[2])
    it = min(int(np.searchsorted(arr["tw"], th_n, side="right")) - 1, nt - 1)
    ip = 0
    if nphi > 1:
        f = math.atan2(nv[1], nv[0]) % (2 * math.pi)
        ip = min(int(np.searchsorted(arr["pw"], f, side="right")) - 1, nphi - 1)
    col = nr * (it + nt * ip)
    Rs, Ts = arr["stars"][0][:2]
    F = math.pi * Rs ** 2 / (pix * AU) ** 2 * 2 * H_PL * nu ** 3 / C_L ** 2 / \
        math.expm1(H_PL * nu / (K_B * Ts))

    def star():
        return F * torch.exp(-(alpha[col:col + nr] * (rw[1:] - rw[:-1])).sum())

    centre = (npix // 2) * npix + npix // 2
    if gimg is None:
        with torch.no_grad():
            img = render(X, Y, 0)
            img[centre] += star()
            return img.reshape(npix, npix)
    w = torch.tensor(gimg, device=dev).double().reshape(-1)
    img = torch.empty(npix * npix, dtype=dt, device=dev)
    gl, gt = torch.zeros_like(logrho), torch.zeros_like(T)
    step = 2048 if dev == "cpu" else 8192
    for k in range(0, X.numel(), step):
        I, _ = trace(X[k:k + step], Y[k:k + step])
        L = (I * w[k:k + step]).sum()
        img[k:k + step] = I.detach()
        a, b = torch.autograd.grad(L, (logrho, T), retain_graph=True)
        gl, gt = gl + a, gt + b
    Is = star()
    a, = torch.autograd.grad(Is * w[centre], logrho, retain_graph=True)
    img[centre] += Is.detach()
    return [img.reshape(npix, npix), gl + a, gt]
