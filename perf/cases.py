"""The framework's work as its users call it, for measuring.

Every case goes through the public entry points (gpuvmem_amd.device,
gpuvmem_amd.warmstart and the C ABI of include/gvm_hip.h) on a seeded
synthetic observation: an antenna array, its earth-rotation tracks in time
order (as measurement sets hold them), a sky of Gaussian components and
thermal noise.  The image sizes, arrays, tracks and objectives are those of
the repository's workloads (512^2 + alpha in 32 of its 256 channels), and
odd ones between.

kind "evaluate"  one objective value and its gradient (an optimiser iteration's
                 pair of calls), any number of channels, each adjoint form
kind "probe"     one line-search probe: the trial image and its objective value
kind "optimise"  a whole optimiser call with given step lengths
kind "grid"      Briggs weighting and convolutional gridding of raw rows
kind "train"     one training step of the warm-start network
kind "predict"   the warm start's initial image from a dirty image (host arrays)
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from gpuvmem_amd import native
from gpuvmem_amd.device import Context, DeviceBuffer, Objective, fw_config
from gpuvmem_amd.gridding import GriddingKernel, apply_weighting_dev
from gpuvmem_amd.problem import Problem
from gpuvmem_amd.warmstart import UNet, WarmStart, unet_shapes

LIGHT = 2.99792458e8
RAD = math.pi / 180.0
CELL = 0.05  # arcsec, of every workload
DISH, PB_FACTOR = 12.0, 1.13
NOISE = 1e-3  # Jy per visibility
LAMBDAS = (0.01, 1e-3, 2e-4)
PRIORS = {"entropy": ("Entropy", 0, 0.001), "tsv": ("TotalSquaredVariation", 1, 0.0),
          "laplacian": ("Laplacian", 2, 0.0)}


def _observe(npix, antennas, dumps, radius_m, **kw):
    """antennas * (antennas - 1) / 2 baselines at `dumps` times per channel."""
    d = dict(kind="evaluate", npix=npix, antennas=antennas, dumps=dumps, radius_m=radius_m,
             layout="gaussian", hours=4.0, ghz=230.0, channels=1, flagged=0.0, components=8,
             adjoint="bf16x3", flag=0, priors="entropy tsv")
    d.update(kw)
    return d


def listed():
    return [
        # the smallest problems: interactive runs and tests, launches and latency
        _observe(64, 8, 61, 250.0, name="evaluate 64sq", hours=1.0, priors="entropy"),
        # the 256^2 / 36,000-visibility workload and its objective
        _observe(256, 25, 120, 250.0, name="evaluate 256sq", layout="uniform", hours=1.0,
                 priors="entropy"),
        # the 512^2 warm-start workload's rows in the FP16 split form
        _observe(512, 50, 840, 500.0, name="evaluate 512sq f16x3", layout="uniform",
                 hours=7.0 / 3.0, adjoint="f16x3", priors="entropy"),
        # the headline: 1024^2, 1,764,000 visibilities, chi2 + entropy + TSV
        _observe(1024, 50, 1440, 1000.0, name="evaluate 1024sq", components=200),
        # the plain FP32 form on a ragged row count (43 antennas, 1,084,503 rows)
        _observe(1024, 43, 1201, 1000.0, name="evaluate 1024sq f32", adjoint="f32",
                 components=40),
        # the 2048^2 / 4,354,560-visibility precision workload, all three priors
        _observe(2048, 64, 2160, 2500.0, name="evaluate 2048sq", layout="uniform", hours=6.0,
                 ghz=60.0, components=200, priors="entropy tsv laplacian"),
        # multi-frequency synthesis: I_nu_0 + alpha, flagged channels of uneven
        # length, the alpha gradient of the flag schedule
        _observe(512, 35, 504, 1000.0, name="evaluate mfs 512sq", hours=1.4, channels=32,
                 flagged=0.4, components=35, flag=1, priors="entropy"),
        # a line-search probe of the headline problem: about 15 per gradient
        _observe(1024, 50, 1440, 1000.0, name="probe 1024sq", kind="probe", components=200),
        # a whole optimiser call on the 256^2 workload
        _observe(256, 25, 120, 250.0, name="optimise 256sq", kind="optimise", layout="uniform",
                 hours=1.0, priors="entropy", iterations=4),
        # the gridded mode's set-up of the headline rows with a 7 x 7 kernel
        _observe(1024, 50, 1440, 1000.0, name="grid 1024sq", kind="grid", taps=7, robust=0.0),
        # training the warm start at 512^2 (6 levels, 32 channels, BF16 weights)
        dict(name="train 512sq", kind="train", npix=512, levels=6, base=32, batch=4),
        # the warm start of one 1024^2 observation with the committed network's shape
        dict(name="predict 1024sq", kind="predict", npix=1024, levels=5, base=16, images=1),
    ]


def draw(rng):
    def logint(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["evaluate"] * 5 + ["probe", "optimise", "grid", "train", "predict"])
    if kind == "train":
        npix = rng.choice([64, 96, 128, 192, 256, 384])
        return dict(kind="train", npix=npix, levels=rng.choice([3, 4, 5]),
                    base=rng.choice([8, 12, 16, 32]), batch=rng.randint(1, 8))
    if kind == "predict":
        return dict(kind="predict", npix=rng.choice([128, 256, 320, 512, 768, 1024]),
                    levels=rng.choice([3, 4, 5]), base=rng.choice([8, 16, 24]),
                    images=rng.randint(1, 3))
    npix = rng.choice([64, 128, 256, 512, 1024, 2048]) if kind in ("evaluate", "probe") else \
        rng.choice([64, 128, 256, 512])
    most = 60_000 if kind == "optimise" else 1_800_000
    antennas = logint(5, 60)
    baselines = antennas * (antennas - 1) // 2
    dumps = max(1, min(logint(3, 1500), most // baselines))
    ghz = 60.0 if npix == 2048 else rng.uniform(100.0, 230.0)
    # baselines inside the uv plane of the cell size (Nyquist at 2.06e6 wavelengths)
    radius = 0.5 * rng.uniform(0.2, 0.6) * 2.06e6 * LIGHT / (ghz * 1e9)
    c = _observe(npix, antennas, dumps, round(radius, 1), kind=kind, ghz=round(ghz, 3),
                 layout=rng.choice(["uniform", "gaussian"]), hours=round(rng.uniform(0.3, 6.0), 2),
                 components=logint(3, 100), priors=rng.choice(
                     ["", "entropy", "entropy tsv", "entropy tsv laplacian"]))
    if kind == "evaluate":
        c["adjoint"] = rng.choice(["bf16x3", "bf16x3", "f16x3", "f32"])
        if npix <= 512 and rng.random() < 0.4:
            c.update(channels=rng.randint(2, 12), flagged=round(rng.uniform(0.0, 0.4), 3),
                     flag=rng.choice([0, 1]), dumps=max(1, dumps // 12))
    if kind == "optimise":
        c.update(iterations=rng.randint(2, 5))
    if kind == "grid":
        c.update(taps=rng.choice([1, 3, 5, 7]), robust=round(rng.uniform(-2.0, 2.0), 2),
                 dumps=max(1, min(dumps, 400_000 // baselines)))
    return c


# ---------------------------------------------------------------------------
# the observation (torch, FP64)
# ---------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(g, n, a, b):
    return a + (b - a) * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def _baselines(case, g):
    """(rows, 3) uvw in metres, time-major."""
    n, r = case["antennas"], case["radius_m"]
    th = _uniform(g, n, 0.0, 2.0 * math.pi)
    if case["layout"] == "uniform":
        rad = r * torch.sqrt(_uniform(g, n, 0.0, 1.0))
    else:  # Gaussian-radial, folded into the disk
        rad = (0.5 * r * torch.randn(n, generator=g, device="cuda", dtype=torch.float64)).abs() % r
    east, north = rad * torch.cos(th), rad * torch.sin(th)
    a, b = torch.triu_indices(n, n, 1, device="cuda")
    de, dn = east[b] - east[a], north[b] - north[a]
    lat, dec = -23.03 * RAD, -30.0 * RAD
    lx, ly, lz = -math.sin(lat) * dn, de, math.cos(lat) * dn
    t = (torch.arange(case["dumps"], device="cuda", dtype=torch.float64) + 0.5) / case["dumps"]
    h = ((t - 0.5) * case["hours"] * 15.0 * RAD)[:, None]
    sh, ch = torch.sin(h), torch.cos(h)
    sd, cd = math.sin(dec), math.cos(dec)
    u = sh * lx + ch * ly
    v = -sd * ch * lx + sd * sh * ly + cd * lz
    w = cd * ch * lx - cd * sh * ly + sd * lz
    return torch.stack([u.reshape(-1), v.reshape(-1), w.reshape(-1)], 1)


def _sky(case, g):
    """(x, y, sigma in pixels from the centre, flux, alpha) per component."""
    k = case["components"]
    r = 0.22 * case["npix"] * torch.sqrt(_uniform(g, k, 0.0, 1.0))
    th = _uniform(g, k, 0.0, 2.0 * math.pi)
    flux = torch.exp(_uniform(g, k, math.log(1e-2), 0.0))
    multi = case["channels"] > 1
    return (torch.round(r * torch.cos(th)), torch.round(r * torch.sin(th)), _uniform(g, k, 1.0, 8.0),
            flux, _uniform(g, k, -1.0, 3.0) if multi else torch.zeros_like(flux))


def _frequencies(case):
    nu = case["ghz"] * 1e9
    if case["channels"] == 1:
        return [float(np.float32(nu))]
    k = np.arange(case["channels"])
    return [float(f) for f in np.float32(nu * (1.0 + (k + 0.5 - 0.5 * k.size) * 0.1333 / k.size))]


def _wavelength(freq):
    return float(np.float32(LIGHT) / np.float32(freq))


def _rows(case, seed):
    """Per channel (freq, uvw metres, Vo, weight), and the sky."""
    g = _generator(seed)
    uvw = _baselines(case, g)
    x, y, sig, flux, alpha = _sky(case, g)
    cell = CELL / 3600.0 * RAD
    freqs = _frequencies(case)
    nu0 = case["ghz"] * 1e9
    out = []
    for f in freqs:
        rows = uvw
        if case["flagged"] > 0.0:  # flagged rows are left out, another share of each channel
            share = case["flagged"] * float(_uniform(g, 1, 0.0, 1.0))
            rows = uvw[_uniform(g, len(uvw), 0.0, 1.0) >= share]
            rows = rows if len(rows) else uvw[:1]
        n = len(rows)
        u, v = rows[:, 0] / _wavelength(f), rows[:, 1] / _wavelength(f)
        vis = torch.zeros(n, device="cuda", dtype=torch.complex128)
        fx = flux * (f / nu0) ** alpha
        for k in range(len(flux)):
            amp = float(fx[k]) * torch.exp(-2.0 * math.pi ** 2 * (float(sig[k]) * cell) ** 2 * (u * u + v * v))
            ph = 2.0 * math.pi * (-u * float(x[k]) + v * float(y[k])) * cell
            vis += torch.polar(amp, ph)
        noise = torch.randn(n, 2, generator=g, device="cuda", dtype=torch.float64) * NOISE
        vo = (torch.view_as_real(vis) + noise).float().contiguous()
        weight = (_uniform(g, n, 0.5, 1.5) / NOISE ** 2).float().contiguous()
        out.append((f, rows.contiguous(), vo, weight))
    return out, (x, y, sig, flux, alpha)


def _beam(npix, freq):
    """The Gaussian primary beam, FP64, before the library's rounding to float."""
    o = torch.arange(npix, device="cuda", dtype=torch.float64) - npix // 2
    arc2 = ((o * CELL / 3600.0 * RAD) ** 2)[:, None] + ((o * CELL / 3600.0 * RAD) ** 2)[None]
    fwhm = PB_FACTOR * (LIGHT / freq) / DISH
    return torch.exp(-4.0 * math.log(2.0) * arc2 / fwhm ** 2)


def _problem(case, rows, sky):
    """What the set-up hands the objective: geometry, noise image and mask."""
    npix = case["npix"]
    nu0 = float(np.float32(case["ghz"] * 1e9))
    suu = svv = sw = 0.0
    for f, uvw, _, w in rows:
        w = w.double()
        suu += float((w * (uvw[:, 0] / _wavelength(f)) ** 2).sum())
        svv += float((w * (uvw[:, 1] / _wavelength(f)) ** 2).sum())
        sw += float(w.sum())
    cell = CELL / 3600.0 * RAD
    beam_px = max(1.0, 1.0 / (2.0 * math.pi * math.sqrt(suu * svv) / sw * cell * cell))
    jypix = 0.5 * math.sqrt(1.0 / sw) / beam_px
    pb = _beam(npix, nu0).float().double()
    noise = (jypix * pb.max() / pb).float()
    fg = float(noise.min())
    x, y, sig, flux, _ = sky
    o = torch.arange(npix, device="cuda", dtype=torch.float64) - npix // 2
    gx = torch.exp(-0.5 * ((o[None] - x[:, None]) / sig[:, None]) ** 2)
    gy = torch.exp(-0.5 * ((o[None] - y[:, None]) / sig[:, None]) ** 2)
    image = (gy * (flux / (2.0 * math.pi * sig ** 2))[:, None]).T @ gx
    nothing = np.zeros((0, 3))
    return Problem(
        M=npix, N=npix, deltax=-CELL / 3600.0, deltay=CELL / 3600.0, x0=float(npix // 2),
        y0=float(npix // 2), freq=rows[0][0], nu_0=nu0, uvw=nothing, vo=nothing[:, :2],
        weight=nothing[:, 0], noise=noise.cpu().numpy(), fg_scale=fg,
        noise_cut=float(np.float32(10.0 * fg)), beam_kind=native.GVM_BEAM_GAUSSIAN,
        antenna_diameter=DISH, pb_factor=float(np.float32(PB_FACTOR)),
        pb_cutoff=float(np.float32(10.0 * PB_FACTOR * _wavelength(min(r[0] for r in rows)) / DISH))), image


def _start_image(case, p, sky_image, seed):
    """An image part of the way to the sky, in the framework's units, with a
    spectral index where there are channels."""
    g = _generator(seed + 77)
    img = torch.zeros(2, p.N, p.M, device="cuda", dtype=torch.float64)
    img[0] = torch.clamp(0.5 * sky_image / p.fg_scale, min=p.minpix)
    if case["channels"] > 1:
        img[1] = _uniform(g, p.N * p.M, -1.0, 3.0).reshape(p.N, p.M)
    return img.float().contiguous()


def _direction(p, sky_image, img):
    """A search direction: from the image towards the sky."""
    d = torch.zeros_like(img)
    d[0] = (sky_image / p.fg_scale).float() - img[0]
    return d


class Memory:
    """A torch tensor as the framework's callers see device memory."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()

    def free(self):
        pass


class _View:
    """A framework buffer for torch.as_tensor: the tensor keeps this object, and
    with it the buffer's memory, alive after the network itself is gone."""

    def __init__(self, buf, shape, typestr="<f4"):
        self.buf = buf
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(buf.ptr, False),
                                             version=2)


def _tensor(buf, shape):
    return torch.as_tensor(_View(buf, tuple(shape)), device="cuda")


def _terms(case):
    return [("Chi2", -1, 0.0)] + [PRIORS[k] for k in case["priors"].split()]


def _steps(case, p, rows):
    """Step lengths of a damped descent: a share of the inverse of the weights' sum."""
    total = sum(float(r[3].double().sum()) for r in rows) * p.fg_scale ** 2
    return [0.3 / total] * case["iterations"]


def prepare(case, seed):
    if case["kind"] in ("train", "predict"):
        return _prepare_network(case, seed)
    rows, sky = _rows(case, seed)
    p, sky_image = _problem(case, rows, sky)
    state = dict(case=case)
    ctx = Context(p, adjoint=case["adjoint"], add_data=False)
    img = _start_image(case, p, sky_image, seed)
    if case["kind"] == "grid":
        n = len(rows[0][1])
        dx = p.deltax * RAD
        state.update(rows=rows, n=n, work=torch.empty(n, device="cuda"),
                     uvw=torch.zeros(ctx.n, 3, device="cuda", dtype=torch.float64),
                     vo=torch.zeros(ctx.n, 2, device="cuda"), w=torch.zeros(ctx.n, device="cuda"),
                     kernel=GriddingKernel.from_taps(_taps(case)), ctx=ctx, dx=dx)
        torch.cuda.synchronize()
        return state
    torch.cuda.synchronize()
    for f, uvw, vo, w in rows:
        ctx.add_dev(f, Memory(uvw), Memory(vo), Memory(w), len(uvw))
    obj = Objective(ctx, fw_config(_terms(case), lambdas=LAMBDAS, flag_opt=case["flag"]))
    xi = torch.zeros_like(img)
    state.update(obj=obj, image=Memory(img), xi=Memory(xi), ctx=ctx)
    torch.cuda.synchronize()
    if case["kind"] == "optimise":
        state.update(first=Memory(img.clone()), steps=_steps(case, p, rows))
        torch.cuda.synchronize()
        return state
    # an optimiser has evaluated before: the objective is past its first iteration
    obj.value(state["image"])
    obj.gradient(state["image"], state["xi"], 1)
    ctx.sync()
    if case["kind"] == "probe":
        state["direction"] = Memory(_direction(p, sky_image, img))
        state["trial"] = Memory(torch.zeros_like(img))
        torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "evaluate":
        obj = state["obj"]
        value = obj.value(state["image"])
        obj.gradient(state["image"], state["xi"], 1)
        return dict(value=value, gradient=state["xi"].tensor, image=state["image"].tensor)
    if case["kind"] == "probe":
        ctx, obj = state["ctx"], state["obj"]
        p = ctx.problem
        for k in (0, 1):
            native.check(ctx.lib.gvm_evaluate_xt(ctx.ctx, state["trial"].ptr, state["image"].ptr,
                                                 state["direction"].ptr, 0.25, k, int(k == 0),
                                                 p.minpix, p.eta), "gvm_evaluate_xt")
        return dict(value=obj.value(state["trial"]), image=state["trial"].tensor)
    if case["kind"] == "optimise":
        ctx, obj = state["ctx"], state["obj"]
        native.check(ctx.lib.gvm_vec_copy(ctx.ctx, state["image"].ptr, state["first"].ptr,
                                          2 * ctx.n), "gvm_vec_copy")
        obj.set_line_search_replay(state["steps"])
        result, path = obj.optimize(state["image"], "CG-FRPRMN", case["iterations"])
        return dict(value=result.final_value, path=path, image=state["image"].tensor)
    if case["kind"] == "grid":
        return _run_grid(state)
    if case["kind"] == "train":
        net = state["net"]
        net.forward()
        loss = net.loss(state["target"])
        net.backward()
        net.adam(lr=1e-4)
        return dict(loss=loss, output=state["y"], gradients=state["grads"], weights=state["weights"])
    return dict(image=state["ws"].predict(state["dirty"]))


# ---------------------------------------------------------------------------
# gridding
# ---------------------------------------------------------------------------
def _taps(case):
    k = np.arange(case["taps"]) - case["taps"] // 2
    t = np.exp(-0.5 * (k / max(1.0, case["taps"] / 4.0)) ** 2)
    return (t[:, None] * t[None]).astype(np.float32)


def _run_grid(state):
    ctx, case = state["ctx"], state["case"]
    freq, uvw, vo, weight = state["rows"][0]
    work = Memory(state["work"])
    native.check(ctx.lib.gvm_vec_copy(ctx.ctx, work.ptr, weight.data_ptr(), state["n"]), "copy")
    ctx.sync()
    apply_weighting_dev(ctx, "briggs", [(freq, Memory(uvw), work, state["n"])],
                        robust=case["robust"])
    count = C.c_long()
    kernel = state["kernel"].as_c()
    native.check(ctx.lib.gvm_grid_visibilities_dev(
        ctx.ctx, C.byref(kernel), freq, state["n"], uvw.data_ptr(), vo.data_ptr(), work.ptr,
        state["uvw"].data_ptr(), state["vo"].data_ptr(), state["w"].data_ptr(), ctx.n,
        C.byref(count)), "gvm_grid_visibilities_dev")
    # the gridded rows are the first `count` of each buffer
    return dict(count=count.value, weights=work.tensor, uvw=state["uvw"], vo=state["vo"],
                weight=state["w"])


def _exact_grid(case, seed):
    rows, sky = _rows(case, seed)
    p, _ = _problem(case, rows, sky)
    freq, uvw, vo, weight = rows[0]
    n = p.N
    lam = _wavelength(freq)
    du, dv = 1.0 / (n * p.deltax * RAD), 1.0 / (n * p.deltay * RAD)
    u, v = uvw[:, 0] / lam, uvw[:, 1] / lam
    w = weight.double()
    # Briggs weighting, rows with u < 0 mirrored
    s = torch.where(u < 0.0, -1.0, 1.0)
    x = (s * u / abs(du) + n // 2 + 0.5).to(torch.int64)
    y = (s * v / abs(dv) + n // 2 + 0.5).to(torch.int64)
    on = (x >= 0) & (x < n) & (y >= 0) & (y < n)
    at = torch.where(on, y * n + x, n * n)
    cells = torch.zeros(n * n + 1, device="cuda", dtype=torch.float64).index_add_(0, at, w)
    cells[n * n] = 0.0
    g = cells[: n * n].reshape(n, n)
    average = float((g[:, n // 2:] ** 2).sum()) / float(w.sum())
    f2 = (5.0 * 10.0 ** -case["robust"]) ** 2 / average
    w = torch.where(on, w / (1.0 + cells[at] * f2), 0.0)
    # every row and its Hermitian twin over the kernel's taps
    taps = torch.as_tensor(_taps(case), device="cuda").double()
    k, h = case["taps"], case["taps"] // 2
    sums = torch.zeros(4, n * n + 1, device="cuda", dtype=torch.float64)
    re, im = vo[:, 0].double(), vo[:, 1].double()
    for sign in (1.0, -1.0):
        j = (sign * u / du + n // 2 + 0.5).to(torch.int64)
        i = (sign * v / dv + n // 2 + 0.5).to(torch.int64)
        for a in range(k):
            for b in range(k):
                jj, ii = j + b - h, i + a - h
                ok = (jj >= 0) & (jj < n) & (ii >= 0) & (ii < n)
                at = torch.where(ok, ii * n + jj, n * n)
                t = float(taps[a, b])
                for q, val in enumerate((w * t, w * t * t, w * re * t, w * im * sign * t)):
                    sums[q].index_add_(0, at, val)
    ws, aux, sr, si = sums[:, : n * n]
    keep = torch.nonzero(torch.where(aux != 0.0, ws * ws / aux, 0.0) > 0.0)[:, 0]
    vo_out = torch.stack([sr[keep] / ws[keep], si[keep] / ws[keep]], 1)
    uu, vv = (keep % n - n // 2) * du * lam, (keep // n - n // 2) * dv * lam

    def whole(t):
        out = torch.zeros(n * n, *t.shape[1:], device="cuda", dtype=torch.float64)
        out[: len(t)] = t
        return out

    return dict(count=None, weights=w, uvw=whole(torch.stack([uu, vv, torch.zeros_like(uu)], 1)),
                vo=whole(vo_out), weight=whole(ws[keep] ** 2 / aux[keep]))


# ---------------------------------------------------------------------------
# the warm-start network
# ---------------------------------------------------------------------------
def _dirty(npix, count, g):
    """Blobs on sidelobe noise, as a dirty image looks."""
    o = torch.arange(npix, device="cuda", dtype=torch.float64) - npix / 2
    out = 0.02 * torch.randn(count, npix, npix, generator=g, device="cuda", dtype=torch.float64)
    for k in range(count):
        for x, y, s, a in zip(*(_uniform(g, 6, lo, hi).tolist() for lo, hi in
                                ((-0.25 * npix, 0.25 * npix), (-0.25 * npix, 0.25 * npix),
                                 (2.0, 10.0), (0.05, 1.0)))):
            out[k] += a * torch.exp(-0.5 * ((o - y) / s) ** 2)[:, None] * \
                torch.exp(-0.5 * ((o - x) / s) ** 2)[None]
    return out


def _bare_context():
    noise = np.ones((64, 64), np.float32)
    nothing = np.zeros((0, 3))
    return Context(Problem(
        M=64, N=64, deltax=-CELL / 3600.0, deltay=CELL / 3600.0, x0=32.0, y0=32.0, freq=230e9,
        nu_0=230e9, uvw=nothing, vo=nothing[:, :2], weight=nothing[:, 0], noise=noise,
        fg_scale=1.0, noise_cut=10.0, beam_kind=native.GVM_BEAM_GAUSSIAN, antenna_diameter=DISH,
        pb_factor=PB_FACTOR, pb_cutoff=1.0), add_data=False)


def _parameters(case, seed):
    """The network's start, (Co, Ci, K, K) weights scaled by the fan-in and biases, flat."""
    g = _generator(seed + 5)
    parts = []
    for name, co, ci, k in unet_shapes(case["levels"], case["base"]):
        std = math.sqrt((1.0 if name == "out" else 2.0) / (ci * k * k))
        parts.append(torch.randn(co * ci * k * k, generator=g, device="cuda") * std)
        parts.append(0.01 * torch.randn(co, generator=g, device="cuda"))
    return torch.cat(parts)


def _batch(case, seed):
    g = _generator(seed)
    x = _dirty(case["npix"], case["batch"], g)
    y = torch.clamp(x, min=0.0) + 0.1 * torch.rand(x.shape, generator=g, device="cuda",
                                                   dtype=torch.float64)
    return x.float()[:, None].contiguous(), y.float()[:, None].contiguous()


def _prepare_network(case, seed):
    ctx = _bare_context()
    n = case["npix"]
    flat = _parameters(case, seed).cpu().numpy()
    if case["kind"] == "predict":
        ws = WarmStart(ctx, levels=case["levels"], base=case["base"], batch=1, npix=n)
        ws.net.set_params(flat)
        dirty = _dirty(n, case["images"], _generator(seed)).float().cpu().numpy()
        return dict(case=case, ws=ws, dirty=dirty, ctx=ctx)
    net = UNet(ctx, levels=case["levels"], base=case["base"], batch=case["batch"], H=n, W=n,
               bf16=True)
    net.set_params(flat)
    x, y = _batch(case, seed)
    net.set_input(x.cpu().numpy())
    target = DeviceBuffer.from_array(y.cpu().numpy())
    return dict(case=case, net=net, target=target, y=_tensor(net.y, x.shape),
                grads=_tensor(net.grads, (net.nparams,)), weights=_tensor(net.params, (net.nparams,)),
                ctx=ctx)


class _Conv(torch.autograd.Function):
    """A K x K convolution with zero padding as a sum over taps of matrix products."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        b, ci, h, wd = x.shape
        co, _, k, _ = w.shape
        xp = torch.nn.functional.pad(x, [k // 2] * 4)
        out = x.new_zeros(b, co, h * wd)
        for dy in range(k):
            for dx in range(k):
                for n in range(b):
                    out[n].addmm_(w[:, :, dy, dx], xp[n, :, dy:dy + h, dx:dx + wd].reshape(ci, -1))
        return out.reshape(b, co, h, wd)

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        b, ci, h, wd = x.shape
        k = w.shape[2]
        xp = torch.nn.functional.pad(x, [k // 2] * 4)
        gx, gw = torch.zeros_like(xp), torch.zeros_like(w)
        for dy in range(k):
            for dx in range(k):
                wt = w[:, :, dy, dx].t().contiguous()
                for n in range(b):
                    gn = g[n].reshape(g.shape[1], -1)
                    gx[n, :, dy:dy + h, dx:dx + wd] += (wt @ gn).reshape(ci, h, wd)
                    gw[:, :, dy, dx] += gn @ xp[n, :, dy:dy + h, dx:dx + wd].reshape(ci, -1).t().contiguous()
        p = k // 2
        return gx[:, :, p:p + h, p:p + wd].contiguous(), gw


def _exact_forward(case, master, x):
    """Output of the network in FP64 with BF16-rounded weights; the leaves to differentiate."""
    leaves, off = {}, 0
    for name, co, ci, k in unet_shapes(case["levels"], case["base"]):
        w = master[off: off + co * ci * k * k].reshape(co, ci, k, k).bfloat16().double()
        off += w.numel()
        leaves[name] = (w.requires_grad_(), master[off: off + co].double().requires_grad_())
        off += co

    def conv(name, v, relu=True):
        w, b = leaves[name]
        v = _Conv.apply(v, w) + b[:, None, None]
        return torch.relu(v) if relu else v

    levels, skips, v = case["levels"], [], x
    for k in range(levels):
        v = conv(f"e{k}b", conv(f"e{k}a", v))
        if k < levels - 1:
            skips.append(v)
            v = 0.25 * (v[:, :, ::2, ::2] + v[:, :, ::2, 1::2] + v[:, :, 1::2, ::2] + v[:, :, 1::2, 1::2])
    for k in range(levels - 2, -1, -1):
        up = v.repeat_interleave(2, 2).repeat_interleave(2, 3)
        v = conv(f"d{k}b", conv(f"d{k}a", torch.cat([up, skips[k]], 1)))
    return conv("out", v, relu=False), leaves


def _exact_network(case, seed):
    master = _parameters(case, seed)
    if case["kind"] == "predict":
        dirty = _dirty(case["npix"], case["images"], _generator(seed)).float()
        scale = dirty.abs().amax(dim=(1, 2)).double()
        x = (dirty.cpu().numpy() / scale.float().cpu().numpy()[:, None, None]).astype(np.float32)
        x = torch.as_tensor(x, device="cuda").double()[:, None]
        with torch.no_grad():
            y, _ = _exact_forward(case, master, x)
        return dict(image=(y[:, 0] * scale[:, None, None]).cpu().numpy())
    x, target = _batch(case, seed)
    y, leaves = _exact_forward(case, master, x.double())
    loss = ((y - target.double()) ** 2).mean()
    loss.backward()
    grads = torch.cat([t.grad.reshape(-1) for pair in leaves.values() for t in pair])
    # the first Adam step: moments at zero
    weights = master.double() - 1e-4 * grads / (grads.abs() + 1e-8)
    return dict(loss=float(loss), output=y.detach(), gradients=grads, weights=weights)


# ---------------------------------------------------------------------------
# the objective in FP64
# ---------------------------------------------------------------------------
class _Exact:
    """chi2 and the priors, value and gradient, as the reference defines them."""

    def __init__(self, case, p, rows):
        self.case, self.p = case, p
        n = p.N
        self.mask = torch.as_tensor(p.noise, device="cuda") < p.noise_cut
        self.o = torch.arange(n, device="cuda", dtype=torch.float64) - n // 2
        cell = CELL / 3600.0 * RAD
        self.x, self.y = -self.o * cell, self.o * cell
        self.slices = []
        for f, uvw, vo, w in rows:
            r = uvw / _wavelength(f)
            flip = r[:, 0] > 0.0
            s = torch.where(flip, -1.0, 1.0)
            u, v, ww = r[:, 0] * s, r[:, 1] * s, r[:, 2]
            vis = torch.complex(vo[:, 0].double(), vo[:, 1].double() * s)
            ux, uy = u * (n * -cell), v * (n * cell)
            ux, uy = torch.where(ux < 0, ux + n, ux), torch.where(uy < 0, uy + n, uy)
            on = (ux >= 0) & (ux < n) & (uy >= 0) & (uy < n)
            pb = _beam(n, f).float().double()
            self.slices.append((float(np.float32(f) / np.float32(p.nu_0)), u, v, ww, vis,
                                torch.where(on, w.double(), 0.0), ux, uy, on, pb))

    def clip(self, img):
        off = torch.as_tensor(self.p.noise, device="cuda") > self.p.noise_cut
        img = img.clone()
        img[0][off] = float(np.float32(self.p.minpix))  # eta = -1: the floor
        img[1][off] = 0.0
        if self.case["flag"] > 0:
            img[1][~off & (img[0] < self.p.threshold)] = 0.0
        return img

    def chi2(self, img):
        p, n = self.p, self.p.N
        floor = float(np.float32(p.minpix))
        fg = float(np.float32(p.fg_scale))
        total, residuals = 0.0, []
        js = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)
        rot = torch.polar(torch.ones_like(js), -2.0 * math.pi * (n // 2) / n * js)
        for nudiv, u, v, w, vis, wt, ux, uy, on, pb in self.slices:
            inu = torch.clamp(img[0] * nudiv ** img[1], min=floor)
            grid = torch.fft.ifft2(inu * pb * fg) * (n * n) * rot[:, None] * rot[None]
            i1, j1 = ux.floor().long() % n, uy.floor().long() % n
            du, dv = ux - ux.floor(), uy - uy.floor()
            i2, j2 = (i1 + 1) % n, (j1 + 1) % n
            m = (1 - du) * (1 - dv) * grid[j1, i1] + (1 - du) * dv * grid[j2, i1] + \
                du * (1 - dv) * grid[j1, i2] + du * dv * grid[j2, i2]
            r = vis - torch.where(on, m, torch.zeros_like(m))
            total += float((wt * (r.real ** 2 + r.imag ** 2)).sum())
            residuals.append(r)
        return 0.5 * total, residuals

    def chi2_gradient(self, img, residuals):
        p, n = self.p, self.p.N
        fg = float(np.float32(p.fg_scale))
        out = torch.zeros(2, n, n, device="cuda", dtype=torch.float64)
        fx = -(self.x ** 2) / (1.0 + torch.sqrt(1.0 - self.x ** 2))
        k = self.case["flag"] % 2
        for (nudiv, u, v, w, vis, wt, ux, uy, on, pb), r in zip(self.slices, residuals):
            c = wt * r.conj()
            g = torch.zeros(n, n, device="cuda", dtype=torch.float64)
            step = max(2048, (1 << 27) // n // 8)
            for a in range(0, len(u), step):
                s = slice(a, a + step)
                ex = torch.outer(u[s], self.x) + torch.outer(w[s], fx)
                ey = torch.outer(v[s], self.y) + torch.outer(w[s], fx) + (c[s].angle() / (2 * math.pi))[:, None]
                ex, ey = (ex - ex.round()) * (2 * math.pi), (ey - ey.round()) * (2 * math.pi)
                amp = c[s].abs()[:, None]
                g.addmm_((amp * torch.cos(ey)).t().contiguous(), torch.cos(ex))
                g.addmm_((amp * torch.sin(ey)).t().contiguous(), torch.sin(ex), alpha=-1.0)
            d = -fg * pb * g
            di = nudiv ** img[1]
            if k == 0:
                out[0] += torch.where(self.mask, d * di, 0.0)
            else:
                chain = d * img[0] * di * fg * math.log(nudiv) if nudiv != 1.0 else torch.zeros_like(d)
                out[1] += torch.where(self.mask & (img[0] > p.threshold), chain, 0.0)
        return out

    def prior(self, kind, im):
        """(value, gradient) of one prior on one image, without its factor."""
        n, eta, prior = self.p.N, -1.0, float(np.float32(0.001))
        c = im
        z = torch.zeros_like(c)
        if kind == "entropy":
            val = c * torch.log(c / prior + (eta + 1.0))
            grad = torch.log(c / prior + (eta + 1.0)) + 1.0
        elif kind == "tsv":
            val = c.clone()
            val[:-1, :-1] = (c[:-1, :-1] - c[:-1, 1:]) ** 2 + (c[:-1, :-1] - c[1:, :-1]) ** 2
            grad = c.clone()
            grad[1:-1, 1:-1] = 8.0 * c[1:-1, 1:-1] - 2.0 * (
                c[:-2, 1:-1] + c[1:-1, :-2] + c[2:, 1:-1] + c[1:-1, 2:])
        else:
            val = c.clone()
            lap = c[1:-1, :-2] + c[1:-1, 2:] + c[:-2, 1:-1] + c[2:, 1:-1] - 4.0 * c[1:-1, 1:-1]
            val[1:-1, 1:-1] = 0.5 * lap ** 2
            grad = z
            m = c[2:-2, 2:-2]
            d, up, r, le = c[3:-1, 2:-2], c[1:-3, 2:-2], c[2:-2, 3:-1], c[2:-2, 1:-3]
            corners = c[3:-1, 1:-3] + c[3:-1, 3:-1] + c[1:-3, 1:-3] + c[1:-3, 3:-1]
            far = c[4:, 2:-2] + c[2:-2, 4:] + c[:-4, 2:-2] + c[2:-2, :-4]
            grad = z.clone()
            # the reference's sign pattern: -8 (d - r - u - l)
            grad[2:-2, 2:-2] = 20.0 * m - 8.0 * (d - r - up - le) + 2.0 * corners + far
        return float(val[self.mask].sum()), torch.where(self.mask, grad, z)

    def value(self, img, iteration):
        """(objective, clipped image, residuals)."""
        img = self.clip(img)
        total, residuals = self.chi2(img)
        if iteration > 0:
            for kind in self.case["priors"].split():
                lam = float(np.float32(LAMBDAS[PRIORS[kind][1]]))
                total += lam * self.prior(kind, img[0])[0]
        return total, img, residuals

    def gradient(self, img, residuals, iteration):
        out = self.chi2_gradient(img, residuals)
        if iteration > 0 and self.case["flag"] % 2 == 0:
            for kind in self.case["priors"].split():
                out[0] += float(np.float32(LAMBDAS[PRIORS[kind][1]])) * self.prior(kind, img[0])[1]
        return out


def exact(case, seed):
    if case["kind"] in ("train", "predict"):
        return _exact_network(case, seed)
    if case["kind"] == "grid":
        return _exact_grid(case, seed)
    rows, sky = _rows(case, seed)
    p, sky_image = _problem(case, rows, sky)
    e = _Exact(case, p, rows)
    img = _start_image(case, p, sky_image, seed).double()
    if case["kind"] == "optimise":
        return _exact_optimise(case, p, rows, e, img)
    value, clipped, residuals = e.value(img, 1)
    if case["kind"] == "evaluate":
        return dict(value=value, gradient=e.gradient(clipped, residuals, 1), image=clipped)
    trial = clipped + 0.25 * _direction(p, sky_image, img.float()).double()
    trial[0] = torch.clamp(trial[0], min=float(np.float32(p.minpix)))
    value, trial, _ = e.value(trial, 1)
    return dict(value=value, image=trial)


def _exact_optimise(case, p, rows, e, img):
    """CG-FRPRMN with given step lengths (src/frprmn.cu:85-195 of the reference)."""
    floor = float(np.float32(p.minpix))

    def trial(p0, d, x):
        t = p0 + x * d
        t[0] = torch.clamp(t[0], min=floor)
        return t

    cur, path, it = img, [], 0
    _, cur, res = e.value(cur, it)
    xi = -e.gradient(cur, res, 0)
    g, h = xi.clone(), xi.clone()
    for k, x in enumerate(_steps(case, p, rows)):
        path.append(e.value(trial(cur, xi, x), it)[0])
        moved = trial(cur, xi, x)
        _, cur, res = e.value(moved, it)
        it = k + 1
        xi = e.gradient(cur, res, it)
        gg, dgg = float((g * g).sum()), float(((xi + g) * xi).sum())
        g = -xi
        h = g + max(0.0, dgg / gg) * h
        xi = h.clone()
    value, cur, _ = e.value(cur, it)
    return dict(value=value, path=path, image=cur)


def work(case):
    """Each input read once and each output written once; the operations of the
    transforms and interpolations (fast transforms: a direct sum over pixels and
    visibilities is not counted), or of the network's convolutions."""
    n = case["npix"]
    if case["kind"] in ("train", "predict"):
        images = case.get("batch", 0) or case["images"]
        flops = params = 0
        for name, co, ci, k in unet_shapes(case["levels"], case["base"]):
            level = 0 if name == "out" else int(name[1])
            flops += 2.0 * co * ci * k * k * images * (n >> level) ** 2
            params += co * ci * k * k + co
        if case["kind"] == "predict":
            return dict(bytes=8.0 * images * n * n + 2.0 * params, flops=flops)
        return dict(bytes=12.0 * images * n * n + 28.0 * params, flops=3.0 * flops)
    rows = case["antennas"] * (case["antennas"] - 1) // 2 * case["dumps"]
    rows *= case["channels"] * (1.0 - 0.5 * case["flagged"])
    if case["kind"] == "grid":
        return dict(bytes=36.0 * rows + 36.0 * n * n, flops=2.0 * rows * case["taps"] ** 2 * 8.0)
    transform = 5.0 * n * n * math.log2(n * n) * case["channels"]
    value = dict(bytes=24.0 * rows + (12.0 + 4.0 * case["channels"]) * n * n,
                 flops=transform + 40.0 * rows)
    if case["kind"] == "probe":
        return dict(bytes=value["bytes"] + 24.0 * n * n, flops=value["flops"])
    both = dict(bytes=value["bytes"] + 20.0 * rows + 16.0 * n * n,
                flops=2.0 * value["flops"])
    if case["kind"] == "optimise":
        k = case["iterations"]
        return dict(bytes=(k + 1) * (value["bytes"] + both["bytes"]),
                    flops=(k + 1) * (value["flops"] + both["flops"]))
    return both
