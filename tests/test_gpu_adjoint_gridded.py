"""The gridded form of the adjoint where it can go wrong, against the FP64
oracle's direct sums (the reference's formula, exact w term) on sampled
pixels: every image size, rows beyond the Nyquist column (the half grid
folds them) and beyond +-N/2 in v (the grid wraps), rows on the fold and on
tile edges, a phase centre off the image centre, many rows in one tile
(several work items merged), w terms of one plane, of several plane groups
and too many planes for it (the GEMM takes the call), slices of very
different length, and rows that are not numbers.

Tolerance: the FP32 transform of (2N)^2 points rounds about 2 log2(2N) <= 26
times per value at 6e-8 each, at random, times 3 for the kernel correction off
the centre (its rms over the image: it grows to 3.1 along each axis, 9.5 at a corner,
and the corners have a test of their own): 3 sqrt(26) 6e-8 = 9e-7, plus 1e-7 each for
the kernel's evaluation, the spreading sums and the final float: 1.5e-6.  The
GEMM's cases keep the 1e-5 that its own tests use."""
import numpy as np
import pytest

import oracle
from gpuvmem_amd import native
from gpuvmem_amd.device import Context, DeviceBuffer
from gpuvmem_amd.problem import small_problem

pytestmark = pytest.mark.gpu

TOL = 1.5e-6


def _direct_sums(p, sl, vr, pix):
    """-fg PB sum_v w (Re Vr cos phi + Im Vr sin phi) at pixels of one slice, FP64,
    with z - 1 formed without cancellation: at these angles (1e-5 rad) sqrt(1 -
    r^2) - 1 itself is off by 3e-6 of its value, 2e-6 per turn of w phase."""
    f, uvw, vo, w = sl
    x = (pix[:, 1] - int(p.x0)) * p.deltax * np.pi / 180.0
    y = (pix[:, 0] - int(p.y0)) * p.deltay * np.pi / 180.0
    r2 = x * x + y * y
    t = np.outer(x, uvw[:, 0]) + np.outer(y, uvw[:, 1]) + \
        np.outer(-r2 / (1.0 + np.sqrt(1.0 - r2)), uvw[:, 2])
    ph = 2.0 * np.pi * (t - np.rint(t))
    pb = oracle.Oracle(p, slices=[sl]).pb(f)
    s = (np.cos(ph) * vr.real + np.sin(ph) * vr.imag) @ w.astype(np.float64)
    return -float(np.float32(p.fg_scale)) * np.array([pb[i, j] for i, j in pix]) * s


def _check(p, slices, mode="bf16x3", flag=0, seed=0, pixels=160, tol=TOL, repeat=False,
           direct=False):
    rng = np.random.default_rng(seed)
    img = p.initial_image()
    img[0] += (rng.random((p.N, p.M)) * 20.0).astype(np.float32)
    if len(slices) > 1:
        img[1] = rng.uniform(-1.0, 2.0, (p.N, p.M)).astype(np.float32)
    ctx = Context(p, adjoint=mode, add_data=False)
    for f, u, v, w in slices:
        ctx.add(f, u, v, w)
    d = ctx.image(img)
    ctx.chi2(d, flag_opt=flag)
    out = []
    for _ in range(2 if repeat else 1):
        r = ctx.zeros(2 * p.M * p.N)
        ctx.dchi2(d, r, flag_opt=flag)
        ctx.sync()
        out.append(r.download(np.float32, (2, p.N, p.M)))
    ctx.close()
    if repeat:
        assert np.array_equal(out[0], out[1])
    orc = oracle.Oracle(p, slices=slices)
    _, vr, clipped = orc.chi2(img, flag_opt=flag)
    inside = np.argwhere(p.noise < p.noise_cut)
    pix = inside[rng.choice(len(inside), min(pixels, len(inside)), replace=False)]
    if direct:
        ref = _direct_sums(p, slices[0], np.asarray(vr).reshape(-1), pix)
    else:
        ref = np.asarray(orc.dchi2_pixels_all(clipped, vr, pix, flag_opt=flag))[:, flag % 2]
    got = np.array([out[0][flag % 2, i, j] for i, j in pix], np.float64)
    err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"{p.M}^2 {[s[1].shape[0] for s in slices]} {mode} flag {flag}: rel L2 {err:.2e}",
          flush=True)
    assert err < tol
    assert np.all(out[0][:, p.noise >= p.noise_cut] == 0)
    return err


def _rows(p, cells, w=None, seed=1):
    """A slice with rows at grid positions (ux, uy) in cells of the N x N grid."""
    rng = np.random.default_rng(seed)
    cells = np.asarray(cells, np.float64)
    dx, dy = p.deltax * np.pi / 180.0, p.deltay * np.pi / 180.0
    uvw = np.zeros((len(cells), 3))
    uvw[:, 0], uvw[:, 1] = cells[:, 0] / (p.M * dx), cells[:, 1] / (p.N * dy)
    if w is not None:
        uvw[:, 2] = w
    vo = (rng.standard_normal((len(cells), 2)) * 2.0).astype(np.float32)
    return (p.freq, uvw, vo, rng.uniform(0.5, 2.0, len(cells)).astype(np.float32))


def _open_mask(p):
    """Every pixel on the mask."""
    p.noise = np.full_like(p.noise, p.fg_scale)
    return p


@pytest.mark.parametrize("npix", [64, 128, 256, 512, 1024, 2048])
def test_sizes_and_the_whole_plane(npix):
    """Rows over the whole grid: ux in [0, N) (beyond N/2 the half grid
    folds), uy in (-N, N), among them the fold, the ends and tile edges."""
    p = _open_mask(small_problem(npix=npix, n_antennas=5, seed=npix))
    rng = np.random.default_rng(npix)
    n = npix
    cells = np.stack([rng.uniform(0, n, 3000), rng.uniform(-n + 1, n - 1, 3000)], 1)
    edge = [0.0, 0.25, 1.75, 2.0, 3.75, 4.0, n / 2 - 2.25, n / 2 - 0.25, n / 2 - 0.01, n / 2,
            n / 2 + 0.25, n / 2 + 2.25, n - 2.0, n - 0.25, n - 1e-4]
    cells = np.concatenate([cells, [(a, b) for a in edge for b in
                                    [0.0, -0.25, 1.75, -2.0, n / 2, n / 2 - 0.25, -n / 2, n - 1.5]]])
    _check(p, [_rows(p, cells, w=rng.uniform(-1e5, 1e5, len(cells)))], seed=npix, repeat=True,
           pixels=160 if npix < 2048 else 60)


@pytest.mark.parametrize("mode", ["bf16x3", "f16x3", "f32"])
@pytest.mark.parametrize("x0,y0", [(0.0, 63.0), (40.6, 20.0)])
def test_phase_centre_off_the_image_centre(mode, x0, y0):
    p = _open_mask(small_problem(npix=64, n_antennas=6, seed=3))
    p.x0, p.y0 = x0, y0
    rng = np.random.default_rng(5)
    cells = np.stack([rng.uniform(0, 40, 2500), rng.uniform(-31, 31, 2500)], 1)
    _check(p, [_rows(p, cells, w=rng.uniform(-1e6, 1e6, 2500))], mode=mode)


@pytest.mark.parametrize("rows", [1, 3, 63, 64, 65, 511, 513, 40000])
def test_rows_of_one_tile(rows):
    p = _open_mask(small_problem(npix=128, n_antennas=4, seed=8))
    rng = np.random.default_rng(rows)
    cells = np.stack([rng.uniform(20.0, 23.9, rows), rng.uniform(-12.0, -8.1, rows)], 1)
    _check(p, [_rows(p, cells)], seed=rows, repeat=True)


@pytest.mark.parametrize("turns", [0.0, 1e-6, 0.02, 0.3, 1.2, 2.0, 2.6])
def test_w_terms(turns):
    """w up to `turns` of phase at the farthest pixel: 1 to 32 planes; 2.6
    turns need more, and the GEMM takes the call."""
    p = _open_mask(small_problem(npix=64, n_antennas=6, seed=4))
    rng = np.random.default_rng(6)
    x = 32 * abs(p.deltax) * np.pi / 180.0
    f = 2 * x * x / (1 + np.sqrt(1 - 2 * x * x))
    cells = np.stack([rng.uniform(0, 60, 6000), rng.uniform(-31, 31, 6000)], 1)
    _check(p, [_rows(p, cells, w=rng.uniform(-1, 1, 6000) * turns / f)],
           tol=TOL if turns < 2.5 else 1e-5, direct=True)


@pytest.mark.parametrize("flag", [0, 1])
def test_slices_of_different_length(flag):
    p = small_problem(npix=64, n_antennas=6, seed=4)
    rng = np.random.default_rng(7)
    slices = []
    for k, n in enumerate((1, 700, 20000, 64)):
        cells = np.stack([rng.uniform(0, 31, n), rng.uniform(-31, 31, n)], 1)
        f, u, v, w = _rows(p, cells, w=rng.uniform(-1e4, 1e4, n), seed=k)
        slices.append((float(np.float32(f * (1 + 0.02 * k))), u, v, w))
    _check(p, slices, flag=flag)


@pytest.mark.parametrize("bad", ["visibility", "w"])
def test_rows_that_are_not_numbers(bad):
    """A NaN visibility, or an infinite w (the GEMM takes that call), reaches
    every pixel on the mask, as in the sums, and none off it."""
    p = small_problem(npix=64, n_antennas=6, seed=4)
    rng = np.random.default_rng(9)
    cells = np.stack([rng.uniform(0, 31, 4000), rng.uniform(-31, 31, 4000)], 1)
    f, u, v, w = _rows(p, cells)
    if bad == "w":
        u[5, 2] = np.inf
    else:
        v[17, 0] = np.nan
    on = p.noise < p.noise_cut
    ctx = Context(p, add_data=False)
    ctx.add(f, u, v, w)
    d = ctx.image(p.initial_image())
    ctx.chi2(d)
    r = ctx.zeros(2 * p.M * p.N)
    ctx.dchi2(d, r)
    ctx.sync()
    g = r.download(np.float32, (2, p.N, p.M))[0]
    ctx.close()
    assert on.any() and np.all(np.isnan(g[on])) and np.all(g[~on] == 0)


@pytest.mark.parametrize("mode", ["bf16x3", "direct"])
@pytest.mark.parametrize("flag,nsl", [(0, 1), (1, 1), (0, 3), (1, 3), (0, 0)])
def test_a_result_that_is_set(mode, flag, nsl):
    """gvm_dchi2_set into any memory gives what gvm_dchi2 adds to a cleared one."""
    print(f"case: set {mode} flag {flag} slices {nsl}", flush=True)
    p = small_problem(npix=64, n_antennas=6, seed=31)
    rng = np.random.default_rng(nsl)
    img = p.initial_image()
    img[0] += (rng.random((p.N, p.M)) * 20.0).astype(np.float32)
    img[1] = rng.uniform(-1.0, 2.0, (p.N, p.M)).astype(np.float32)
    ctx = Context(p, adjoint=mode, add_data=False)
    for s in range(nsl):
        cells = np.stack([rng.uniform(0, 40, 400), rng.uniform(-31, 31, 400)], 1)
        ctx.add(p.freq * (1.0 + 0.1 * s), *_rows(p, cells, w=rng.uniform(-1e4, 1e4, 400))[1:])
    d = ctx.image(img)
    if nsl == 0:  # (a context may refuse to evaluate nothing: then there is no gradient either)
        try:
            ctx.chi2(d, flag_opt=flag)
        except native.GvmError:
            ctx.close()
            return
    else:
        ctx.chi2(d, flag_opt=flag)
    out = []
    for fn, fill in ((ctx.lib.gvm_dchi2, 0.0), (ctx.lib.gvm_dchi2_set, np.nan)):
        r = DeviceBuffer.from_array(np.full(2 * p.M * p.N, fill, np.float32))
        native.check(fn(ctx.ctx, d.ptr, r.ptr, flag, 1), "dchi2")
        ctx.sync()
        out.append(r.download(np.float32))
    ctx.close()
    assert np.array_equal(out[0], out[1])


def test_the_largest_image():
    """4096^2 has blocks of its own: two columns (8,192-point transforms), rows of
    1,024 threads."""
    n = 4096
    p = _open_mask(small_problem(npix=n, n_antennas=4, seed=7, dump_seconds=600.0))
    rng = np.random.default_rng(n)
    cells = np.stack([rng.uniform(0, n, 3000), rng.uniform(-n + 1, n - 1, 3000)], 1)
    edge = [0.0, 3.75, n / 2 - 0.25, n / 2, n / 2 + 2.25, n - 1e-4]
    cells = np.concatenate([cells, [(a, b) for a in edge for b in [0.0, -2.0, n / 2, n - 1.5]]])
    s = _rows(p, cells, w=rng.uniform(-1e5, 1e5, len(cells)))
    _check(p, [s], seed=n, repeat=True, pixels=60)
    ctx = Context(p, add_data=False)
    ctx.add(*s)
    d = ctx.image(p.initial_image())
    ctx.chi2(d)
    r = ctx.zeros(2 * n * n)
    ctx.dchi2(d, r)
    ctx.sync()
    assert ctx.adjoint_gridded()
    ctx.close()


@pytest.mark.parametrize("npix,turns", [(64, 0.0), (256, 0.3), (1024, 0.02), (2048, 0.02)])
def test_corner_pixels(npix, turns):
    """The corners by themselves: the kernel's transform falls to 1 / 3.1 at an
    edge and 1 / 9.5 at a corner, and rounding is multiplied by as much there.  sqrt(26)
    6e-8 of the transforms times 9.5, plus 1e-7 each for the spreading sums, the final
    float and the kernel's evaluation times its share at a corner: 2.9e-6 + 0.3e-6."""
    p = _open_mask(small_problem(npix=npix, n_antennas=5, seed=npix))
    p.antenna_diameter, p.pb_cutoff = 1.0, 1.0  # a beam that reaches the corners
    rng = np.random.default_rng(npix + 1)
    n, m = npix, 4000
    x = n / 2 * abs(p.deltax) * np.pi / 180.0
    f = 2 * x * x / (1 + np.sqrt(1 - 2 * x * x))
    cells = np.stack([rng.uniform(0, 0.48 * n, m), rng.uniform(-0.48 * n, 0.48 * n, m)], 1)
    s = _rows(p, cells, w=rng.uniform(-1, 1, m) * turns / f)
    ctx = Context(p, add_data=False)
    ctx.add(*s)
    d = ctx.image(p.initial_image())
    ctx.chi2(d)
    vr = ctx.residuals(0, m).astype(np.float64)
    e = np.r_[0:6, n - 6:n]
    pix = np.array([(i, j) for i in e for j in e])
    ref = _direct_sums(p, s, vr[:, 0] + 1j * vr[:, 1], pix)
    got = {}
    for when, form in (("always", "f32"), ("never", "f32"), ("never", "bf16x3")):
        ctx.set_gridding(when)
        ctx.set_adjoint(form)
        r = ctx.zeros(2 * n * n)
        ctx.dchi2(d, r)
        ctx.sync()
        g = r.download(np.float32, (2, n, n))[0]
        got[when, form] = np.linalg.norm(g[pix[:, 0], pix[:, 1]] - ref) / np.linalg.norm(ref)
    print(f"{n}^2 {turns} turns, corners: {got}", flush=True)
    assert got["always", "f32"] < 3.2e-6
    ctx.close()


@pytest.mark.parametrize("flag", [0, 1])
def test_a_result_that_is_set_over_several_batches(flag):
    """Eleven slices at 1024^2 with 6 planes (51 MB of transforms each): ten share the
    workspace, the last has it for itself and writes the result straight."""
    p = small_problem(npix=1024, n_antennas=5, seed=12)
    rng = np.random.default_rng(flag)
    x = 512 * abs(p.deltax) * np.pi / 180.0
    f = 2 * x * x / (1 + np.sqrt(1 - 2 * x * x))
    img = p.initial_image()
    img[0] += (rng.random((p.N, p.M)) * 20.0).astype(np.float32)
    img[1] = rng.uniform(-1.0, 2.0, (p.N, p.M)).astype(np.float32)
    ctx = Context(p, add_data=False)
    ctx.set_gridding("always")
    for k in range(11):
        cells = np.stack([rng.uniform(0, 400, 100), rng.uniform(-400, 400, 100)], 1)
        ctx.add(p.freq * (1.0 + 0.02 * k),
                *_rows(p, cells, w=rng.uniform(-1, 1, 100) * 0.02 / f, seed=k)[1:])
    d = ctx.image(img)
    ctx.chi2(d, flag_opt=flag)
    out = []
    for fn, fill, when in ((ctx.lib.gvm_dchi2, 0.0, "always"), (ctx.lib.gvm_dchi2_set, np.nan, "always"),
                           (ctx.lib.gvm_dchi2_set, np.nan, "never")):
        ctx.set_gridding(when)
        r = DeviceBuffer.from_array(np.full(2 * p.M * p.N, fill, np.float32))
        native.check(fn(ctx.ctx, d.ptr, r.ptr, flag, 1), "dchi2")
        ctx.sync()
        assert ctx.adjoint_gridded() == (when == "always")
        out.append(r.download(np.float32))
    ctx.close()
    assert np.array_equal(out[0], out[1])
    assert np.linalg.norm(out[0] - out[2]) < 1.15e-5 * np.linalg.norm(out[2])
