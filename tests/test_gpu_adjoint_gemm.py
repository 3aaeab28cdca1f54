"""The GEMM forms of the adjoint, which gridding stands in for wherever it applies:
every operand form, several slices and range lengths, a partial mask and the
full-size workload, with the form that ran asserted.  Against the FP64 oracle where
its sums are short, else against the gridded form, which its own tests hold to
1.5e-6 of the oracle.

Tolerance: 1e-5 relative L2, the gradient's bar; 1.15e-5 against the gridded form."""
import numpy as np
import pytest
import torch

import oracle
from gpuvmem_amd import native
from gpuvmem_amd.device import Context
from gpuvmem_amd.problem import make_problem, small_problem

pytestmark = pytest.mark.gpu

TOL = 1e-5
FORMS = ["bf16x3", "f16x3", "f32"]


def _gradient(ctx, d, flag=0, normalize=False):
    r = ctx.zeros(2 * ctx.n)
    ctx.dchi2(d, r, flag_opt=flag, normalize=normalize)
    ctx.sync()
    p = ctx.problem
    return r.download(np.float32, (2, p.N, p.M))


def _rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


def _image(p, seed):
    rng = np.random.default_rng(seed)
    img = p.initial_image()
    img[0] += (rng.random((p.N, p.M)) * 20.0).astype(np.float32)
    img[1] = rng.uniform(-1.0, 2.0, (p.N, p.M)).astype(np.float32)
    return img


def _slices(p, counts, seed=0):
    """Rows over the half plane, w up to half a turn at the image's corners."""
    rng = np.random.default_rng(seed)
    dx = abs(p.deltax) * np.pi / 180.0
    x = p.N / 2 * dx
    wmax = 0.5 / (2 * x * x / (1 + np.sqrt(1 - 2 * x * x)))
    out = []
    for k, n in enumerate(counts):
        c = np.stack([rng.uniform(0, 0.45 * p.N, n), rng.uniform(-0.45 * p.N, 0.45 * p.N, n)], 1)
        uvw = np.concatenate([c / (p.N * dx) * [np.sign(p.deltax), 1.0],
                              rng.uniform(-wmax, wmax, (n, 1))], 1)
        vo = (rng.standard_normal((n, 2)) * 2.0).astype(np.float32)
        out.append((float(np.float32(p.freq * (1 + 0.02 * k))), uvw, vo,
                    rng.uniform(0.5, 2.0, n).astype(np.float32)))
    return out


@pytest.mark.parametrize("mode", FORMS)
@pytest.mark.parametrize("flag,normalize", [(0, False), (1, True)])
def test_slices_and_range_lengths(mode, flag, normalize):
    p = small_problem(npix=128, n_antennas=8, seed=5)
    y, x = np.mgrid[:p.N, :p.M]
    on = (x - 40) ** 2 + (y - 70) ** 2 < 45 ** 2  # whole sub-tiles off the mask
    p.noise = np.where(on, 0.5, 2.0).astype(np.float32) * np.float32(p.noise_cut)
    slices = _slices(p, (1, 4000, 700, 20000))
    img = _image(p, 1)
    orc = oracle.Oracle(p, slices=slices)
    _, vr, clipped = orc.chi2(img, flag_opt=flag, normalize=normalize)
    ref = orc.dchi2(clipped, vr, flag_opt=flag, normalize=normalize)[flag]
    ctx = Context(p, adjoint=mode, add_data=False)
    ctx.set_gridding("never")
    for s in slices:
        ctx.add(*s)
    d = ctx.image(img)
    ctx.chi2(d, flag_opt=flag, normalize=normalize)
    for length in (256, 1536, 6144, 16384):
        ctx.set_split_vis(length)
        g = _gradient(ctx, d, flag, normalize)
        assert not ctx.adjoint_gridded()
        err = _rel(g[flag], ref)
        print(f"{mode} ranges of {length}: rel L2 {err:.2e}", flush=True)
        assert err < TOL
        assert np.all(g[1 - flag] == 0) and np.all(g[:, ~on] == 0)
    ctx.close()


@pytest.fixture(scope="module")
def full():
    p = make_problem(1)
    img = p.initial_image()
    img[0] = np.maximum(p.sky / p.fg_scale * 0.5, p.minpix).astype(np.float32)
    ctx = Context(p)
    d = ctx.image(img)
    ctx.chi2(d)
    g = _gradient(ctx, d)[0]
    assert ctx.adjoint_gridded()
    ctx.close()
    return p, img, g


@pytest.mark.parametrize("mode", FORMS)
def test_full_size(full, mode):
    """The whole 1024^2 image, 1,764,000 rows: no pixel of a skipped sub-tile is
    lost, at the shortest and the default range length."""
    p, img, ref = full
    on = p.noise < p.noise_cut
    ctx = Context(p, adjoint=mode)
    ctx.set_gridding("never")
    d = ctx.image(img)
    ctx.chi2(d)
    assert ctx.adjoint_computed_pixels() < p.M * p.N
    for length in (1536, 6144):
        ctx.set_split_vis(length)
        g = _gradient(ctx, d)[0]
        assert not ctx.adjoint_gridded()
        err = _rel(g[on], ref[on])
        print(f"{mode} ranges of {length}: rel L2 {err:.2e} from the gridded form", flush=True)
        assert err < 1.15e-5 and np.all(g[~on] == 0)
    ctx.close()


def test_the_choice():
    """never / auto / always, back and forth; DIRECT is never gridded."""
    p = small_problem(npix=64, n_antennas=8, seed=5)
    ctx = Context(p)
    d = ctx.image(_image(p, 2))
    ctx.chi2(d)
    ran = {}
    for when, form in (("auto", "bf16x3"), ("never", "bf16x3"), ("always", "f32"), ("never", "f32"),
                       ("always", "direct"), ("auto", "f16x3")):
        ctx.set_gridding(when)
        ctx.set_adjoint(form)
        ran[when, form] = _gradient(ctx, d)[0]
        assert ctx.adjoint_gridded() == (when != "never" and form != "direct")
    assert np.array_equal(ran["auto", "bf16x3"], ran["always", "f32"])
    assert not np.array_equal(ran["auto", "bf16x3"], ran["never", "bf16x3"])
    for g in ran.values():
        assert _rel(g, ran["always", "direct"].astype(np.float64)) < TOL
    with pytest.raises(native.GvmError):
        native.check(ctx.lib.gvm_set_gridding(ctx.ctx, 3), "gvm_set_gridding")
    ctx.close()


def test_the_autotuner_times_the_gemm(tmp_path, monkeypatch):
    """While the gradients run by gridding, range lengths are still the GEMM's: its
    times are what is compared and kept, and the gradient is what it was before."""
    monkeypatch.setenv("GVM_TUNE_CACHE", str(tmp_path / "tune.txt"))
    p = small_problem(npix=512, n_antennas=8, seed=77)
    p.noise = np.full_like(p.noise, 0.5 * p.noise_cut)
    ctx = Context(p, add_data=False)
    for s in _slices(p, (150000, 49983), seed=3):
        ctx.add(*s)
    d = ctx.image(_image(p, 4))
    ctx.chi2(d)
    before = _gradient(ctx, d)
    ctx.reset_timing()
    for _ in range(5):
        _gradient(ctx, d)
    gridded_ms = ctx.adjoint_time_ms()[0]
    r = ctx.autotune([512, 1536, 6144])
    print(f"gridded {gridded_ms:.3f} ms, GEMM by range length {r}", flush=True)
    # 2e11 products of three 16-bit MFMA products: 0.5 ms at the matrix units' peak
    assert not r["cached"] and min(r["ms"].values()) > 0.5 > gridded_ms
    assert np.array_equal(_gradient(ctx, d), before) and ctx.adjoint_gridded()
    ctx.close()


@pytest.mark.parametrize("npix,nsl,rows,turns,gridded", [
    (256, 64, 10, 0.3, False),   # many slices of few rows, 12 planes
    (64, 1, 10, 2.0, False),     # few rows, 30 planes
    (64, 1, 6000, 2.0, True),
    (256, 2, 10, 0.02, True),
    (256, 64, 10, 0.0, True),    # one plane
    (1024, 1, 30, 0.3, False),   # below the line of few rows: the faster form
    (1024, 1, 1000, 0.0, True),
])
def test_few_rows_on_many_transforms(npix, nsl, rows, turns, gridded):
    """The form is chosen by slices and planes as well as by rows."""
    print(f"case: {npix}^2 {nsl} slices of {rows} rows, {turns} turns", flush=True)
    p = small_problem(npix=npix, n_antennas=6, seed=4)
    p.noise = np.full_like(p.noise, 0.5 * p.noise_cut)
    slices = [(f, uvw * [1.0, 1.0, 2.0 * turns], vo, w)
              for f, uvw, vo, w in _slices(p, (rows,) * nsl, seed=npix)]
    ctx = Context(p, add_data=False)
    for s in slices:
        ctx.add(*s)
    d = ctx.image(_image(p, 5))
    ctx.chi2(d)
    g = _gradient(ctx, d)[0]
    assert ctx.adjoint_gridded() == gridded
    other = {True: "never", False: "always"}[gridded]
    ctx.set_gridding(other)
    assert _rel(g, _gradient(ctx, d)[0].astype(np.float64)) < TOL
    assert ctx.adjoint_gridded() != gridded
    ctx.close()


def test_the_form_that_does_not_run_keeps_little_memory():
    """4096^2 with 60,000 rows: a plan of 1.9 GiB (8 planes) and a GEMM workspace of 1.5;
    going from one to the other gives back what is over 1 GiB."""
    p = small_problem(npix=4096, n_antennas=4, seed=6, dump_seconds=3600.0)
    p.noise = np.full_like(p.noise, 0.5 * p.noise_cut)
    slices = [(f, uvw * [1.0, 1.0, 0.2], vo, w) for f, uvw, vo, w in _slices(p, (60000,))]
    ctx = Context(p, add_data=False)
    ctx.add(*slices[0])
    d = ctx.image(p.initial_image())
    ctx.chi2(d)
    r = ctx.zeros(2 * ctx.n)
    ctx.sync()
    base, used = torch.cuda.mem_get_info()[0], {}
    for k, when in enumerate(("always", "never", "always", "never")):
        ctx.set_gridding(when)
        ctx.dchi2(d, r)
        ctx.sync()
        assert ctx.adjoint_gridded() == (when == "always")
        used[k] = (base - torch.cuda.mem_get_info()[0]) / 2 ** 30
    print(f"GiB in use: {used}", flush=True)
    assert 1.5 < used[0] < 2.25 and 1.25 < used[1] < 1.75
    assert abs(used[2] - used[0]) < 0.25 and abs(used[3] - used[1]) < 0.25
    ctx.close()
