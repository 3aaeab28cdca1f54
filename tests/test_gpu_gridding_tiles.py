"""The tiled gridder and the weighting sums where they can go wrong, bit for bit
against the oracle's single-thread float sums: kernels that span one to many
tiles and more taps than LDS holds, supports off the kernel's middle, rows beyond
every edge, one crowded cell, a single row, and runs around the lengths at
which a wave takes over from a thread.  Whole results, so no tolerance."""
import numpy as np
import pytest

import oracle
from gpuvmem_amd.device import Context, DeviceBuffer
from gpuvmem_amd.gridding import GriddingKernel, apply_weighting_dev, grid_visibilities_dev
from gpuvmem_amd.problem import small_problem

pytestmark = pytest.mark.gpu


def _rows(p, n, seed, centre=None):
    """Rows over a plane a little larger than the grid, or all in one cell."""
    rng = np.random.default_rng(seed)
    lam = float(np.float32(2.99792458e8) / np.float32(p.freq))
    du = lam / (p.M * abs(p.deltax) * np.pi / 180.0)
    span = 0.62 * p.M
    cells = rng.uniform(-span, span, (n, 2)) if centre is None else \
        np.asarray(centre) + rng.uniform(-0.45, 0.45, (n, 2))
    uvw = np.concatenate([cells * du, np.zeros((n, 1))], 1)
    vo = rng.standard_normal((n, 2)).astype(np.float32)
    w = rng.uniform(0.1, 3.0, n).astype(np.float32)
    w[rng.random(n) < 0.05] = 0.0
    return uvw, vo, w


def _grid_both(p, k, uvw, vo, w):
    ctx = Context(p, add_data=False)
    bufs = [DeviceBuffer.from_array(a) for a in (uvw, vo, w)]
    out = [grid_visibilities_dev(ctx, k, p.freq, *bufs, uvw.shape[0]) for _ in range(2)]
    ctx.close()
    ref = oracle.grid_visibilities(p.M, p.N, p.deltax, p.deltay, p.freq, uvw, vo, w, k.taps,
                                   k.support_x, k.support_y)
    for got in out:  # the second call runs in the first one's workspace
        for a, b in zip(got, ref):
            assert a.shape == b.shape and np.array_equal(a, b)
    return ref[0].shape[0]


@pytest.mark.parametrize("m,n", [(1, 1), (2, 2), (7, 9), (9, 10), (11, 17), (31, 33), (33, 35)])
def test_kernel_sizes(m, n):
    p = small_problem(npix=64, n_antennas=5, seed=2)
    k = GriddingKernel.from_taps(np.random.default_rng(m * n).uniform(0.1, 1.0, (m, n))
                                 .astype(np.float32))
    print(f"case: gridder {m} x {n} taps", flush=True)
    assert _grid_both(p, k, *_rows(p, 900, m + n)) > 0


def test_supports_off_the_middle():
    p = small_problem(npix=64, n_antennas=5, seed=2)
    k = GriddingKernel.from_taps(np.random.default_rng(1).uniform(0.1, 1.0, (5, 6))
                                 .astype(np.float32))
    for sx, sy in ((0, 0), (1, 4), (6, 2)):
        k.support_x, k.support_y = sx, sy
        assert _grid_both(p, k, *_rows(p, 700, sx + sy)) > 0


@pytest.mark.parametrize("rows,centre", [(1, None), (1, (0, 0)), (257, (3, -5)), (20000, (0, 0)),
                                         (5000, (31, -31))])
def test_crowded_cells(rows, centre):
    p = small_problem(npix=64, n_antennas=5, seed=2)
    k = GriddingKernel.from_taps(np.random.default_rng(7).uniform(0.1, 1.0, (7, 7))
                                 .astype(np.float32))
    print(f"case: gridder {rows} rows at {centre}", flush=True)
    _grid_both(p, k, *_rows(p, rows, rows, centre))


@pytest.mark.parametrize("npix,m,n,rows,support", [
    (64, 1, 1, 5000, None), (64, 1, 1, 60000, None),    # single taps
    (64, 2, 2, 300000, None),                           # crowded cells of a small grid
    (2048, 1, 1, 1, None), (2048, 7, 9, 100, None), (1024, 3, 2, 33, None),  # few rows
    (2048, 5, 6, 120, (6, 2)), (2048, 33, 35, 3, None),
])
def test_sums_by_entry(npix, m, n, rows, support):
    p = small_problem(npix=npix, n_antennas=5, seed=2, dump_seconds=3600.0)
    k = GriddingKernel.from_taps(np.random.default_rng(m * n).uniform(0.1, 1.0, (m, n))
                                 .astype(np.float32))
    if support:
        k.support_x, k.support_y = support
    print(f"case: gridder by entry {npix}^2 {m} x {n} taps {rows} rows", flush=True)
    _grid_both(p, k, *_rows(p, rows, rows + m))


@pytest.mark.parametrize("runs", [(1, 2, 3, 5000), (15, 16, 17, 32, 4000), (79, 80, 81, 144, 6000),
                                  (63, 64, 65, 128, 200, 1, 6000)])
def test_runs_of_entries(runs):
    """Cells of the given row counts, rows interleaved, one tap."""
    p = small_problem(npix=64, n_antennas=5, seed=2)
    parts = [_rows(p, n, 10 + i, centre=(3 * i + 1, 2 * i - 9)) for i, n in enumerate(runs)]
    uvw, vo, w = (np.concatenate([q[c] for q in parts]) for c in range(3))
    order = np.random.default_rng(len(uvw)).permutation(len(uvw))
    k = GriddingKernel.from_taps(np.full((1, 1), 0.7, np.float32))
    print(f"case: runs {runs}", flush=True)
    assert _grid_both(p, k, uvw[order], vo[order], w[order]) > 0


@pytest.mark.parametrize("scheme", ["uniform", "briggs"])
@pytest.mark.parametrize("runs", [(1,), (15, 16, 17, 1), (63, 64, 65, 79, 80, 81), (4000, 2, 9)])
def test_weighting_runs(scheme, runs):
    """Cells of the given row counts, rows interleaved; one slice and two."""
    p = small_problem(npix=64, n_antennas=5, seed=2)
    rng = np.random.default_rng(sum(runs))
    parts = [_rows(p, n, 10 + i, centre=(3 * i + 1, 2 * i - 9)) for i, n in enumerate(runs)]
    uvw = np.concatenate([q[0] for q in parts])
    w = np.concatenate([q[2] for q in parts]) + np.float32(0.25)
    order = rng.permutation(len(uvw))
    uvw, w = np.ascontiguousarray(uvw[order]), np.ascontiguousarray(w[order])
    f = float(np.float32(p.freq))
    for slices in ([(f, uvw, w)], [(f, uvw, w), (f, uvw[:1], w[:1])]):
        ctx = Context(p, add_data=False)
        bufs = [(fr, DeviceBuffer.from_array(u), DeviceBuffer.from_array(x), u.shape[0])
                for fr, u, x in slices]
        apply_weighting_dev(ctx, scheme, bufs, robust=-0.5)
        dev = [b[2].download(np.float32) for b in bufs]
        ctx.close()
        ref = oracle.weighting(scheme, slices, p.M, p.N, p.deltax, p.deltay, robust=-0.5,
                               taper=None, float_totals=False)
        for a, b in zip(dev, ref):
            assert np.array_equal(a, b)
