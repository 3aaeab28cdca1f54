"""One context's set-up workspace used from several threads: the gridder on the null
stream beside the adjoint's plan on the context's stream, and griddings beside each
other.  Whole results, so no tolerance."""
import threading

import numpy as np
import pytest

from gpuvmem_amd.device import Context, DeviceBuffer
from gpuvmem_amd.gridding import GriddingKernel, apply_weighting_dev, grid_visibilities_dev
from gpuvmem_amd.problem import small_problem

pytestmark = pytest.mark.gpu


def _rows(p, n, seed):
    rng = np.random.default_rng(seed)
    lam = float(np.float32(2.99792458e8) / np.float32(p.freq))
    du = lam / (p.M * abs(p.deltax) * np.pi / 180.0)
    uvw = np.concatenate([rng.uniform(-0.45 * p.M, 0.45 * p.M, (n, 2)) * du, np.zeros((n, 1))], 1)
    return [DeviceBuffer.from_array(a) for a in
            (uvw, rng.standard_normal((n, 2)).astype(np.float32),
             rng.uniform(0.5, 2.0, n).astype(np.float32))]


def test_gridding_and_gradients_from_several_threads():
    p = small_problem(npix=128, n_antennas=12, seed=9)
    ctx = Context(p)
    d = ctx.image(p.initial_image())
    ctx.chi2(d)
    kernels = [GriddingKernel.from_taps(np.random.default_rng(m).uniform(0.1, 1.0, (m, m))
                                        .astype(np.float32)) for m in (1, 5)]
    jobs = [(kernels[i % 2], _rows(p, n, i), n) for i, n in enumerate((40000, 9000, 90000))]

    def grid(k, bufs, n):
        return grid_visibilities_dev(ctx, k, p.freq, *bufs, n)

    def weights(bufs, n):
        w = DeviceBuffer.from_array(bufs[2].download(np.float32))
        apply_weighting_dev(ctx, "briggs", [(p.freq, bufs[0], w, n)], robust=0.3)
        return [w.download(np.float32)]

    def gradient():
        # the plan is laid out anew each time
        ctx.set_gridding("never")
        r = ctx.zeros(2 * ctx.n)
        ctx.dchi2(d, r)
        ctx.set_gridding("always")
        ctx.add(*extra)
        ctx.chi2(d)
        r = ctx.zeros(2 * ctx.n)
        ctx.dchi2(d, r)
        ctx.sync()
        assert ctx.adjoint_gridded()
        return r.download(np.float32)

    extra = (p.freq, p.uvw[:50], p.vo[:50], p.weight[:50])
    calls = [lambda j=j: grid(*j) for j in jobs] + [lambda: weights(jobs[0][1], jobs[0][2])]
    alone = [c() for c in calls]
    errors = []

    def loop(call, want):
        try:
            for _ in range(12):
                for a, b in zip(call(), want):
                    assert np.array_equal(a, b)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=loop, args=a) for a in zip(calls, alone)]
    for t in threads:
        t.start()
    together = [gradient() for _ in range(12)]
    for t in threads:
        t.join()
    assert not errors, errors
    ctx.close()
    # the same gradients without the other threads
    ctx = Context(p)
    d = ctx.image(p.initial_image())
    ctx.chi2(d)
    for g in together:
        assert np.array_equal(g, gradient())
    ctx.close()
