"""The network kernels where their tiles end: channels and pixels that are no
multiple of a tile, each shape of tile and of weight-gradient block, FP32 and
BF16 weights, against the same layers in FP64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from gpuvmem_amd import native
from gpuvmem_amd.device import Context, DeviceBuffer
from gpuvmem_amd.problem import small_problem

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.fixture(scope="module")
def ctx():
    c = Context(small_problem(npix=64, n_antennas=5, seed=41), add_data=False)
    yield c
    c.close()


def _dev(t):
    return DeviceBuffer.from_array(np.ascontiguousarray(t.numpy(), np.float32))


def _get(buf, shape):
    n = int(np.prod(shape))
    return torch.from_numpy(buf.download(np.float32)[:n].reshape(shape).astype(np.float64))


def _within(got, ref, size, n):
    """A sum of n FP32 products is off by at most n units of rounding of the sum of
    their magnitudes; two more for the bias and the result."""
    assert torch.isfinite(got).all()
    assert ((got - ref).abs() <= (n + 2) * EPS * size + 1e-30).all()


@pytest.mark.parametrize("B,Ci,Co,H,W,K,relu,bf16", [
    (1, 9, 33, 9, 35, 3, True, False),     # 8 x 8 tiles forward; 32 + 64 channel blocks
    (2, 40, 20, 11, 17, 3, True, True),
    (1, 64, 40, 9, 33, 3, False, True),    # pairs of both channels
    (1, 161, 5, 8, 16, 3, True, True),     # more than four groups of input channels
    (1, 1, 1, 1, 1, 3, False, False),
    (2, 3, 65, 126, 510, 3, True, True),   # 8 x 32 tiles of 64 channels, forward
    (2, 65, 3, 126, 510, 3, True, False),  # and for the input gradient
    (1, 33, 5, 9, 33, 1, True, True),
    (2, 5, 70, 8, 31, 1, False, False),
    (2, 3, 65, 126, 510, 1, True, True),
])
def test_convolutions_at_the_edges_of_tiles(ctx, B, Ci, Co, H, W, K, relu, bf16):
    print(f"case: conv {B} {Ci}->{Co} {H}x{W} K={K} relu={relu} bf16={bf16}", flush=True)
    g = torch.Generator().manual_seed(Ci * 1000 + Co)
    x = torch.randn(B, Ci, H, W, generator=g)
    w = torch.randn(Co, Ci, K, K, generator=g) * 0.3
    if bf16:
        w = w.bfloat16().float()
    b = torch.randn(Co, generator=g)
    dy = torch.randn(B, Co, H, W, generator=g)
    dx, dw, db, ddy = _dev(x), _dev(w), _dev(b), _dev(dy)
    if bf16:
        full, dw = dw, DeviceBuffer(2 * w.numel())
        native.check(ctx.lib.gvm_nn_to_bf16(ctx.ctx, full.ptr, dw.ptr, w.numel()), "to_bf16")
    fwd = ctx.lib.gvm_nn_conv_fwd_bf16 if bf16 else ctx.lib.gvm_nn_conv_fwd
    bwd = ctx.lib.gvm_nn_conv_bwd_bf16 if bf16 else ctx.lib.gvm_nn_conv_bwd
    out = ctx.zeros(dy.numel())
    native.check(fwd(ctx.ctx, dx.ptr, dw.ptr, db.ptr, out.ptr, B, Ci, Co, H, W, K, int(relu)), "fwd")
    din, dwg, dbg = ctx.zeros(x.numel()), ctx.zeros(w.numel()), ctx.zeros(Co)
    native.check(bwd(ctx.ctx, dx.ptr, dw.ptr, out.ptr if relu else None, ddy.ptr, din.ptr, dwg.ptr,
                     dbg.ptr, B, Ci, Co, H, W, K, int(relu)), "bwd")
    ctx.sync()
    x, w, b, dy = (t.double() for t in (x, w, b, dy))
    y = _get(out, dy.shape)
    ref = F.conv2d(x, w, b, padding=K // 2)
    size = F.conv2d(x.abs(), w.abs(), b.abs(), padding=K // 2)
    _within(y, ref.clamp(min=0.0) if relu else ref, size, Ci * K * K)
    if relu:
        dy = dy * (y > 0.0)
    back = torch.nn.grad
    _within(_get(din, x.shape), back.conv2d_input(x.shape, w, dy, padding=K // 2),
            back.conv2d_input(x.shape, w.abs(), dy.abs(), padding=K // 2), Co * K * K)
    # FP32 sums of at most 8192 pixels, then FP64
    n = min(B * H * W, 8192)
    _within(_get(dwg, w.shape), back.conv2d_weight(x, w.shape, dy, padding=K // 2),
            back.conv2d_weight(x.abs(), w.shape, dy.abs(), padding=K // 2), n)
    _within(_get(dbg, b.shape), dy.sum((0, 2, 3)), dy.abs().sum((0, 2, 3)), 1)


@pytest.mark.parametrize("H,W,shift", [(2, 2, 0), (6, 4, 0), (34, 66, 0), (18, 20, 1), (2, 1028, 3)])
def test_plane_kernels_at_every_alignment(ctx, H, W, shift):
    """Wide and narrow accesses: rows of 2 mod 4 pixels, pointers `shift` floats
    past the alignment of an allocation."""
    print(f"case: planes {H}x{W} shift={shift}", flush=True)
    B, Cc, Cd, lib = 2, 3, 5, ctx.lib
    x = torch.randn(B, Cc, H, W, generator=torch.Generator().manual_seed(H * W))
    src = DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.float32), x.numpy().ravel()]))
    h, w = H // 2, W // 2

    def run(fn, shape, *args):
        buf = ctx.zeros(shift + int(np.prod(shape)) + 4)
        native.check(fn(ctx.ctx, src.ptr + 4 * shift, buf.ptr + 4 * shift, *args), "plane")
        ctx.sync()
        n = int(np.prod(shape))
        a = buf.download(np.float32)
        assert not a[:shift].any() and not a[shift + n:].any()
        return torch.from_numpy(a[shift:shift + n].reshape(shape).copy())

    got = run(lib.gvm_nn_pool_fwd, (B, Cc, h, w), B, Cc, H, W)
    assert torch.allclose(got, F.avg_pool2d(x, 2), rtol=0, atol=4 * EPS * float(x.abs().max()))
    got = run(lib.gvm_nn_up_fwd, (B, Cd, 2 * H, 2 * W), B, Cc, Cd, 1, H, W)
    up = x.repeat_interleave(2, 2).repeat_interleave(2, 3)
    assert torch.equal(got[:, 1:4], up) and not got[:, 0].any() and not got[:, 4].any()
    # x as the gradient of a pooled 2H x 2W image, and of one upsampled from h x w
    got = run(lib.gvm_nn_pool_bwd, (B, Cc, 2 * H, 2 * W), B, Cc, 2 * H, 2 * W)
    assert torch.equal(got, 0.25 * up)
    got = run(lib.gvm_nn_up_bwd, (B, 2, h, w), B, 2, Cc, 1, h, w)
    assert torch.allclose(got, 4.0 * F.avg_pool2d(x[:, 1:], 2), rtol=0,
                          atol=16 * EPS * float(x.abs().max()))
    got = run(lib.gvm_nn_copy_channels, (B, Cd, H, W), B, 2, Cc, 1, Cd, 2, H * W)
    assert torch.equal(got[:, 2:4], x[:, 1:]) and not got[:, :2].any() and not got[:, 4].any()


def _conv(ctx, x, w, b, relu, split=None):
    """Forward on the device of x viewed as images of `split` pixels (1 x 1 layers)."""
    B, Ci, H, W = x.shape
    Co, _, K, _ = w.shape
    H, W = split or (H, W)
    out = ctx.zeros(B * Co * H * W)
    bufs = [_dev(t) for t in (x, w, b)]
    native.check(ctx.lib.gvm_nn_conv_fwd(ctx.ctx, *(t.ptr for t in bufs), out.ptr, B, Ci, Co, H, W,
                                         K, int(relu)), "fwd")
    ctx.sync()
    return out.download(np.float32).reshape(B, Co, *x.shape[2:])


@pytest.mark.parametrize("B,Ci,Co,H,W,K,relu,bf16", [
    (5, 12, 20, 3, 2, 3, True, False),      # images much smaller than a tile
    (3, 2, 70, 40, 1, 3, True, True),       # and narrower
    (2, 17, 33, 1, 300, 1, True, False),
    (130, 40, 66, 1, 1, 1, False, False),
    (1, 1, 66, 67, 65, 3, True, False),     # one input channel; one output for its gradient
    (2, 16, 65, 126, 510, 3, True, True),   # 8 x 32 tiles of 64 channels, forward
    (2, 65, 16, 126, 510, 3, True, False),  # and for the input gradient
    (2, 20, 30, 125, 260, 1, True, False),  # 1 x 1: full tiles
    (1, 30, 90, 15, 17, 1, False, True),    # 8 x 8 tiles
    (2, 8, 30, 33, 70, 1, True, False),
    (1, 70, 65, 4, 4, 3, True, False),      # 16 pixels: the whole weight gradient at once
    (3, 9, 80, 5, 1, 3, True, True),
    (1, 130, 3, 1, 1, 1, False, False),
    (1, 7, 5, 17, 1, 3, True, False),       # and one more
    (2, 65, 70, 4, 4, 3, True, False),      # 32
    (1, 65, 70, 11, 3, 3, True, False),     # 33: in ranges
])
def test_convolutions_of_small_and_narrow_images(ctx, B, Ci, Co, H, W, K, relu, bf16):
    test_convolutions_at_the_edges_of_tiles(ctx, B, Ci, Co, H, W, K, relu, bf16)


@pytest.mark.parametrize("M,C,K", [(64, 32, 3), (33, 20, 3), (20, 18, 1)])
def test_an_image_does_not_depend_on_its_batch(ctx, M, C, K):
    """The kernel is chosen by the sizes of the whole call; K's order is the same in
    all, so an image gives the same bits alone as among 2,048 (or its pixels as a
    line)."""
    g = torch.Generator().manual_seed(M)
    w, b = torch.randn(M, C, K, K, generator=g) * 0.3, torch.randn(M, generator=g)
    if K == 1:
        x = torch.randn(1, C, 256, 256, generator=g)
        assert np.array_equal(_conv(ctx, x, w, b, True), _conv(ctx, x, w, b, True, (65536, 1)))
        return
    x = torch.randn(2048, C, 4, 4, generator=g)
    all_of_them = _conv(ctx, x, w, b, True)
    for i in (0, 700, 2047):
        assert np.array_equal(_conv(ctx, x[i:i + 1], w, b, True)[0], all_of_them[i])


def test_sixteen_million_images_of_one_pixel(ctx):
    """A block per image would be a launch of 2^32 threads, which is refused."""
    n = 1 << 24
    x = torch.arange(n, dtype=torch.float32).reshape(n, 1, 1, 1) - 1000.0
    w, b = torch.full((1, 1, 1, 1), 0.5), torch.ones(1)
    y = _conv(ctx, x, w, b, True)
    assert np.array_equal(y, (0.5 * x.numpy() + 1.0).clip(min=0.0))


@pytest.mark.parametrize("B,C,H,W,shift", [(300, 7, 2, 2, 0), (41, 5, 4, 4, 0), (9, 13, 6, 10, 1),
                                           (1, 1, 2, 2, 0), (700, 100, 2, 4, 0)])
def test_planes_smaller_than_a_block(ctx, B, C, H, W, shift):
    """Several planes per block, whose count they do not divide."""
    print(f"case: {B} x {C} planes {H}x{W}", flush=True)
    lib = ctx.lib
    x = torch.randn(B, C, H, W, generator=torch.Generator().manual_seed(B))
    src = DeviceBuffer.from_array(np.concatenate([np.zeros(shift, np.float32), x.numpy().ravel()]))

    def run(fn, shape, *args):
        n = int(np.prod(shape))
        buf = ctx.zeros(shift + n + 4)
        native.check(fn(ctx.ctx, src.ptr + 4 * shift, buf.ptr + 4 * shift, *args), "plane")
        ctx.sync()
        a = buf.download(np.float32)
        assert not a[:shift].any() and not a[shift + n:].any()
        return torch.from_numpy(a[shift:shift + n].reshape(shape).copy())

    up = x.repeat_interleave(2, 2).repeat_interleave(2, 3)
    four = 4 * EPS * float(x.abs().max())
    assert torch.equal(run(lib.gvm_nn_up_fwd, (B, C, 2 * H, 2 * W), B, C, C, 0, H, W), up)
    assert torch.equal(run(lib.gvm_nn_pool_bwd, (B, C, 2 * H, 2 * W), B, C, 2 * H, 2 * W), 0.25 * up)
    mean = F.avg_pool2d(x, 2)
    got = run(lib.gvm_nn_pool_fwd, mean.shape, B, C, H, W)
    assert torch.allclose(got, mean, rtol=0, atol=four)
    got = run(lib.gvm_nn_up_bwd, mean.shape, B, C, C, 0, H // 2, W // 2)
    assert torch.allclose(got, 4.0 * mean, rtol=0, atol=4 * four)
    got = run(lib.gvm_nn_copy_channels, (B, C + 2, H, W), B, C, C, 0, C + 2, 1, H * W)
    assert torch.equal(got[:, 1:-1], x) and not got[:, 0].any() and not got[:, -1].any()


def test_more_weights_than_threads_of_a_launch(ctx):
    """21,846 x 21,846 channels of 3 x 3 taps are more than 2^32 weights: their
    gradient's sums are taken by a loop, not by a thread each."""
    Ci = Co = 21846
    B, H, W, n = 33, 1, 1, 21846 * 21846 * 9
    assert n > 1 << 32
    print(f"case: {n} weights", flush=True)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((B, Ci)).astype(np.float32)
    dy = rng.standard_normal((B, Co)).astype(np.float32)
    dx, ddy, dw, db = (DeviceBuffer.from_array(x), DeviceBuffer.from_array(dy), DeviceBuffer(4 * n),
                       ctx.zeros(Co))
    native.check(ctx.lib.gvm_nn_conv_bwd(ctx.ctx, dx.ptr, dx.ptr, None, ddy.ptr, None, dw.ptr, db.ptr,
                                         B, Ci, Co, H, W, 3, 0), "bwd")
    ctx.sync()
    row = np.empty((Ci, 3, 3), np.float32)
    for co in (0, 9999, Co - 1):
        native.check(ctx.lib.gvm_memcpy_d2h(row.ctypes.data, dw.ptr + 4 * co * Ci * 9, row.nbytes), "copy")
        ref = dy[:, co].astype(np.float64) @ x.astype(np.float64)
        size = np.abs(dy[:, co]).astype(np.float64) @ np.abs(x)
        assert np.all(np.abs(row[:, 1, 1] - ref) <= (B + 2) * EPS * size)
        row[:, 1, 1] = 0.0
        assert not row.any()
    assert np.allclose(db.download(np.float32), dy.sum(0, dtype=np.float64), rtol=1e-5, atol=1e-5)


def test_a_thousand_million_pixels(ctx):
    """Images are taken in parts that a launch has room for."""
    n = (1 << 30) + 77
    print(f"case: {n} images of one pixel", flush=True)
    x = torch.arange(n, dtype=torch.int32, device="cuda").remainder_(4096).float()
    y, w, b = torch.full_like(x, -1.0), _dev(torch.full((1,), 0.5)), _dev(torch.ones(1))
    torch.cuda.synchronize()
    native.check(ctx.lib.gvm_nn_conv_fwd(ctx.ctx, x.data_ptr(), w.ptr, b.ptr, y.data_ptr(), n, 1, 1,
                                         1, 1, 1, 1), "fwd")
    ctx.sync()
    assert torch.equal(y, x.mul_(0.5).add_(1.0))


def test_pixels_beyond_the_weight_gradients_indices(ctx):
    """Refused before anything is launched: the last range would end past 2^31."""
    z = ctx.zeros(4)
    st = ctx.lib.gvm_nn_conv_bwd(ctx.ctx, z.ptr, z.ptr, None, z.ptr, None, z.ptr, z.ptr,
                                 (1 << 31) - 100, 1, 1, 1, 1, 1, 0)
    with pytest.raises(native.GvmError):
        native.check(st, "bwd")
