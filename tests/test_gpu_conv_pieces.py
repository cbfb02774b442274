"""The convolution kernels that take every float as three bf16 pieces
(conv_split.hip, conv_wsplit.hip): forward, input gradient and weight
gradient against 64-bit references where their tiles, channel chunks and K
parts end, and infinities and NaNs.

Bound, per output: the six piece products kept of a*b leave out less than
2^-24 |ab|, and a matrix instruction adds 16 products at once, so with
K' = k*k*ceil(C/16) instructions (and a few more additions for K parts)
|error| <= (K' + 8) 2^-24 sum |a||b|.  That bound is for indexing: over long
sums it would hide a missing piece product, which outputs of a single product
each (test_single_products) show at once."""
import ctypes as C

import numpy as np
import pytest

import aetcnn
import refs64
from aetcnn import DeviceArray as D, check

pytestmark = pytest.mark.gpu

SHAPES = [
    # (B, C, H, W, F, k, p)
    (1, 16, 8, 16, 32, 3, 1),      # one tile, one chunk, one wave of filters
    (2, 17, 5, 5, 1, 3, 1),        # ragged chunk of one channel, one filter, images in a tile
    (3, 31, 9, 7, 33, 3, 1),       # 33 filters: two waves along M, ragged N
    (2, 48, 13, 13, 65, 3, 1),     # 65 filters: three waves, three chunks
    (1, 47, 37, 29, 97, 3, 1),     # 97 filters: four waves
    (2, 64, 16, 16, 130, 3, 1),    # M tiles of 128 with a ragged second
    (1, 32, 6, 64, 40, 3, 1),      # two rows of 64 per tile
    (1, 16, 3, 130, 24, 3, 1),     # rows wider than a tile
    (3, 24, 4, 4, 20, 3, 0),       # no padding: the input gradient pads by 2
    (2, 32, 7, 6, 48, 3, 2),       # padding 2
    (9, 40, 8, 8, 16, 3, 1),       # two images per tile, odd batch
    (5, 20, 9, 9, 30, 5, 2),       # 5x5
    (2, 33, 27, 27, 96, 5, 2),     # 5x5 on odd planes: one LDS buffer
    (2, 16, 8, 8, 16, 5, 0),       # 5x5 without padding
    (64, 128, 8, 8, 128, 3, 1),    # K slices
    (128, 96, 13, 13, 256, 3, 1),  # a grid between one and two rounds
    (8, 128, 28, 28, 100, 3, 1),   # two K groups of a workgroup, slices, ragged filters
    (2, 512, 16, 16, 384, 3, 1),   # two K groups in each of 16 slices
]


def bound(absref, k, c):
    return (k * k * -(-c // 16) + 8) * 2.0 ** -24 * absref


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_forward_and_input_gradient(gpu, shape):
    B, Cc, H, W, F, k, p = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    w = rng.standard_normal((F, Cc, k, k)).astype(np.float32)
    oh, ow = H + 2 * p - k + 1, W + 2 * p - k + 1
    dy = rng.standard_normal((B, F, oh, ow)).astype(np.float32)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, 1, p)
    nb = max(gpu.ach_conv_fwd_workspace(C.byref(d)), gpu.ach_conv_bwd_data_workspace(C.byref(d)))
    ws, dx_, dw, ddy = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D.from_numpy(dy)
    y, dx = D(dy.shape), D(x.shape)
    check(gpu.ach_conv_fwd(C.byref(d), dx_.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    check(gpu.ach_conv_bwd_data(C.byref(d), ddy.ptr, dw.ptr, dx.ptr, ws.ptr, nb, None))
    ref, mag = refs64.conv_ref(x, w, 1, p), refs64.conv_ref(abs(x), abs(w), 1, p)
    assert np.all(abs(y.numpy() - ref) <= bound(mag, k, Cc))
    ref = refs64.dgrad_ref(dy, w, x.shape, 1, p)
    mag = refs64.dgrad_ref(abs(dy), abs(w), x.shape, 1, p)
    assert np.all(abs(dx.numpy() - ref) <= bound(mag, k, F))


# the piece products left out (below 2^-24 of a product, and 2^-10 of that),
# the rounding of the sum of the small ones and that of the result
ONE_PRODUCT = 2.1 * 2.0 ** -24


def one_each(rng, groups, members):
    """A member for each group, every member in turn in a random order."""
    return np.resize(rng.permutation(members), groups)


@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[3], SHAPES[4], SHAPES[5], SHAPES[12],
                                   SHAPES[14], SHAPES[16], SHAPES[17]],
                         ids=lambda s: "x".join(map(str, s)))
def test_single_products(gpu, shape):
    """Filters with one nonzero weight for each output (and, for the input
    gradient, for each input channel): every sum is one product, which all
    six piece products make exact to ONE_PRODUCT and any five do not."""
    B, Cc, H, W, F, k, p = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    oh, ow = H + 2 * p - k + 1, W + 2 * p - k + 1
    dy = rng.standard_normal((B, F, oh, ow)).astype(np.float32)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, 1, p)
    nb = max(gpu.ach_conv_fwd_workspace(C.byref(d)), gpu.ach_conv_bwd_data_workspace(C.byref(d)))
    ws, dx_, ddy, y, dx = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(dy), D(dy.shape), D(x.shape)
    for fwd in (True, False):
        w = np.zeros((F, Cc, k, k), np.float32)
        n, m = (F, Cc) if fwd else (Cc, F)
        at = one_each(rng, n, m * k * k)
        a, i, j = at // (k * k), at // k % k, at % k
        v = rng.standard_normal(n).astype(np.float32)
        if fwd:
            w[np.arange(F), a, i, j] = v
        else:
            w[a, np.arange(Cc), i, j] = v
        dw = D.from_numpy(w)
        if fwd:
            check(gpu.ach_conv_fwd(C.byref(d), dx_.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
            got, ref = y.numpy(), refs64.conv_ref(x, w, 1, p)
        else:
            check(gpu.ach_conv_bwd_data(C.byref(d), ddy.ptr, dw.ptr, dx.ptr, ws.ptr, nb, None))
            got, ref = dx.numpy(), refs64.dgrad_ref(dy, w, x.shape, 1, p)
        assert np.all(abs(got - ref) <= ONE_PRODUCT * abs(ref)), fwd


def test_single_products_of_weight_gradients(gpu):
    """One nonzero delta for each filter."""
    for shape in WGRAD:
        B, Cc, H, W, F = shape
        rng = np.random.default_rng(sum(shape))
        x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
        dy = np.zeros((B, F, H, W), np.float32)
        at = one_each(rng, F, B * H * W)
        b, i, j = at // (H * W), at // W % H, at % W
        v = rng.standard_normal(F).astype(np.float32)
        dy[b, np.arange(F), i, j] = v
        got = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32))
        xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1))).astype(np.float64)
        ref = np.stack([np.stack([xp[b, :, i + ki, j + kj] for kj in range(3)], -1)
                        for ki in range(3)], -2) * v.astype(np.float64)[:, None, None, None]
        assert np.all(abs(got - ref) <= ONE_PRODUCT * abs(ref)), shape


@pytest.mark.parametrize("B,K,F", [(33, 128, 128), (64, 300, 130), (130, 520, 256),
                                   (70, 2900, 2890)], ids=str)
def test_single_products_fully_connected(gpu, B, K, F):
    rng = np.random.default_rng(B + K + F)
    x = rng.standard_normal((B, K)).astype(np.float32)
    dy = rng.standard_normal((B, F)).astype(np.float32)
    d = aetcnn.ConvDesc(B, K, 1, 1, F, 1, 1, 0)
    r = C.byref(d)
    nb = max(gpu.ach_conv_fwd_workspace(r), gpu.ach_conv_bwd_data_workspace(r),
             gpu.ach_conv_bwd_filter_workspace(r))
    ws, dx_, ddy = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(dy)
    y, dx, g = D((B, F)), D((B, K)), D((F, K))
    w = np.zeros((F, K), np.float32)
    at = one_each(rng, F, K)
    w[np.arange(F), at] = rng.standard_normal(F)
    dw = D.from_numpy(w)
    check(gpu.ach_conv_fwd(r, dx_.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    ref = x[:, at].astype(np.float64) * w[np.arange(F), at]
    assert np.all(abs(y.numpy() - ref) <= ONE_PRODUCT * abs(ref))
    w = np.zeros((F, K), np.float32)
    at = one_each(rng, K, F)
    w[at, np.arange(K)] = rng.standard_normal(K)
    dw = D.from_numpy(w)
    check(gpu.ach_conv_bwd_data(r, ddy.ptr, dw.ptr, dx.ptr, ws.ptr, nb, None))
    ref = dy[:, at].astype(np.float64) * w[at, np.arange(K)]
    assert np.all(abs(dx.numpy() - ref) <= ONE_PRODUCT * abs(ref))
    one = np.zeros((B, F), np.float32)
    at = one_each(rng, F, B)
    one[at, np.arange(F)] = dy[at, np.arange(F)]
    g.zero()
    done = D.from_numpy(one)
    check(gpu.ach_conv_bwd_filter(r, dx_.ptr, done.ptr, g.ptr, ws.ptr, nb, None))
    ref = dy[at, np.arange(F)].astype(np.float64)[:, None] * x[at]
    assert np.all(abs(g.numpy() - ref) <= ONE_PRODUCT * abs(ref))


@pytest.mark.parametrize("shape", [
    (8, 128, 20, 56, 96, 5, 2),    # fp32: 13 parts of K
    (8, 128, 20, 66, 96, 5, 2),
    (2, 512, 10, 10, 64, 5, 2),    # few tiles, long sums
    (4, 500, 12, 12, 30, 3, 1),
    (8, 512, 8, 8, 512, 3, 1),
], ids=lambda s: "x".join(map(str, s)))
def test_error_against_fp32_form(gpu, shape):
    """No further from 64 bits than the fp32 form of the same call, which adds
    up K in many parts on small grids."""
    B, Cc, H, W, F, k, p = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    w = rng.standard_normal((F, Cc, k, k)).astype(np.float32)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, 1, p)
    nb = gpu.ach_conv_fwd_workspace(C.byref(d))
    ws, dx, dw, wt = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D(w.size)
    job = aetcnn.FilterJob(d, dw.ptr, wt.ptr, None)
    check(gpu.ach_conv_prepare_filters(1, C.byref(job), None))
    a, b = D((B, F, H, W)), D((B, F, H, W))
    check(gpu.ach_conv_fwd_prepared(C.byref(d), dx.ptr, wt.ptr, a.ptr, ws.ptr, nb, None))
    check(gpu.ach_conv_fwd_train_prepared(C.byref(d), dx.ptr, wt.ptr, None, aetcnn.LINEAR, b.ptr,
                                          ws.ptr, nb, None))
    ref = refs64.conv_ref(x, w, 1, p)
    e = [rel_rms(t.numpy(), ref) for t in (a, b)]
    print(f"{shape}: {e[0]:.2e}, fp32 {e[1]:.2e}")
    assert e[0] <= e[1]


@pytest.mark.parametrize("shape", [(2, 32, 9, 9, 48, 3, 1), (64, 128, 8, 8, 128, 3, 1)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.float32(3.4e38)])
def test_non_finite_and_largest_values(gpu, shape, value):
    """A non-finite (or just finite) input or weight gives what fp32
    arithmetic gives: the outputs of the fp32 form of the same call agree in
    their infinities and NaNs, and elsewhere to rounding."""
    B, Cc, H, W, F, k, p = shape
    rng = np.random.default_rng(5)
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    w = rng.standard_normal((F, Cc, k, k)).astype(np.float32)
    x[0, 3, 4, 4] = value
    w[7, 1, 0, 2] = value if abs(value) > 3.39e38 else 1.0
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, 1, p)
    nb = gpu.ach_conv_fwd_workspace(C.byref(d))
    ws, dx, dw = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w)
    wt = D(w.size)
    job = aetcnn.FilterJob(d, dw.ptr, wt.ptr, None)
    check(gpu.ach_conv_prepare_filters(1, C.byref(job), None))
    a, b = D((B, F, H, W)), D((B, F, H, W))
    check(gpu.ach_conv_fwd_prepared(C.byref(d), dx.ptr, wt.ptr, a.ptr, ws.ptr, nb, None))
    check(gpu.ach_conv_fwd_train_prepared(C.byref(d), dx.ptr, wt.ptr, None, aetcnn.LINEAR, b.ptr,
                                          ws.ptr, nb, None))
    a, b = a.numpy().astype(np.float64), b.numpy().astype(np.float64)
    fin = np.isfinite(b)
    assert not fin.all() and fin.any()
    assert np.array_equal(np.isnan(a), np.isnan(b))
    assert np.array_equal(a[np.isinf(b)], b[np.isinf(b)])
    near = fin & (abs(b) < 1e30)  # sums without the large value
    assert np.all(abs(a[near] - b[near]) <= 1e-5 * abs(b[near]).max())
    assert np.all(abs(a[fin] - b[fin]) <= 1e-5 * abs(b[fin]) + 1e-5 * abs(b[near]).max())


# magnitudes (input, filter): inputs with subnormals among them, filters near
# the largest float, inputs whose pieces would be below bf16's normal range
SCALES = [(1e-37, 1e10), (1e-38, 1e20), (1e30, 1e-36), (1e-35, 1.0)]


@pytest.mark.parametrize("sx,sw", SCALES, ids=str)
def test_extreme_magnitudes(gpu, sx, sw):
    """The bounds of ordinary magnitudes hold over the floats' whole range."""
    rng = np.random.default_rng(11)

    def draw(scale, *shape):
        return (rng.standard_normal(shape) * scale).astype(np.float32)

    B, Cc, H, W, F, k, p = 8, 64, 8, 8, 64, 3, 1
    x, w = draw(sx, B, Cc, H, W), draw(sw, F, Cc, k, k)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, 1, p)
    nb = gpu.ach_conv_fwd_workspace(C.byref(d))
    ws, dx, dw, y = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D((B, F, H, W))
    check(gpu.ach_conv_fwd(C.byref(d), dx.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    ref, mag = refs64.conv_ref(x, w, 1, p), refs64.conv_ref(abs(x), abs(w), 1, p)
    assert np.all(abs(y.numpy() - ref) <= bound(mag, k, Cc))
    B, Cc, H, W, F = WGRAD[0]
    x, dy = draw(sx, B, Cc, H, W), draw(sw, B, F, H, W)
    got = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32)).astype(np.float64)
    x, dy = x.astype(np.float64), dy.astype(np.float64)
    size = np.sqrt(wgrad_ref(x * x, dy * dy))
    n = 6 * B * H * -(-W // 8) / 2 + 64
    assert np.all(abs(got - wgrad_ref(x, dy)) <= 8 * n ** 0.5 * 2.0 ** -25 * size)
    B, K, F = 64, 512, 256
    x, w = draw(sx, B, K), draw(sw, F, K)
    d = aetcnn.ConvDesc(B, K, 1, 1, F, 1, 1, 0)
    nb = gpu.ach_conv_fwd_workspace(C.byref(d))
    ws, dx, dw, y = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D((B, F))
    check(gpu.ach_conv_fwd(C.byref(d), dx.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    x, w = x.astype(np.float64), w.astype(np.float64)
    assert np.all(abs(y.numpy() - x @ w.T) <= (K // 16 + 40) * 2.0 ** -24 * (abs(x) @ abs(w.T)))


# shapes large enough for the three-piece weight gradient
WGRAD = [
    (32, 512, 8, 8, 512),     # one segment per row: image pairs
    (65, 256, 8, 8, 500),     # a last image without a partner, ragged filters
    (64, 250, 13, 13, 384),   # rows of 13 of 16 positions, ragged channels
    (1, 256, 128, 64, 256),   # one image, four units per row
    (128, 64, 32, 32, 64),    # one tile, most slices
]


def wgrad_ref(x, dy):
    B, Cc, H, W = x.shape
    xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
    out = np.zeros((dy.shape[1], Cc, 3, 3), x.dtype)
    for i in range(3):
        for j in range(3):
            out[:, :, i, j] = np.tensordot(dy, xp[:, :, i:i + H, j:j + W],
                                           axes=([0, 2, 3], [0, 2, 3]))
    return out


def run_wgrad(gpu, x, dy, dw0):
    B, Cc, H, W = x.shape
    d = aetcnn.ConvDesc(B, Cc, H, W, dy.shape[1], 3, 1, 1)
    nb = gpu.ach_conv_bwd_filter_workspace(C.byref(d))
    ws, dx, ddy, ddw = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(dy), D.from_numpy(dw0)
    check(gpu.ach_conv_bwd_filter(C.byref(d), dx.ptr, ddy.ptr, ddw.ptr, ws.ptr, nb, None))
    return ddw.numpy()


@pytest.mark.parametrize("shape", WGRAD, ids=lambda s: "x".join(map(str, s)))
def test_weight_gradient(gpu, shape):
    """n = 6 roundings per 16 positions, random: 8 standard deviations of
    sqrt(n) half-ulps of the largest partial sum."""
    B, Cc, H, W, F = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    dy = rng.standard_normal((B, F, H, W)).astype(np.float32)
    dw0 = rng.standard_normal((F, Cc, 3, 3)).astype(np.float32)
    got = run_wgrad(gpu, x, dy, dw0).astype(np.float64)
    x, dy = x.astype(np.float64), dy.astype(np.float64)
    ref = dw0 + wgrad_ref(x, dy)
    # the partial sums' size: the norms of the products' rows
    size = np.sqrt(wgrad_ref(x * x, dy * dy)) + abs(dw0)
    n = 6 * B * H * -(-W // 8) / 2 + 64
    assert np.all(abs(got - ref) <= 8 * n ** 0.5 * 2.0 ** -25 * size)


@pytest.mark.parametrize("relu", [False, True], ids=["signed", "relu"])
@pytest.mark.parametrize("shape,slices", [((128, 64, 32, 32, 64), 256), ((64, 250, 13, 13, 384), 10),
                                          ((32, 512, 8, 8, 512), 4)], ids=str)
def test_weight_gradient_error(gpu, shape, slices, relu):
    """Relative rms error: a slice's two groups take half of its steps each,
    and a step rounds its sums twice (leading products, small products); the
    slices are added in four chains.  A rounding is uniform within half a
    unit and the sums grow evenly over a chain, whose squares therefore add
    to half the chain's length: error <=
    2^-24 sqrt((2 steps / 2 + (slices / 4 + 4) / 2) / 3).  The mean error, to
    which roundings in one direction would add, stays below a quarter of it."""
    B, Cc, H, W, F = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    if relu:
        x = np.maximum(x, 0)
    dy = rng.standard_normal((B, F, H, W)).astype(np.float32)
    err = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32)).astype(np.float64)
    ref = wgrad_ref(x.astype(np.float64), dy.astype(np.float64))
    err -= ref
    rms = np.sqrt((ref ** 2).mean())
    steps = B * H * -(-W // 8) / 2 / (2 * slices)
    limit = 2.0 ** -24 * ((steps + (slices / 4 + 4) / 2) / 3) ** 0.5
    e = np.sqrt((err ** 2).mean()) / rms
    print(f"{shape}: {e:.2e}, bound {limit:.2e}, mean {err.mean() / rms:.2e}")
    assert e <= limit and abs(err.mean()) / rms <= limit / 4


def test_weight_gradient_error_of_few_slices(gpu):
    """Many tiles leave few slices of K; the chains still stay short enough
    for the error that the fp32 kernel has at this shape, measured 2.5e-7 and
    on inputs after a relu 1.9e-7 (parts of about 144 products)."""
    B, Cc, H, W, F = 10, 349, 43, 43, 463
    rng = np.random.default_rng(4)
    dy = rng.standard_normal((B, F, H, W)).astype(np.float32)
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    for relu, limit in ((False, 2.5e-7), (True, 1.9e-7)):
        x = np.maximum(x, 0) if relu else x
        got = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32)).astype(np.float64)
        e = rel_rms(got, wgrad_ref(x.astype(np.float64), dy.astype(np.float64)))
        print(f"relu {relu}: {e:.2e}, fp32 kernel {limit:.2e}")
        assert e <= limit


@pytest.mark.parametrize("value", [np.inf, np.nan])
def test_weight_gradient_non_finite(gpu, value):
    """One non-finite input reaches its channel's nine taps of every filter
    and nothing else, as in fp32 arithmetic."""
    B, Cc, H, W, F = WGRAD[0]
    rng = np.random.default_rng(3)
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    dy = rng.standard_normal((B, F, H, W)).astype(np.float32)
    x[5, 70, 3, 3] = value
    got = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32))
    want = np.zeros(got.shape, bool)
    want[:, 70] = True
    assert np.array_equal(~np.isfinite(got), want)
    if np.isinf(value):  # its sign: that of the dy it meets
        for i in range(3):
            for j in range(3):
                assert np.array_equal(np.sign(got[:, 70, i, j]), np.sign(dy[5, :, 4 - i, 4 - j]))


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("shape", [WGRAD[0], WGRAD[2]], ids=lambda s: "x".join(map(str, s)))
def test_weight_gradient_non_finite_delta(gpu, shape, value):
    """A non-finite delta meets the padding around the input as zeros, as in
    im2col: every tap that looks beyond an edge from its position is NaN."""
    B, Cc, H, W, F = shape
    rng = np.random.default_rng(7)
    x = rng.standard_normal((B, Cc, H, W)).astype(np.float32)
    dy = rng.standard_normal((B, F, H, W)).astype(np.float32)
    at = {0: (0, 0, 0), 40: (B - 1, H - 1, W - 1), 70: (1, 0, W // 2), 131: (B // 2, H - 1, 1),
          200: (2, H // 2, W - 1), 255: (3, H // 2, 2)}  # filter: image, row, column
    for f, (b, i, j) in at.items():
        dy[b, f, i, j] = value
    got = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32))
    with np.errstate(invalid="ignore"):
        ref = refs64.wgrad_ref(x, dy[:, list(at)], 3, 1, 1)
    some = got[list(at)]
    if np.isinf(value):  # taps within the image are infinite, those beyond it NaN
        assert not np.isnan(ref[5]).any() and np.isnan(ref[0]).sum() == 5 * Cc
    assert np.array_equal(np.isnan(some), np.isnan(ref))
    assert np.array_equal(some[np.isinf(ref)], ref[np.isinf(ref)])
    assert np.isfinite(np.delete(got, list(at), 0)).all()


def rel_rms(a, ref):
    return float(np.linalg.norm(a - ref) / np.linalg.norm(ref))


def test_large_values_error(gpu):
    """Values above 2^103 take the fp32 instructions, in blocks of L products
    whose sums are added one by one.  With roundings uniform within half a
    unit and sums that grow evenly: relative rms error <=
    2^-24 sqrt((L + blocks) / 6)."""
    rng = np.random.default_rng(21)

    def draw(scale, *shape):
        return (rng.standard_normal(shape) * scale).astype(np.float32)

    def bound(block, blocks):
        return 2.0 ** -24 * ((block + blocks) / 6) ** 0.5

    B, Cc, H, W, F = 8, 128, 16, 16, 128
    x, w = draw(1e35, B, Cc, H, W), draw(1e-36, F, Cc, 3, 3)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, 3, 1, 1)
    nb = gpu.ach_conv_fwd_workspace(C.byref(d))
    ws, dx, dw, y = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D((B, F, H, W))
    check(gpu.ach_conv_fwd(C.byref(d), dx.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    e = rel_rms(y.numpy(), refs64.conv_ref(x, w, 1, 1))
    print(f"forward {e:.2e}, bound {bound(9 * 16, Cc // 16):.2e}")
    assert e <= bound(9 * 16, Cc // 16)
    # 832 row steps in at least ten slices
    B, Cc, H, W, F = WGRAD[2]
    x, dy = draw(1e35, B, Cc, H, W), draw(1e-36, B, F, H, W)
    got = run_wgrad(gpu, x, dy, np.zeros((F, Cc, 3, 3), np.float32)).astype(np.float64)
    e = rel_rms(got, wgrad_ref(x.astype(np.float64), dy.astype(np.float64)))
    print(f"weight gradient {e:.2e}, bound {bound(16, 84):.2e}")
    assert e <= bound(16, 84)
    B, K, F = 128, 2900, 2900
    x, w, dy = draw(1e35, B, K), draw(1e-36, F, K), draw(1e-36, B, F)
    d = aetcnn.ConvDesc(B, K, 1, 1, F, 1, 1, 0)
    nb = max(gpu.ach_conv_fwd_workspace(C.byref(d)), gpu.ach_conv_bwd_filter_workspace(C.byref(d)))
    ws, dx, dw, ddy, y, g = D(nb // 4 + 64), *map(D.from_numpy, (x, w, dy)), D((B, F)), D((F, K))
    g.zero()
    check(gpu.ach_conv_fwd(C.byref(d), dx.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    check(gpu.ach_conv_bwd_filter(C.byref(d), dx.ptr, ddy.ptr, g.ptr, ws.ptr, nb, None))
    x, w, dy = (a.astype(np.float64) for a in (x, w, dy))
    for name, a, ref, n in (("fc forward", y, x @ w.T, K), ("fc weight gradient", g, dy.T @ x, B)):
        e = rel_rms(a.numpy(), ref)
        print(f"{name} {e:.2e}, bound {bound(32, n / 32):.2e}")
        assert e <= bound(32, n / 32)


@pytest.mark.parametrize("dims", [(128, 128, 32, 32, 128, 3, 1), (128, 96, 27, 27, 256, 5, 2),
                                  (128, 4096, 1, 1, 4096, 1, 0)], ids=lambda s: "x".join(map(str, s)))
def test_time_of_non_finite_calls(gpu, dims):
    """A diverged network's calls stay within ten times a finite call's time
    (every tile is then computed twice, once on the slower instructions)."""
    B, Cc, H, W, F, k, p = dims
    rng = np.random.default_rng(2)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, 1, p)
    r = C.byref(d)
    nb = max(gpu.ach_conv_fwd_workspace(r), gpu.ach_conv_bwd_data_workspace(r),
             gpu.ach_conv_bwd_filter_workspace(r))
    ws, w = D(nb // 4 + 64), D.from_numpy(rng.standard_normal((F, Cc, k, k)).astype(np.float32))
    finite = D.from_numpy(rng.standard_normal(B * max(Cc, F) * H * W).astype(np.float32))
    nans = D.from_numpy(np.full(B * max(Cc, F) * H * W, np.nan, np.float32))
    out = D(max(B * max(Cc, F) * H * W, F * Cc * k * k))
    ev = [C.c_void_p() for _ in range(2)]
    for e in ev:
        check(gpu.ach_event_create(C.byref(e)))

    def time(call):
        ms = C.c_float()
        call()
        check(gpu.ach_event_record(ev[0], None))
        call()
        check(gpu.ach_event_record(ev[1], None))
        check(gpu.ach_event_sync(ev[1]))
        check(gpu.ach_event_elapsed_ms(ev[0], ev[1], C.byref(ms)))
        return ms.value

    for name, call in (
            ("forward", lambda a: gpu.ach_conv_fwd(r, a.ptr, w.ptr, out.ptr, ws.ptr, nb, None)),
            ("input gradient",
             lambda a: gpu.ach_conv_bwd_data(r, a.ptr, w.ptr, out.ptr, ws.ptr, nb, None)),
            ("weight gradient",
             lambda a: gpu.ach_conv_bwd_filter(r, a.ptr, a.ptr, out.ptr, ws.ptr, nb, None))):
        t = [time(lambda: check(call(a))) for a in (finite, nans)]
        print(f"{name}: {t[0] * 1e3:.0f} us, NaNs {t[1] * 1e3:.0f} us")
        assert t[1] <= 10 * t[0], name
    for e in ev:
        check(gpu.ach_event_destroy(e))


@pytest.mark.parametrize("shape", [
    # (B, C, H, W, F, k, s, p): input gradients by phases
    (3, 48, 9, 7, 20, 3, 2, 1),
    (2, 33, 8, 11, 70, 5, 2, 2),     # ragged channels: dword filter loads
    (2, 130, 6, 6, 16, 3, 2, 1),     # 128-row tiles, ragged
    (2, 8, 7, 9, 12, 1, 2, 0),       # three phases without taps: zeros
    (2, 8, 10, 10, 12, 2, 3, 0),     # a window narrower than the stride
    (1, 12, 13, 13, 9, 5, 4, 3),
    (2, 5, 23, 17, 6, 11, 4, 0),
    (2, 16, 5, 5, 8, 3, 2, 2),       # padding 2
    (2, 4, 2, 3, 8, 2, 2, 0),        # one or two pixels per phase
    (2, 6, 7, 7, 10, 3, 5, 1),       # a stride above the phases' limit
    (1, 36, 11, 10, 195, 5, 2, 2),   # K parts, the last phase's shorter
], ids=lambda s: "x".join(map(str, s)))
def test_strided_input_gradient(gpu, shape):
    """fp32 sums of at most F*k*k products: |error| <= F k k 2^-24 sum |a||b|."""
    B, Cc, H, W, F, k, s, p = shape
    rng = np.random.default_rng(sum(shape))
    w = rng.standard_normal((F, Cc, k, k)).astype(np.float32)
    oh, ow = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    dy = rng.standard_normal((B, F, oh, ow)).astype(np.float32)
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, s, p)
    nb = gpu.ach_conv_bwd_data_workspace(C.byref(d))
    ref = refs64.dgrad_ref(dy, w, (B, Cc, H, W), s, p)
    mag = refs64.dgrad_ref(abs(dy), abs(w), (B, Cc, H, W), s, p)
    dw, ddy = D.from_numpy(w), D.from_numpy(dy)
    # with the queried workspace, and with one image's columns only
    for n in (nb, Cc * k * k * oh * ow * 4):
        ws, dx = D(n // 4 + 64), D.from_numpy(np.full((B, Cc, H, W), 7.0, np.float32))
        check(gpu.ach_conv_bwd_data(C.byref(d), ddy.ptr, dw.ptr, dx.ptr, ws.ptr, n, None))
        assert np.all(abs(dx.numpy() - ref) <= F * k * k * 2.0 ** -24 * mag)


STRIDED = [
    # (B, C, H, W, F, k, s, p): taps beyond dy's edge at some pixels
    (2, 33, 8, 11, 70, 5, 2, 2),     # filters padded to k-tiles, ragged channels
    (4, 32, 64, 64, 64, 5, 2, 2),    # nine taps of 64 filters
    (2, 64, 28, 28, 96, 3, 2, 1),
    (1, 12, 13, 13, 9, 5, 4, 3),
]


def run_strided(gpu, dy, w, shape):
    B, Cc, H, W, F, k, s, p = shape
    d = aetcnn.ConvDesc(B, Cc, H, W, F, k, s, p)
    nb = gpu.ach_conv_bwd_data_workspace(C.byref(d))
    ws, ddy, dw, dx = D(nb // 4 + 64), D.from_numpy(dy), D.from_numpy(w), D((B, Cc, H, W))
    check(gpu.ach_conv_bwd_data(C.byref(d), ddy.ptr, dw.ptr, dx.ptr, ws.ptr, nb, None))
    return dx.numpy().astype(np.float64)


def strided_data(shape):
    B, Cc, H, W, F, k, s, p = shape
    rng = np.random.default_rng(sum(shape))
    w = rng.standard_normal((F, Cc, k, k)).astype(np.float32)
    oh, ow = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    return rng.standard_normal((B, F, oh, ow)).astype(np.float32), w


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("shape", STRIDED, ids=lambda s: "x".join(map(str, s)))
def test_strided_input_gradient_non_finite(gpu, shape, value):
    """A non-finite weight or delta reaches the pixels that its taps meet and
    no other: a tap beyond dy's edge adds nothing (col2im adds no such term),
    where a product with a padding zero would add a NaN."""
    B, Cc, H, W, F, k, s, p = shape
    for i, j in ((0, 0), (k - 1, k - 1), (k // 2, 0)):
        dy, w = strided_data(shape)
        w[F - 1, 1, i, j] = value
        dy[0, 0, 0, 0] = dy[B - 1, 2, -1, -1] = value
        got = run_strided(gpu, dy, w, shape)
        with np.errstate(invalid="ignore"):
            ref = refs64.dgrad_ref(dy, w, (B, Cc, H, W), s, p)
        assert np.isfinite(ref).any() and not np.isfinite(ref).all()
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
        fin = np.isfinite(ref)
        assert np.all(abs(got[fin] - ref[fin]) <= 1e-5 * abs(ref[fin]).max())


@pytest.mark.parametrize("shape", STRIDED[1:3], ids=lambda s: "x".join(map(str, s)))
def test_strided_input_gradient_error(gpu, shape):
    """Each tap's sum over the filters stands by itself.  A rounding of a sum
    is uniform within half a unit in the last place, at most 2^-24 / sqrt(3)
    of it; a chain of F products rounds at most F times while the sum grows
    evenly, so the squares add to F/2 of the last one's, and the taps'
    additions to another half of their number:
    relative rms error <= 2^-24 sqrt((F + taps) / 2 / 3).  (One chain over
    filters and taps is at 1.3 to 2.5 times the error of these sums.)"""
    B, Cc, H, W, F, k, s, p = shape
    dy, w = strided_data(shape)
    ref = refs64.dgrad_ref(dy, w, (B, Cc, H, W), s, p)
    err = np.linalg.norm(run_strided(gpu, dy, w, shape) - ref) / np.linalg.norm(ref)
    taps = (k / s) ** 2
    limit = 2.0 ** -24 * ((F + taps) / 6) ** 0.5
    print(f"{shape}: {err:.2e}, bound {limit:.2e}")
    assert err <= limit


@pytest.mark.parametrize("B,K,F", [
    (33, 128, 128),      # two row fragments, one of them a single row; one tile
    (64, 300, 130),      # K not a multiple of 8, ragged features
    (65, 1024, 700),     # two 64-row fragments
    (130, 520, 256),     # two row tiles, K slices
    (70, 2900, 2890),    # large enough for the weight gradient's tiles
], ids=lambda v: str(v))
def test_fully_connected(gpu, B, K, F):
    """Forward, input gradient and weight gradient (with and without the SGD
    step in its pass) of a fully connected layer."""
    rng = np.random.default_rng(B + K + F)
    x = rng.standard_normal((B, K)).astype(np.float32)
    w = rng.standard_normal((F, K)).astype(np.float32)
    dy = rng.standard_normal((B, F)).astype(np.float32)
    d = aetcnn.ConvDesc(B, K, 1, 1, F, 1, 1, 0)
    nb = max(gpu.ach_conv_fwd_workspace(C.byref(d)), gpu.ach_conv_bwd_data_workspace(C.byref(d)),
             gpu.ach_conv_bwd_filter_workspace(C.byref(d)))
    ws, dx_, dw_, ddy = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D.from_numpy(dy)
    y, dx = D((B, F)), D((B, K))
    check(gpu.ach_conv_fwd(C.byref(d), dx_.ptr, dw_.ptr, y.ptr, ws.ptr, nb, None))
    check(gpu.ach_conv_bwd_data(C.byref(d), ddy.ptr, dw_.ptr, dx.ptr, ws.ptr, nb, None))
    x8, w8, d8 = (a.astype(np.float64) for a in (x, w, dy))
    for got, a, b, n in ((y, x8, w8.T, K), (dx, d8, w8, F)):
        lim = (-(-n // 16) + 40) * 2.0 ** -24 * (abs(a) @ abs(b))
        assert np.all(abs(got.numpy() - a @ b) <= lim)
    v0 = rng.standard_normal((F, K)).astype(np.float32)
    wa, va, wb, vb = (D.from_numpy(a) for a in (w, v0, w, v0))
    dc, lc, mom = np.float32(-5e-4 * B), np.float32(0.01 / B), np.float32(0.9)
    check(gpu.ach_conv_bwd_filter(C.byref(d), dx_.ptr, ddy.ptr, va.ptr, ws.ptr, nb, None))
    lim = (B + 8) * 2.0 ** -24 * (abs(d8.T) @ abs(x8) + abs(v0))
    assert np.all(abs(va.numpy() - (v0 + d8.T @ x8)) <= lim)
    check(gpu.ach_sgd_update(w.size, wa.ptr, va.ptr, dc, lc, mom, None))
    check(gpu.ach_conv_bwd_filter_sgd(C.byref(d), dx_.ptr, ddy.ptr, wb.ptr, vb.ptr, dc, lc, mom,
                                      ws.ptr, nb, None))
    assert np.array_equal(wa.numpy().view(np.uint32), wb.numpy().view(np.uint32))
    assert np.array_equal(va.numpy().view(np.uint32), vb.numpy().view(np.uint32))


def test_fully_connected_non_finite(gpu):
    B, K, F = 64, 512, 256
    rng = np.random.default_rng(1)
    x = rng.standard_normal((B, K)).astype(np.float32)
    w = rng.standard_normal((F, K)).astype(np.float32)
    x[3, 100], w[17, 9] = np.inf, np.nan
    d = aetcnn.ConvDesc(B, K, 1, 1, F, 1, 1, 0)
    nb = gpu.ach_conv_fwd_workspace(C.byref(d))
    ws, dx, dw, y = D(nb // 4 + 64), D.from_numpy(x), D.from_numpy(w), D((B, F))
    check(gpu.ach_conv_fwd(C.byref(d), dx.ptr, dw.ptr, y.ptr, ws.ptr, nb, None))
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w.T.astype(np.float64)
    got = y.numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fin = np.isfinite(ref)
    assert np.all(abs(got[fin] - ref[fin]) <= 1e-5 * abs(ref[fin]).max())


def float_aligned(a):
    """A device copy of a whose address is a multiple of 4 bytes only, and
    what keeps it allocated."""
    base = D(a.size + 5)
    v = D.wrap(base.ptr + 4, a.shape)
    v.upload(a)
    return v, base


@pytest.mark.parametrize("dims", [
    (32, 256, 8, 8, 256, 3, 1, 1),   # 16-byte loads of whole segments, slices
    (2, 64, 16, 16, 130, 3, 1, 1),
    (4, 64, 20, 40, 64, 5, 1, 2),
    (16, 48, 13, 13, 72, 3, 2, 1),   # by phases, float4 filter loads
    (70, 512, 1, 1, 256, 1, 1, 0),   # fully connected, row-major 16-byte loads
    (70, 2904, 1, 1, 2896, 1, 1, 0),
], ids=lambda s: "x".join(map(str, s)))
def test_addresses_of_floats(gpu, dims):
    """Tensors at addresses that are a float's multiple only: the same bits."""
    B, Cc, H, W, F, k, s, p = dims
    rng = np.random.default_rng(sum(dims))
    oh, ow = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    host = [rng.standard_normal(v).astype(np.float32)
            for v in ((B, Cc, H, W), (F, Cc, k, k), (B, F, oh, ow))]
    d = aetcnn.ConvDesc(*dims)
    r = C.byref(d)
    nb = max(gpu.ach_conv_fwd_workspace(r), gpu.ach_conv_bwd_data_workspace(r),
             gpu.ach_conv_bwd_filter_workspace(r))
    ws = D(nb // 4 + 64)
    got = []
    for put in (lambda a: (D.from_numpy(a), None), float_aligned):
        bufs = [put(a) for a in host + [np.zeros_like(a) for a in host]]
        x, w, dy, dx, dw, y = (b[0] for b in bufs)
        check(gpu.ach_conv_fwd(r, x.ptr, w.ptr, y.ptr, ws.ptr, nb, None))
        check(gpu.ach_conv_bwd_data(r, dy.ptr, w.ptr, dx.ptr, ws.ptr, nb, None))
        check(gpu.ach_conv_bwd_filter(r, x.ptr, dy.ptr, dw.ptr, ws.ptr, nb, None))
        got.append([a.numpy().view(np.uint32) for a in (y, dx, dw)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dims", [
    (8, 128, 28, 28, 100, 3, 1, 1), (2, 512, 16, 16, 384, 3, 1, 1), (2, 64, 16, 16, 130, 3, 1, 1),
    (8, 96, 20, 40, 128, 5, 1, 2), (32, 256, 8, 8, 256, 3, 1, 1), (10, 349, 20, 21, 463, 3, 1, 1),
    (1, 36, 11, 10, 195, 5, 2, 2), (16, 48, 13, 13, 72, 3, 2, 1), (130, 520, 1, 1, 256, 1, 1, 0),
], ids=lambda s: "x".join(map(str, s)))
def test_workspace_limits(gpu, dims):
    """Any workspace is refused or enough: nothing is written beyond it, and
    the result is that of the queried size to rounding."""
    B, Cc, H, W, F, k, s, p = dims
    rng = np.random.default_rng(sum(dims))
    oh, ow = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    x, w, dy = (D.from_numpy(rng.standard_normal(v).astype(np.float32))
                for v in ((B, Cc, H, W), (F, Cc, k, k), (B, F, oh, ow)))
    d = aetcnn.ConvDesc(*dims)
    r = C.byref(d)
    out = {"fwd": D(dy.shape), "data": D(x.shape), "filter": D(w.shape)}
    query = {"fwd": gpu.ach_conv_fwd_workspace(r), "data": gpu.ach_conv_bwd_data_workspace(r),
             "filter": gpu.ach_conv_bwd_filter_workspace(r)}
    guard = np.full(1 << 16, 123.0, np.float32)
    for op, n in query.items():
        ref, ran = None, 0
        for nb in sorted({n, n - 4, n * 3 // 4, n // 2, n // 3, n // 5, n // 9, n // 20} - {-4},
                         reverse=True):
            nb = nb // 4 * 4
            ws = D(nb // 4 + guard.size)
            D.wrap(ws.ptr + nb, guard.shape).upload(guard)
            out[op].zero()
            a = {"fwd": (x.ptr, w.ptr), "data": (dy.ptr, w.ptr), "filter": (x.ptr, dy.ptr)}[op]
            f = {"fwd": gpu.ach_conv_fwd, "data": gpu.ach_conv_bwd_data,
                 "filter": gpu.ach_conv_bwd_filter}[op]
            rc = f(r, *a, out[op].ptr, ws.ptr, nb, None)
            assert rc in (aetcnn.ACH_OK, aetcnn.ACH_EWORKSPACE) and (rc == 0 or nb < n)
            got = out[op].numpy().astype(np.float64)
            assert np.array_equal(D.wrap(ws.ptr + nb, guard.shape).numpy(), guard), (op, nb)
            if rc == 0:
                ran += 1
                ref = got if ref is None else ref
                assert np.linalg.norm(got - ref) <= 3e-6 * np.linalg.norm(ref), (op, nb)
        assert ran
