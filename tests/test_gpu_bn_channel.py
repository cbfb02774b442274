"""Batch-norm of tensors small enough for one workgroup per channel and one
launch per direction: every size class of values per thread, float4 and float
access, against 64-bit references."""
import numpy as np
import pytest

import aetcnn
import refs64
from aetcnn import DeviceArray as D, check

pytestmark = pytest.mark.gpu

SHAPES = [
    # (B, C, H, W): values per channel from one thread's to the limit
    (1, 3, 2, 2), (2, 5, 1, 1), (5, 7, 13, 13), (16, 16, 32, 32), (16, 4, 16, 64),
    (16, 72, 19, 15), (3, 9, 27, 25), (9, 33, 7, 7), (13, 2, 35, 36), (11, 40, 31, 47),
    (16, 20, 32, 33),   # past the limit: two launches
]


@pytest.mark.parametrize("act", [aetcnn.LEAKY, aetcnn.RELU, aetcnn.LINEAR])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_small_tensors(gpu, shape, act):
    B, Cc, H, W = shape
    n = B * H * W
    rng = np.random.default_rng(sum(shape))
    x = (rng.standard_normal(shape) * 1.5 + 0.3).astype(np.float32)
    d = rng.standard_normal(shape).astype(np.float32)
    s = rng.uniform(0.5, 1.5, Cc).astype(np.float32)
    b = rng.uniform(-0.3, 0.3, Cc).astype(np.float32)
    rm, rv = np.full(Cc, 0.2, np.float32), np.full(Cc, 0.7, np.float32)
    dx, dd, ds, db, drm, drv = (D.from_numpy(a) for a in (x, d, s, b, rm, rv))
    y, mean, var, su, md, vd = D(shape), *(D(Cc) for _ in range(5))
    su.zero()
    nb = gpu.ach_bn_workspace(B, Cc, H * W)
    ws = D(nb // 4 + 64)
    check(gpu.ach_bn_train_fwd_from_x(dx.ptr, y.ptr, B, Cc, H * W, ds.ptr, db.ptr, mean.ptr,
                                      var.ptr, drm.ptr, drv.ptr, act, ws.ptr, nb, None))
    x8 = x.astype(np.float64)
    m = x8.mean((0, 2, 3))
    v = ((x8 - m[None, :, None, None]) ** 2).sum((0, 2, 3)) / (n - 1)
    assert np.allclose(mean.numpy(), m, rtol=1e-6, atol=1e-6)
    assert np.allclose(var.numpy(), v, rtol=2e-5)
    assert np.allclose(drm.numpy(), 0.9 * rm + 0.1 * m, rtol=1e-6, atol=1e-6)
    assert np.allclose(drv.numpy(), 0.9 * rv + 0.1 * v, rtol=2e-5)
    # from the stored float moments on, each output is a few fp32 operations
    fm, fv = (a.numpy().astype(np.float64)[None, :, None, None] for a in (mean, var))
    z = (x8 - fm) / (np.sqrt(fv) + 1e-6) * s[None, :, None, None] + b[None, :, None, None]
    slope = {aetcnn.LEAKY: 0.1, aetcnn.RELU: 0.0, aetcnn.LINEAR: 1.0}[act]
    assert np.allclose(y.numpy(), np.where(z > 0, z, z * slope), rtol=1e-5, atol=3e-6)
    near = abs(z) < 1e-5  # rounding decides the branch: no delta there
    d[near] = 0.0
    dd = D.from_numpy(d)
    check(gpu.ach_bn_bwd(dd.ptr, B, Cc, H * W, dx.ptr, None, mean.ptr, var.ptr, ds.ptr, db.ptr,
                         su.ptr, md.ptr, vd.ptr, act, ws.ptr, nb, None))
    g = np.where(z > 0, d, d * slope)
    ref, dgamma = refs64.bn_backward_ref(g, None, x, mean.numpy(), var.numpy(), s, act_leaky=False)
    scale = np.sqrt((g.astype(np.float64) ** 2).sum((0, 2, 3))) + 1e-30
    assert np.all(abs(su.numpy() - dgamma) <= 1e-5 * scale * 3)
    # (a channel of a few values cancels: the bound is relative to its terms)
    lim = 1e-5 * (abs(g).max() * s.max() / np.sqrt(fv.min() + 1e-5) + abs(ref).max())
    assert np.all(abs(dd.numpy() - ref) <= lim)
