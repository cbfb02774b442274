"""A training step's gradients at the benchmark batch, layer by layer against
64-bit sums: every weight gradient from the step's own activations and deltas,
and every delta from the one of the layer above, with the branches that the
step itself took (the signs of its outputs, the indexes of its pools).  A
whole-network reference cannot hold them this closely, as values near a kink
take another branch in it."""
import numpy as np
import pytest

import aetcnn
import refs64
from aetcnn import configs

pytestmark = pytest.mark.gpu

OUTPUT, DELTA, WEIGHTS, UPDATES, SCALES, MEAN, VARIANCE, X, INDEXES = 0, 1, 2, 3, 6, 10, 11, 12, 14
# fp32 sums of up to 131072 products: 1e-7 to 9e-7 of the tensor (kernels'
# errors); a delta takes a batch-norm or a pool's additions on top
WGRAD_TOL, DELTA_TOL = 2e-6, 4e-6
SAMPLE = 8  # filters of a weight gradient, channels of a delta


def wgrad64(x, dy, k, s, p):
    B, c, H, W = x.shape
    F, oh, ow = dy.shape[1:]
    xp = np.pad(x, ((0, 0), (0, 0), (p, p), (p, p))).astype(np.float64)
    d = np.ascontiguousarray(dy.transpose(1, 0, 2, 3)).reshape(F, -1).astype(np.float64)
    out = np.zeros((F, c, k, k))
    for i in range(k):
        for j in range(k):
            t = xp[:, :, i:i + s * (oh - 1) + 1:s, j:j + s * (ow - 1) + 1:s]
            out[:, :, i, j] = d @ np.ascontiguousarray(t.transpose(0, 2, 3, 1)).reshape(-1, c)
    return out


def dgrad64(dy, w, shape, p):
    """stride 1; w of the channels wanted"""
    B, _, H, W = shape
    F, c, k, _ = w.shape
    oh, ow = dy.shape[2:]
    d, w = dy.reshape(B, F, -1).astype(np.float64), w.astype(np.float64)
    out = np.zeros((B, c, H + 2 * p, W + 2 * p))
    for i in range(k):
        for j in range(k):
            t = np.matmul(np.ascontiguousarray(w[:, :, i, j].T), d)
            out[:, :, i:i + oh, j:j + ow] += t.reshape(B, c, oh, ow)
    return out[:, :, p:p + H, p:p + W]


def rel(a, b):
    return float(np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b))


@pytest.mark.parametrize("name,batch", [("darknet", 128), ("alexnet", 128), ("tiny", 16)])
def test_step_gradients(gpu, name, batch):
    cfg = configs.CONFIGS[name]
    layers = cfg["layers"]
    B, h, w, c = configs.dims(name, batch)
    aetcnn.net_lib().an_rand_seed(3)
    net = aetcnn.Network(B, h, w, c)
    configs.build(net, name)
    net.finalize()
    rng = np.random.default_rng(17)
    x, truth, _ = configs.synthetic_batch(name, 23, B)
    shapes, w0, s0 = [], {}, {}  # (input, output) of each layer
    for i, lay in enumerate(layers):
        inp = (B, c, h, w)
        if lay[0] == "conv":
            n, k, s, p = lay[1:5]
            w0[i] = net.buffer(i, WEIGHTS).reshape(n, c, k, k)
            s0[i] = net.buffer(i, SCALES) if lay[6] else None
            c, h, w = n, (h + 2 * p - k) // s + 1, (w + 2 * p - k) // s + 1
        elif lay[0] == "maxpool":
            k, s, p = lay[1:4]
            h, w = (h + p - k) // s + 1, (w + p - k) // s + 1
        elif lay[0] == "avgpool":
            h = w = 1
        shapes.append((inp, (B, c, h, w)))
    assert np.isfinite(net.train(x, truth))
    convs = [i for i, lay in enumerate(layers) if lay[0] == "conv"]
    for i in convs:
        n, k, s, p = layers[i][1:5]
        xin = x if i == 0 else net.buffer(i - 1, OUTPUT).reshape(shapes[i][0])
        dy = net.buffer(i, DELTA).reshape(shapes[i][1])
        f = np.sort(rng.choice(n, min(n, SAMPLE), replace=False))
        got = net.buffer(i, UPDATES).reshape(w0[i].shape)[f] / np.float32(cfg["momentum"])
        decay = -cfg["decay"] * B * w0[i][f].astype(np.float64)
        ref = wgrad64(xin, dy[:, f], k, s, p) + decay
        e = rel(got, ref)
        # a planted mistake: the reference without the last image's last row
        short = dy[:, f].copy()
        short[-1, :, -1] = 0
        planted = rel(got, wgrad64(xin, short, k, s, p) + decay)
        print(f"{name} layer {i}: weight gradient {e:.2e} (planted {planted:.2e})")
        assert e <= WGRAD_TOL < planted, (name, i, e)
        # the delta of the convolution below, through pools only
        j = i - 1
        while j >= 0 and layers[j][0] == "maxpool":
            j -= 1
        if j < 0 or layers[j][0] != "conv":
            continue
        shape = shapes[i][0]
        ch = np.sort(rng.choice(shape[1], min(shape[1], SAMPLE), replace=False))
        d = dgrad64(dy, w0[i][:, ch], shape, p)
        for q in range(i - 1, j, -1):
            bb, cc, hh, ww = shapes[q][0]
            at = net.buffer(q, INDEXES).reshape(shapes[q][1])[:, ch].astype(np.int64)
            plane = at % (hh * ww) + hh * ww * np.arange(B * len(ch)).reshape(B, len(ch), 1, 1)
            d = np.bincount(plane.ravel(), d.ravel(), B * len(ch) * hh * ww).reshape(
                B, len(ch), hh, ww)
        y = net.buffer(j, OUTPUT).reshape(shapes[j][1])[:, ch]
        slope = {configs.LEAKY: 0.1, configs.RELU: 0.0, configs.LINEAR: 1.0}[layers[j][5]]
        d = np.where(y > 0, d, d * np.float64(np.float32(slope)))
        if layers[j][6]:
            z = net.buffer(j, X).reshape(shapes[j][1])[:, ch]
            d, _ = refs64.bn_backward_ref(d, None, z, net.buffer(j, MEAN)[ch],
                                          net.buffer(j, VARIANCE)[ch], s0[j][ch],
                                          act_leaky=False)
        e = rel(net.buffer(j, DELTA).reshape(shapes[j][1])[:, ch], d)
        print(f"{name} layer {j}: delta {e:.2e}")
        assert e <= DELTA_TOL, (name, j, e)
    net.close()
