"""A weight gradient whose workspace is missing or too small is refused before
any launch, whichever kernel the sizes choose."""
import ctypes as C

import pytest

import aetcnn

ACH_EWORKSPACE = -2


@pytest.mark.parametrize("dims", [
    (128, 4096, 1, 1, 4096, 1, 0),   # fully connected, three-piece tiles
    (128, 256, 4, 4, 3000, 4, 0),    # the same behind a plane
    (128, 512, 1, 1, 512, 1, 0),     # fully connected, fp32 kernels
    (32, 512, 8, 8, 512, 3, 1),      # 3x3, three-piece tiles
], ids=lambda d: "x".join(map(str, d)))
def test_weight_gradient_needs_its_workspace(dims):
    ops = aetcnn.ops()
    B, c, h, w, n, k, p = dims
    d = aetcnn.ConvDesc(B, c, h, w, n, k, 1, p)
    assert ops.ach_conv_bwd_filter_workspace(C.byref(d)) > 4
    mem = 256  # never read: the call is refused
    for ws, nb in ((None, 0), (None, 1 << 40), (mem, 4)):
        assert ops.ach_conv_bwd_filter(C.byref(d), mem, mem, mem, ws, nb, None) == ACH_EWORKSPACE
