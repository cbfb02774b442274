"""Launch decisions of the operation library, recorded on the CPU."""
from launches import record

WS = 1 << 40  # a workspace of any size


def test_strided_input_gradient_of_few_images(tmp_path):
    """Small grids split K: no workgroup runs a chain of more than eight
    k-tiles of 16 where the card has room for more of them."""
    shapes = [(1, 64, 14, 14, 96, 3, 2, 1), (1, 400, 40, 40, 300, 3, 2, 1),
              (2, 48, 37, 29, 72, 3, 2, 1), (4, 100, 33, 21, 50, 5, 2, 2)]
    calls = [["ach_conv_bwd_data", [{"conv": s}, "p", "p", "p", "p", WS, None]] for s in shapes]
    for s, r in zip(shapes, record(calls, tmp_path)):
        assert r["rc"] == 0
        B, c, h, w, n, k, st, p = s
        gemm = r["launches"][1]
        parts = gemm["grid"][1] // (st * st)
        taps = (-(-k // st)) ** 2  # of the phase with the most
        tiles = taps * -(-n // 16)
        chain = -(-tiles // parts)
        assert chain <= 8 or gemm["grid"][0] * gemm["grid"][1] > 256 or parts == 16, (s, chain)
