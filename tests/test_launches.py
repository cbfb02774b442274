"""Launch decisions of the operation library, recorded on the CPU."""
from launches import record

WS = 1 << 40  # a workspace of any size


def test_lds_limits_do_not_depend_on_the_layer(tmp_path):
    """A kernel's dynamic LDS limit is process-wide: threads that run
    different layers on the same kernel must all set the same one."""
    shapes = [(4, 64, h, w, f, k, 1, k // 2) for f in (32, 64, 96, 128) for k, h, w in
              ((3, 20, 78), (3, 20, 84), (3, 20, 90), (3, 20, 96), (5, 16, 44), (5, 16, 52),
               (5, 16, 60), (5, 16, 66))]
    calls = [[name, [{"conv": s}, "p", "p", "p", "p", WS, None]] for s in shapes
             for name in ("ach_conv_fwd", "ach_conv_bwd_data")]
    calls += [["ach_conv_bwd_filter", [{"conv": s}, "p", "p", "p", "p", WS, None]]
              for s in ((128, 128, 32, 32, 128, 3, 1, 1), (64, 384, 13, 13, 384, 3, 1, 1))]
    sizes, limits = {}, {}
    for r in record(calls, tmp_path):
        assert r["rc"] == 0
        for v in r["launches"]:
            if v["lds"] > 64 * 1024:
                assert v["lds"] <= v["lds_limit"]
                sizes.setdefault(v["kernel"], set()).add(v["lds"])
                limits.setdefault(v["kernel"], set()).add(v["lds_limit"])
    assert any(len(v) > 1 for v in sizes.values())
    assert all(len(v) == 1 for v in limits.values())


def test_two_k_groups_are_tested(tmp_path):
    """The shapes that stand for workgroups of two K groups still run them."""
    calls = [["ach_conv_fwd", [{"conv": s}, "p", "p", "p", "p", WS, None]]
             for s in ((8, 128, 28, 28, 100, 3, 1, 1), (2, 512, 16, 16, 384, 3, 1, 1))]
    for r in record(calls, tmp_path):
        assert any(v["block"][0] == 512 and v["lds"] > 0 and v["grid"][1] > 1
                   for v in r["launches"])


def test_batchnorm_of_many_channels(tmp_path):
    """One workgroup per channel and one launch only where they are few: a
    fully connected layer's thousands of features of a few values take the
    kernels that share a channel set among small workgroups."""
    one = [(16, 72, 285), (128, 1000, 1), (4, 900, 49), (64, 1000, 16)]
    two = [(32, 4096, 1), (128, 4096, 1), (2, 2048, 100), (32, 1001, 1)]
    calls = [["ach_bn_bwd", ["p", *s, "p", None, *["p"] * 7, 7, "p", WS, None]] for s in one + two]
    calls += [["ach_bn_train_fwd_from_x", ["p", "p", *s, *["p"] * 6, 7, "p", WS, None]]
              for s in ((16, 30, 49), (32, 4096, 1), (32, 1001, 1))]
    got = [len(r["launches"]) for r in record(calls, tmp_path)]
    assert got == [1] * len(one) + [2] * len(two) + [1, 2, 2]


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
