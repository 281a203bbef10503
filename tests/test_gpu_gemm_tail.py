"""Grouped problems whose last, partly filled round of 256 x 256 tiles is a second launch of smaller ones (gemm_tail.h): the same bits
as the 256 x 256 kernel gives on its own (setting an order of its tiles keeps it alone) - both sum K in ascending order in one
accumulator - so the results are compared exactly."""
import numpy as np
import pytest
import torch

import catccos_amd as cc

pytestmark = pytest.mark.gpu

# group sizes, rows of no group, rows cut off the last groups, N; the second launch takes, of 256 CUs' tiles (16 column tiles, the last 2):
CASES = [
    ([513, 577, 575, 448, 704, 449, 0, 830], 5, 0, 4096),       # four remainders of 1, 62, 63 and 65 rows; 192 and 193 stay
    ([300] * 4 + [200] * 11 + [0], 0, 0, 4096),                 # three of four that are alike
    ([300] * 4 + [200] * 11 + [900], 0, 900, 4096),             # the same, the last group past the end of the rows
    ([449] * 9 + [0], 0, 0, 4096),                              # none: 193 rows each
    ([448] * 9 + [0], 0, 0, 4090 // 8 * 8),                     # two of 192 rows; a ragged last column tile
    (list(np.random.default_rng(3).integers(0, 400, 128)), 3, 0, 512),   # about forty of 128 groups, two to four per lane
]


def alone(fn):
    cc.set_option("gemm_tile_order", 2)
    try:
        return fn()
    finally:
        cc.set_option("gemm_tile_order", -1)


def check(fn):
    got, want = fn(), alone(fn)
    for a, b in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("sizes,spare,cut,n", CASES)
def test_same_bits(sizes, spare, cut, n):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n + len(sizes))
    e, t, k = len(sizes), int(sum(sizes)) + spare - cut, 4096
    gs = torch.tensor([int(s) for s in sizes], dtype=torch.int32, device="cuda")

    def codes(*shape):
        return torch.randint(0, 120, shape, dtype=torch.uint8, device="cuda", generator=gen)

    def scales(*shape):
        return torch.randint(110, 120, shape, dtype=torch.uint8, device="cuda", generator=gen)

    rows = torch.arange(t - 1, -1, -1, dtype=torch.int32, device="cuda")
    rows[::5] = -1
    for fmt, pack in (("e4m3", 1), ("e2m1", 2)):
        kk = k * pack
        a, sa = codes(t, kk // pack), scales(t, kk // 32)
        for trans_b in (0, 1):
            b, sb = codes(e, *((n, kk // pack) if trans_b else (kk, n // pack))), scales(e, n * (kk // 32))
            check(lambda: cc.mx_grouped_matmul(a, sa, b, sb, gs, fmt, trans_b))
            if trans_b:
                if n % 128 == 0:
                    check(lambda: cc.mx_grouped_matmul_swiglu(a, sa, b, sb, gs, fmt, trans_b, out_fmt="e4m3"))

                def mapped():
                    out = torch.full((t, n), 7.0, dtype=torch.bfloat16, device="cuda")
                    cc.mx_grouped_matmul_mapped(a, sa, b, sb, gs, rows, out, fmt, trans_b)
                    return out
                check(mapped)
    x = torch.randint(-127, 128, (t, k), dtype=torch.int8, device="cuda", generator=gen)
    w = torch.randint(-127, 128, (e, n, k), dtype=torch.int8, device="cuda", generator=gen)
    pt, pc = torch.rand(t, device="cuda", generator=gen) * 0.002, torch.rand(e, n, device="cuda", generator=gen) * 0.02
    check(lambda: cc.gmm_dequant(x, w, gs, pt, pc, 1))
    check(lambda: cc.gmm_dequant_swiglu(x, w, gs, pt, pc, 1))
    check(lambda: cc.gmm_dequant(x, w.view(e, k, n), gs, pt, pc, 0))
