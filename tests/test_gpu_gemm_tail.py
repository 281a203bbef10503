"""Grouped problems whose last, partly filled round of 256 x 256 tiles is a second launch of smaller ones (gemm_tail.h), asked for by
number: which rows the second launch takes, against the rule written down on the host, and the same bits as the 256 x 256 kernel
gives on its own - both sum K in ascending order in one accumulator - so the results are compared exactly."""
import numpy as np
import pytest
import torch

import catccos_amd as cc
from catccos_amd import _abi

pytestmark = pytest.mark.gpu
CUS = 256

# group sizes, rows of no group, rows cut off the last groups, N, and the remainders that the second launch takes of 256 CUs' tiles
# (16 column tiles, the last 2)
CASES = [
    ([513, 577, 575, 448, 704, 449, 0, 830], 5, 0, 4096, [1, 62, 63, 65]),    # 192 and 193 rows stay
    ([300] * 4 + [200] * 11 + [0], 0, 0, 4096, [44] * 3),                     # three of four that are alike
    ([300] * 4 + [200] * 11 + [900], 0, 900, 4096, [44] * 3),                 # the same, the last group past the end of the rows
    ([449] * 9 + [0], 0, 0, 4096, []),                                        # 193 rows each: none
    ([448] * 9 + [0], 0, 0, 4090 // 8 * 8, [192] * 2),                        # a ragged last column tile
    ([448] * 10, 0, 0, 4096, []),                                             # four of 192 rows would be 384 small tiles
    (list(np.random.default_rng(3).integers(0, 400, 128)), 3, 0, 512, 46),    # 46 of 128 groups, two to four per lane
]


def on(kernel, fn):
    cc.set_option("gemm_kernel", kernel)
    try:
        return fn()
    finally:
        cc.set_option("gemm_kernel", -1)


def check(fn):
    got, want = on(6, fn), on(0, fn)
    for a, b in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
        assert torch.equal(a, b)


def second_launch(sizes, t, n, swiglu):
    """Rows of each group in the second launch: the smallest remainders (ties by group) that empty the last round of 256-row tiles, if
    there are enough of at most 192 rows and they make at most one tile of 64 rows to a CU."""
    n_out, w = (n // 2, 128) if swiglu else (n, 256)
    cols, small_cols = -(-n_out // w), -(-n_out // (w // 2))
    rows, used = [], 0
    for s in sizes:
        rows.append(min(max(int(s), 0), t - used))
        used += rows[-1]
    total = sum(-(-r // 256) for r in rows) * cols
    want = -(-(total % CUS) // cols) if total >= CUS else 0
    short = sorted((r % 256, g) for g, r in enumerate(rows) if 0 < r % 256 <= 192)[:want]
    taken = [0] * len(rows)
    if len(short) == want and sum(-(-r // 64) for r, _ in short) * small_cols <= CUS:
        for r, g in short:
            taken[g] = r
    return taken


@pytest.mark.parametrize("swiglu", [0, 1])
@pytest.mark.parametrize("sizes,spare,cut,n,remainders", CASES + [
    (list(np.random.default_rng(s).integers(0, 600, e)), s, 100 * s, n, None) for s, (e, n) in enumerate([(5, 7168), (16, 4096), (64, 1024), (65, 1024), (256, 256), (1, 8192)])])
def test_rows_of_the_second_launch(sizes, spare, cut, n, remainders, swiglu):
    t = max(int(sum(sizes)) + spare - cut, 0)
    gs = torch.tensor([int(s) for s in sizes], dtype=torch.int32, device="cuda")
    taken = torch.full((len(sizes),), -1, dtype=torch.int32, device="cuda")
    assert _abi.lib().cch_gemm_tail_rows(gs.data_ptr(), len(sizes), t, n, swiglu, CUS, taken.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    got = taken.cpu().tolist()
    assert got == second_launch(sizes, t, n, swiglu)
    if remainders is not None:
        some = sorted(r for r in got if r)
        assert some == remainders if isinstance(remainders, list) else len(some) == remainders


@pytest.mark.parametrize("sizes,spare,cut,n", [c[:4] for c in CASES])
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
            if n % 128 == 0:
                check(lambda: cc.mx_grouped_matmul_swiglu(a, sa, b, sb, gs, fmt, trans_b, out_fmt="e4m3"))
            if trans_b:
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
    check(lambda: cc.gmm_dequant_swiglu(x, w.view(e, k, n), gs, pt, pc, 0))
