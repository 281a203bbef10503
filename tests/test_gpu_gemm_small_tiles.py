"""The kernels with tiles smaller than 256 x 256 (gemm_stream_kernel.h, gemm_mid_kernel.h) at the edges of their tiles: the one
that a problem goes to against the oracle, and each of them, asked for by number, against the 256 x 256 kernel on the same operands.
Integer sums are exact, so the int8 results are the same bits on every kernel; MX results of the kernels that sum K in one
accumulator are, too, and where K is split over waves the fp32 sums differ by a few 2^-23 of their largest term, which moves a bf16
rounding now and then."""
import numpy as np
import pytest
import torch

import oracle as orc
import catccos_amd as cc
from catccos_amd import _abi

pytestmark = pytest.mark.gpu
FMT = {"e4m3": orc.E4M3, "e5m2": orc.E5M2, "e2m1": orc.E2M1}

ALL = range(7)                 # "gemm_kernel": 256 x 256, 64 x 128, 128 x 128, 128 x 256, K over 4 and 8 waves, 256 x 256 with a second launch
SPLIT_K = (4, 5)

# rows, K, N: one tile row or column more or less than a tile of 32, 64, 128 or 256; K of one step, with a tail, of many steps, of an
# odd number of 64-element blocks (scale rows that start off 4-byte boundaries); few and many tiles to a CU
DENSE = [(1, 64, 64), (31, 192, 136), (33, 2048, 72), (65, 1216, 264), (129, 512, 1032), (257, 1088, 2056), (200, 3584, 1024), (513, 640, 4104), (1000, 2432, 1000)]
# group sizes, spare rows, K, N (a multiple of 64: gate and up halves of whole MX blocks)
GROUPED = [([1, 0, 31, 33], 0, 192, 128), ([64, 65, 127, 0, 129], 7, 576, 1088), ([0, 0, 5], 3, 2048, 64), ([3] * 70, 0, 128, 192),
           ([130, 257, 20, 0, 383, 96], 1, 1024, 2112)]


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def on(kernel, fn):
    """fn() with a kernel asked for; None where that kernel does not take the problem."""
    cc.set_option("gemm_kernel", kernel)
    try:
        return fn()
    except cc.CatccosError as e:
        assert e.code == _abi.ENOSUP and "gemm_kernel %d" % kernel in str(e)
        return None
    finally:
        cc.set_option("gemm_kernel", -1)


def on_every(fn, takes, same):
    """fn() on every kernel against the 256 x 256 one; `takes(kernel)`: whether that kernel takes the problem."""
    want = on(0, fn)
    for kernel in ALL[1:]:
        got = on(kernel, fn)
        assert (got is not None) == takes(kernel), kernel
        if got is not None:
            same(kernel, got, want)


def same_bits(kernel, a, b):
    assert torch.equal(a, b), kernel


def same_or_rounded(kernel, a, b):
    if kernel in SPLIT_K:
        same_but_for_roundings(a, b)
    else:
        assert torch.equal(a, b), kernel


def close(got, want):
    m = orc.compare(got, want)
    assert m["max_rel_floor1"] <= 1e-2 and m["max_rel_floor_rms"] <= 1e-2, m


def same_but_for_roundings(a, b):
    """bf16 results whose fp32 sums differ in their last bits: one bf16 step (2^-8 of the value) on at most one element in a hundred."""
    a, b = a.float(), b.float()
    differ = a != b
    assert float(differ.float().mean()) <= 1e-2
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -20 * b.abs().max())[differ].all())


def same_swiglu(kernel, a, b):
    """The gate and up sums are rounded to bf16 before the activation.  Where K is split, one in a hundred of either moves by a step
    (2^-7 of its value at most); that moves silu(g) * u by (1 + |g|) and by 1 times as much relative to itself (g silu'(g) / silu(g) =
    1 + g (1 - sigmoid(g))), and the output's own rounding by once more: within 2^-3 for |g| <= 13, of unit variance here."""
    if kernel not in SPLIT_K:
        return same_bits(kernel, a, b)
    a, b = a.float(), b.float()
    differ = a != b
    assert float(differ.float().mean()) <= 3e-2, kernel
    assert bool(((a - b).abs() <= 2.0 ** -3 * b.abs() + 2.0 ** -20 * b.abs().max())[differ].all()), kernel


def mx_operands(rng, sizes_rows, k, n, fmt, trans_b, e):
    pa, sa = orc.mx_quant_rows(orc.f32_to_bf16(rng.standard_normal((sizes_rows, k)).astype(np.float32)), FMT[fmt])
    ws = [orc.mx_quant_b(orc.f32_to_bf16((rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)), FMT[fmt], orc.RNE, trans_b) for _ in range(e)]
    return pa, sa, np.stack([w[0] for w in ws]), np.stack([w[1] for w in ws])


def no_room(kernel, fmt, k):
    """128 x 256 tiles have no LDS left for MXFP4 scale rows off 4-byte boundaries."""
    return kernel == 3 and fmt == "e2m1" and k // 64 % 2 == 1


@pytest.mark.parametrize("m,k,n", DENSE)
@pytest.mark.parametrize("trans_b", [0, 1])
def test_dense(m, k, n, trans_b):
    rng = np.random.default_rng(m + k + n)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    b = rng.integers(-127, 128, (k, n)).astype(np.int8)
    pt = rng.uniform(0.001, 0.02, m).astype(np.float32)
    pc = rng.uniform(0.001, 0.02, n).astype(np.float32)
    d = [dev(x) for x in (a, np.ascontiguousarray(b.T) if trans_b else b, pt, pc)]
    for dtype in (torch.bfloat16, torch.float16):
        got = cc.w8a8_matmul_dequant(*d, trans_b, dtype)
        same_bits(-1, got, on(0, lambda: cc.w8a8_matmul_dequant(*d, trans_b, dtype)))
        on_every(lambda: cc.w8a8_matmul_dequant(*d, trans_b, dtype), lambda kernel: kernel != 6, same_bits)
        if dtype == torch.bfloat16:
            close(got.float().cpu().numpy(), orc.gemm_i8_dequant(a, b, pt, pc))
    for fmt in ("e4m3", "e5m2", "e2m1"):
        pa, sa, pb, sb = mx_operands(rng, m, k, n, fmt, trans_b, 1)
        d = [dev(x) for x in (pa, sa, pb[0], sb[0])]
        got = cc.mx_matmul(*d, fmt, trans_b)
        close(got.float().cpu().numpy(), orc.mx_gmm(pa, sa, pb, sb, n, k, FMT[fmt], trans_b))
        same_but_for_roundings(got, on(0, lambda: cc.mx_matmul(*d, fmt, trans_b)))
        on_every(lambda: cc.mx_matmul(*d, fmt, trans_b), lambda kernel: kernel != 6 and not no_room(kernel, fmt, k), same_or_rounded)


@pytest.mark.parametrize("sizes,spare,k,n", GROUPED)
@pytest.mark.parametrize("trans_b", [0, 1])
def test_grouped(sizes, spare, k, n, trans_b):
    rng = np.random.default_rng(len(sizes) + k + n)
    gs, e, t = np.array(sizes, np.int32), len(sizes), sum(sizes) + spare
    x = rng.integers(-127, 128, (t, k)).astype(np.int8)
    w = rng.integers(-127, 128, (e, k, n)).astype(np.int8)
    pt = rng.uniform(0.0001, 0.002, t).astype(np.float32)
    pc = rng.uniform(0.001, 0.02, (e, n)).astype(np.float32)
    d = [dev(v) for v in (x, np.ascontiguousarray(w.transpose(0, 2, 1)) if trans_b else w, gs, pt, pc)]
    act = cc.gmm_dequant_swiglu(*d, trans_b)
    close(act.float().cpu().numpy(), orc.gmm_i8_dequant_swiglu(x, w, gs, pt, pc))
    for fn in (cc.gmm_dequant, cc.gmm_dequant_swiglu, lambda *a: torch.cat([v.flatten() for v in cc.gmm_dequant_swiglu_mx(*a)])):
        same_bits(-1, fn(*d, trans_b), on(0, lambda: fn(*d, trans_b)))
        on_every(lambda: fn(*d, trans_b), lambda kernel: True, same_bits)
    for fmt in ("e4m3", "e2m1"):
        pa, sa, pb, sb = mx_operands(rng, t, k, n, fmt, trans_b, e)
        d = [dev(v) for v in (pa, sa, pb, sb, gs)]
        takes = lambda kernel: not no_room(kernel, fmt, k)
        got = cc.mx_grouped_matmul(*d, fmt, trans_b)
        close(got.float().cpu().numpy(), orc.mx_gmm(pa, sa, pb, sb, n, k, FMT[fmt], trans_b, group_sizes=gs))
        assert not got[t - spare:].any()
        same_but_for_roundings(got, on(0, lambda: cc.mx_grouped_matmul(*d, fmt, trans_b)))
        on_every(lambda: cc.mx_grouped_matmul(*d, fmt, trans_b), takes, same_or_rounded)
        on_every(lambda: cc.mx_grouped_matmul_swiglu(*d, fmt, trans_b), takes, same_swiglu)
        # reversed rows, every fifth dropped
        rows = torch.arange(t - 1, -1, -1, dtype=torch.int32, device="cuda")
        rows[::5] = -1
        keep = (rows >= 0) & (torch.arange(t, device="cuda") < t - spare)
        for kernel in (-1, *ALL):
            if not takes(kernel):
                continue
            # the MX-quantised activation is what the row quantiser makes of the bf16 one
            act = on(kernel, lambda: cc.mx_grouped_matmul_swiglu(*d, fmt, trans_b))
            for out_fmt in ("e4m3", "e2m1"):
                payload, scales = on(kernel, lambda: cc.mx_grouped_matmul_swiglu(*d, fmt, trans_b, out_fmt=out_fmt))
                want = cc.mx_quant(act, out_fmt)
                assert torch.equal(payload, want[0]) and torch.equal(scales, want[1]), kernel
            # mapped output rows
            plain = on(kernel, lambda: cc.mx_grouped_matmul(*d, fmt, trans_b))
            out = torch.full((t, n), 7.0, dtype=torch.bfloat16, device="cuda")
            on(kernel, lambda: cc.mx_grouped_matmul_mapped(*d, rows, out, fmt, trans_b))
            want = torch.full_like(out, 7.0)
            want[rows[keep].long()] = plain[keep]
            assert torch.equal(out, want), kernel
