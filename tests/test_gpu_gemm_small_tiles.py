"""The kernels with tiles smaller than 256 x 256 (gemm_stream_kernel.h, gemm_mid_kernel.h) at the edges of their tiles: against the
oracle, and against the 256 x 256 kernel on the same operands (setting an order of its tiles keeps a problem on it).  Integer sums are
exact, so the int8 results are the same bits on every kernel; MX results of the kernels that sum K in one accumulator are, too, and
where K is split over waves the fp32 sums differ by a few 2^-23 of their largest term, which moves a bf16 rounding now and then."""
import numpy as np
import pytest
import torch

import oracle as orc
import catccos_amd as cc

pytestmark = pytest.mark.gpu
FMT = {"e4m3": orc.E4M3, "e5m2": orc.E5M2, "e2m1": orc.E2M1}

# rows, K, N: one tile row or column more or less than a tile of 32, 64, 128 or 256; K of one step, with a tail, of many steps; few
# and many tiles to a CU (so that each kernel is chosen for some of them, in either weight layout)
DENSE = [(1, 64, 64), (31, 192, 136), (33, 2048, 72), (65, 1216, 264), (129, 512, 1032), (257, 1088, 2056), (200, 3584, 1024), (513, 640, 4104), (1000, 2432, 1000)]
# group sizes, spare rows, K, N (a multiple of 64: gate and up halves of whole MX blocks)
GROUPED = [([1, 0, 31, 33], 0, 192, 128), ([64, 65, 127, 0, 129], 7, 576, 1088), ([0, 0, 5], 3, 2048, 64), ([3] * 70, 0, 128, 192),
           ([130, 257, 20, 0, 383, 96], 1, 1024, 2112)]


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def on_256(fn):
    cc.set_option("gemm_tile_order", 2)
    try:
        return fn()
    finally:
        cc.set_option("gemm_tile_order", -1)


def close(got, want):
    m = orc.compare(got, want)
    assert m["max_rel_floor1"] <= 1e-2 and m["max_rel_floor_rms"] <= 1e-2, m


def same_but_for_roundings(a, b):
    """bf16 results whose fp32 sums differ in their last bits: one bf16 step (2^-8 of the value) on at most one element in a hundred."""
    a, b = a.float(), b.float()
    differ = a != b
    assert float(differ.float().mean()) <= 1e-2
    assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + 2.0 ** -20 * b.abs().max())[differ].all())


def mx_operands(rng, sizes_rows, k, n, fmt, trans_b, e):
    pa, sa = orc.mx_quant_rows(orc.f32_to_bf16(rng.standard_normal((sizes_rows, k)).astype(np.float32)), FMT[fmt])
    ws = [orc.mx_quant_b(orc.f32_to_bf16((rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)), FMT[fmt], orc.RNE, trans_b) for _ in range(e)]
    return pa, sa, np.stack([w[0] for w in ws]), np.stack([w[1] for w in ws])


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
        assert torch.equal(got, on_256(lambda: cc.w8a8_matmul_dequant(*d, trans_b, dtype)))
        if dtype == torch.bfloat16:
            close(got.float().cpu().numpy(), orc.gemm_i8_dequant(a, b, pt, pc))
    for fmt in ("e4m3", "e5m2", "e2m1"):
        pa, sa, pb, sb = mx_operands(rng, m, k, n, fmt, trans_b, 1)
        d = [dev(x) for x in (pa, sa, pb[0], sb[0])]
        got = cc.mx_matmul(*d, fmt, trans_b)
        close(got.float().cpu().numpy(), orc.mx_gmm(pa, sa, pb, sb, n, k, FMT[fmt], trans_b))
        same_but_for_roundings(got, on_256(lambda: cc.mx_matmul(*d, fmt, trans_b)))


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
        assert torch.equal(fn(*d, trans_b), on_256(lambda: fn(*d, trans_b)))
    for fmt in ("e4m3", "e2m1"):
        pa, sa, pb, sb = mx_operands(rng, t, k, n, fmt, trans_b, e)
        d = [dev(v) for v in (pa, sa, pb, sb, gs)]
        got = cc.mx_grouped_matmul(*d, fmt, trans_b)
        close(got.float().cpu().numpy(), orc.mx_gmm(pa, sa, pb, sb, n, k, FMT[fmt], trans_b, group_sizes=gs))
        assert not got[t - spare:].any()
        same_but_for_roundings(got, on_256(lambda: cc.mx_grouped_matmul(*d, fmt, trans_b)))
        # the MX-quantised activation is what the row quantiser makes of the bf16 one
        act = cc.mx_grouped_matmul_swiglu(*d, fmt, trans_b)
        for out_fmt in ("e4m3", "e2m1"):
            payload, scales = cc.mx_grouped_matmul_swiglu(*d, fmt, trans_b, out_fmt=out_fmt)
            want = cc.mx_quant(act, out_fmt)
            assert torch.equal(payload, want[0]) and torch.equal(scales, want[1])
        # mapped output rows: reversed, every fifth dropped
        rows = torch.arange(t - 1, -1, -1, dtype=torch.int32, device="cuda")
        rows[::5] = -1
        out = torch.full((t, n), 7.0, dtype=torch.bfloat16, device="cuda")
        cc.mx_grouped_matmul_mapped(*d, rows, out, fmt, trans_b)
        want = torch.full_like(out, 7.0)
        keep = (rows >= 0) & (torch.arange(t, device="cuda") < t - spare)
        want[rows[keep].long()] = got[keep]
        assert torch.equal(out, want)
