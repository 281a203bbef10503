"""The 192 x 192 tiles of the mid-size GEMM template against the 256 x 256 kernel: the same bits, at the edges of tiles, of K steps and
of scale rows, and where the library chooses them by itself."""
import pytest
import torch

import catccos_amd as cc

pytestmark = pytest.mark.gpu


def both(f):
    cc.set_option("require_tiled_gemm", 1)
    try:
        cc.set_option("gemm_192_tiles", 0)
        cc.set_option("gemm_kernel", 0)
        want = f()
        cc.set_option("gemm_kernel", -1)
        cc.set_option("gemm_192_tiles", 1)
        got = f()
        cc.set_option("gemm_192_tiles", -1)
        return want, got, f()
    finally:
        cc.set_option("gemm_kernel", -1)
        cc.set_option("gemm_192_tiles", -1)
        cc.set_option("require_tiled_gemm", 0)


# one element of a tile to the last row and column of one, one step of K to many, rows of scales that start off 4-byte boundaries (where MXFP4
# has no such kernel: those five sizes compare the one that is chosen instead)
SIZES = [(1, 8, 64), (191, 184, 128), (192, 192, 256), (193, 200, 320), (385, 576, 384), (500, 392, 1984), (577, 1000, 2112), (40, 3000, 448), (1000, 192, 4096)]


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2", "e2m1"])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_same_bits_as_256x256_tiles(m, n, k, fmt):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, sa = cc.mx_quant(torch.randn(m, k, device="cuda", generator=g).bfloat16(), fmt)
    w = [cc.mx_quant_b(torch.randn(k, n, device="cuda", generator=g).bfloat16(), fmt, trans_b=1) for _ in range(3)]
    b, sb = torch.stack([v[0] for v in w]), torch.stack([v[1] for v in w])
    groups = torch.tensor([m // 3, 0, m - m // 3 - m // 8], dtype=torch.int32, device="cuda")   # an empty group, rows of none behind the last
    for dt in (torch.bfloat16, torch.float16):
        for f in (lambda: cc.mx_matmul(a, sa, b[0], sb[0], fmt, 1, dt), lambda: cc.mx_grouped_matmul(a, sa, b, sb, groups, fmt, 1, dt)):
            want, got, _ = both(f)
            assert torch.isfinite(want.float()).all() and torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("m,n,k", [(1, 8, 96), (193, 200, 224), (385, 576, 352), (500, 392, 1248), (577, 1000, 2144)])
def test_mxfp4_ragged_last_step(m, n, k):
    """Scale rows on 4-byte boundaries and a last step of K (256 elements) three or seven eighths full: K no multiple of 64, an odd number of
    blocks, so the weights are quantised as rows."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, sa = cc.mx_quant(torch.randn(m, k, device="cuda", generator=g).bfloat16(), "e2m1")
    b, sb = cc.mx_quant(torch.randn(n, k, device="cuda", generator=g).bfloat16(), "e2m1")
    assert sa.shape[1] % 4 == 0 and k % 64 == 32
    want, got, _ = both(lambda: cc.mx_matmul(a, sa, b, sb, "e2m1", 1))
    assert torch.isfinite(want.float()).all() and want.float().abs().max() > 0 and torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_mapped_output_rows():
    m, n, k = 300, 264, 512
    g = torch.Generator(device="cuda").manual_seed(1)
    a, sa = cc.mx_quant(torch.randn(m, k, device="cuda", generator=g).bfloat16())
    b, sb = cc.mx_quant_b(torch.randn(k, n, device="cuda", generator=g).bfloat16(), trans_b=1)
    groups = torch.tensor([m], dtype=torch.int32, device="cuda")
    row_map = torch.randperm(m + 20, device="cuda", generator=g)[:m].int()
    row_map[7], row_map[8] = -1, m + 20   # dropped
    out = [torch.full((m + 20, n), 3.0, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
    turn = iter(out)
    want, got, _ = both(lambda: cc.mx_grouped_matmul_mapped(a, sa, b[None], sb[None], groups, row_map, next(turn), "e4m3", 1))
    assert torch.equal(got, want)


@pytest.mark.parametrize("m,n,k", [(3000, 3000, 448), (2881, 3072, 128), (1335, 6856, 192)])
def test_chosen_where_they_make_one_round(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(2)
    a, sa = cc.mx_quant(torch.randn(m, k, device="cuda", generator=g).bfloat16())
    b, sb = cc.mx_quant_b(torch.randn(k, n, device="cuda", generator=g).bfloat16(), trans_b=1)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert cc._abi.lib().cch_gemm_kernel_for(0, 0, 0, m, n, k, 1, cus) == 7   # CCH_GEMM_KERNEL_192X192: every kernel gives these bits
    want, got, chosen = both(lambda: cc.mx_matmul(a, sa, b, sb, "e4m3", 1))
    assert torch.equal(got, want) and torch.equal(chosen, want)
