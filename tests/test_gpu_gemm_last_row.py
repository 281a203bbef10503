"""Rows of A that end inside a dword of the scale array: an odd number of rows of an odd number of E8M0 byte pairs (K an odd
multiple of 64).  The last scales of the last row are the array's last two bytes.  Against the oracle; the relative error of a
row of bf16 roundings is below 2^-9, doubled for the sums' own rounding."""
import numpy as np
import pytest
import torch

import oracle as orc
import catccos_amd as cc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1, 192, 64), (33, 1216, 264), (257, 320, 512)])
@pytest.mark.parametrize("trans_b", [0, 1])
@pytest.mark.parametrize("order", [-1, 2], ids=["default", "256x256"])
def test_last_row_keeps_its_last_scales(m, k, n, trans_b, order):
    rng = np.random.default_rng(m + k)
    pa, sa = orc.mx_quant_rows(orc.f32_to_bf16(rng.standard_normal((m, k)).astype(np.float32)), orc.E4M3)
    pb, sb = orc.mx_quant_b(orc.f32_to_bf16(rng.standard_normal((k, n)).astype(np.float32)), orc.E4M3, orc.RNE, trans_b)
    want = orc.mx_gmm(pa, sa, pb, sb, n, k, orc.E4M3, trans_b)
    cc.set_option("gemm_tile_order", order)
    try:
        dev = [torch.from_numpy(np.ascontiguousarray(x)).cuda() for x in (pa, sa, pb, sb)]
        got = cc.mx_matmul(*dev, "e4m3", trans_b).float().cpu().numpy()
    finally:
        cc.set_option("gemm_tile_order", -1)
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 2.0 ** -8, int(err.argmax())
