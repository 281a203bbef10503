"""GPU parity of the MoE routing sort against the oracle (exact integers), and the chain
routing -> gather + dynamic quantisation -> un-permute on the device."""
import numpy as np
import pytest
import torch

import oracle as orc
import catccos_amd as cc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cumsum", [False, True])
@pytest.mark.parametrize("case", [(64, 4), (1000, 16), (1024, 8), (1025, 8), (16384, 32), (50000, 256), (3, 1), (70000, 1024)])
def test_routing_exact(case, cumsum):
    rows, e = case
    rng = np.random.default_rng(rows + e)
    idx = rng.integers(0, e, rows).astype(np.int32)
    if rows > 10:
        idx[rng.integers(0, rows, 3)] = -1          # dropped entries
        idx[rng.integers(0, rows, 2)] = e
        idx[idx == e // 2] = (e // 2 + 1) % e       # an expert nobody routes to (when e > 1)
    d2s, s2d, cnt = cc.moe_init_routing(torch.from_numpy(idx).cuda(), e, cumsum)
    torch.cuda.synchronize()
    wd, ws, wc = orc.moe_init_routing(idx, e, cumsum)
    assert np.array_equal(cnt.cpu().numpy(), wc)
    assert np.array_equal(s2d.cpu().numpy(), ws)
    assert np.array_equal(d2s.cpu().numpy(), wd)


@pytest.mark.parametrize("case", [(1, 1), (63, 3), (64, 256), (1000, 16), (4097, 200), (8192, 256), (8192, 1), (8193, 256), (500, 257)])
def test_routing_one_workgroup_equals_three_launches(case):
    """Up to 1024 rows and 256 experts one workgroup does the whole sort, up to 32768 one launch of a workgroup per 1024; the general path (three launches,
    `routing_three_launches`) and the oracle give the same integers, also past the limit of experts and with dropped routes."""
    rows, e = case
    rng = np.random.default_rng(rows * 7 + e)
    idx = rng.integers(-1, e + 1, rows).astype(np.int32)      # -1 and e are dropped
    want = orc.moe_init_routing(idx, e)
    for cumsum in (False, True):
        res = []
        for three in (0, 1):
            cc.set_option("routing_three_launches", three)
            try:
                res.append([t.cpu().numpy() for t in cc.moe_init_routing(torch.from_numpy(idx).cuda(), e, cumsum)])
            finally:
                cc.set_option("routing_three_launches", 0)
        for a, b in zip(*res):
            assert np.array_equal(a, b)
        if not cumsum:
            for a, w in zip(res[0], want):
                assert np.array_equal(a, w)


@pytest.mark.parametrize("rows", [1023, 1024, 1025, 2048, 2049, 4096, 4097, 8191, 8192])
@pytest.mark.parametrize("e", [1, 64, 65, 256])
def test_routing_one_workgroup_edges(rows, e):
    """The kernels of one launch differ in the groups of 1024 rows that they count (1, 2, 4, 8) and scan experts 64 at a time:
    the row counts and expert counts on either side of each limit, with dropped routes (which leave -1 behind the last)."""
    rng = np.random.default_rng(rows * 31 + e)
    idx = rng.integers(-1, e + 1, rows).astype(np.int32)
    for cumsum in (False, True):
        got = [t.cpu().numpy() for t in cc.moe_init_routing(torch.from_numpy(idx).cuda(), e, cumsum)]
        for a, w in zip(got, orc.moe_init_routing(idx, e, cumsum)):
            assert np.array_equal(a, w)


@pytest.mark.parametrize("rows", [1025, 2047, 2049, 8193, 16384, 16385, 32767, 32768, 32769])
@pytest.mark.parametrize("e", [1, 17, 256])
def test_routing_groups_of_1024(rows, e):
    """Every workgroup places 1024 rows and counts all others: the row counts on either side of each instantiation, all rows on one expert (the
    largest counts, and every lane of a wave on the same one) and spread, with dropped routes; nothing is read from or left in the workspace."""
    L = cc._abi.lib()
    rng = np.random.default_rng(rows + e)
    spread = rng.integers(-1, e + 1, rows).astype(np.int32)
    spread[rng.integers(0, rows, 3)] = [2 ** 31 - 1, -2 ** 31, 256]
    nbytes = L.cch_moe_init_routing_workspace_bytes(rows, e)
    for idx in (spread, np.full(rows, e - 1, np.int32), np.full(rows, -1, np.int32)):
        dev = torch.from_numpy(idx).cuda()
        for cumsum in (0, 1):
            d2s, s2d, cnt = (torch.full((n + 1,), -5, dtype=torch.int32, device="cuda") for n in (rows, rows, e))
            ws = torch.full((nbytes // 4,), 99, dtype=torch.int32, device="cuda")
            cc._abi.check(L.cch_moe_init_routing(dev.data_ptr(), rows, e, d2s.data_ptr(), s2d.data_ptr(), cnt.data_ptr(), cumsum, ws.data_ptr(), nbytes,
                                                 torch.cuda.current_stream().cuda_stream))
            for got, w in zip((d2s, s2d, cnt), orc.moe_init_routing(idx, e, bool(cumsum))):
                assert int(got[-1]) == -5 and np.array_equal(got[:-1].cpu().numpy(), w)
            assert rows > 32768 or bool((ws == 99).all())


@pytest.mark.parametrize("case", [(1, 257), (8192, 1024), (33000, 1), (33000, 65), (33000, 255), (33000, 256), (33000, 257), (9000, 1023), (1024 * 1024, 3),
                                  (1024 * 1024 + 1, 3)])
def test_routing_two_launches(case):
    """Without the scan's launch every workgroup of the placement pass sums the histograms itself, experts over 256 threads and chunks over what is
    left: expert counts on either side of a power of two and of 256, the largest, and the last number of chunks before the scan has its own launch again.
    The result is that of the three launches and the oracle's, for any workspace contents."""
    rows, e = case
    rng = np.random.default_rng(rows * 3 + e)
    idx = rng.integers(-1, e + 1, rows).astype(np.int32)
    idx[rng.integers(0, rows, 5)] = [2 ** 31 - 1, -2 ** 31, e, -1, 1 << e.bit_length()]
    L, dev = cc._abi.lib(), torch.from_numpy(idx).cuda()
    nbytes = L.cch_moe_init_routing_workspace_bytes(rows, e)
    for cumsum in (0, 1):
        want = orc.moe_init_routing(idx, e, bool(cumsum))
        for three, fill in ((0, 0x7FFFFFFF), (0, -7), (1, 5)):
            cc.set_option("routing_three_launches", three)
            try:
                d2s, s2d, cnt = (torch.full((n + 1,), -5, dtype=torch.int32, device="cuda") for n in (rows, rows, e))
                ws = torch.full((nbytes // 4 + 1,), fill, dtype=torch.int32, device="cuda")
                cc._abi.check(L.cch_moe_init_routing(dev.data_ptr(), rows, e, d2s.data_ptr(), s2d.data_ptr(), cnt.data_ptr(), cumsum, ws.data_ptr(), nbytes,
                                                     torch.cuda.current_stream().cuda_stream))
                torch.cuda.synchronize()
            finally:
                cc.set_option("routing_three_launches", 0)
            for got, w in zip((d2s, s2d, cnt), want):
                assert int(got[-1]) == -5 and np.array_equal(got[:-1].cpu().numpy(), w)
            assert int(ws[-1]) == fill


def test_routing_skewed_and_sorted_inputs():
    for idx in (np.zeros(5000, np.int32), np.arange(5000, dtype=np.int32) % 7, np.sort(np.arange(5000, dtype=np.int32) % 7)[::-1].copy()):
        d2s, s2d, cnt = cc.moe_init_routing(torch.from_numpy(idx).cuda(), 7)
        torch.cuda.synchronize()
        wd, ws, wc = orc.moe_init_routing(idx, 7)
        assert np.array_equal(d2s.cpu().numpy(), wd) and np.array_equal(s2d.cpu().numpy(), ws) and np.array_equal(cnt.cpu().numpy(), wc)


def test_routing_empty_and_errors():
    d2s, s2d, cnt = cc.moe_init_routing(torch.zeros(0, dtype=torch.int32, device="cuda"), 4)
    torch.cuda.synchronize()
    assert d2s.numel() == 0 and list(cnt.cpu().numpy()) == [0, 0, 0, 0]
    with pytest.raises(cc.CatccosError):
        cc.moe_init_routing(torch.zeros(8, dtype=torch.int32, device="cuda"), 2000)


def test_routing_feeds_gather_quant_and_unpermute():
    """tokens -> routing -> expert-sorted int8 rows; the same maps bring expert-order rows back to token order."""
    rng = np.random.default_rng(4)
    tokens, k, topk, e = 200, 1024, 2, 8
    xb = orc.f32_to_bf16(rng.standard_normal((tokens, k)).astype(np.float32))
    expert_idx = rng.integers(0, e, (tokens, topk)).astype(np.int32)
    x = torch.from_numpy(xb.view(np.int16)).cuda().view(torch.bfloat16)
    d2s, s2d, cnt = cc.moe_init_routing(torch.from_numpy(expert_idx).cuda(), e)
    q, s = cc.dynamic_quant_i8(x, d2s, topk)
    torch.cuda.synchronize()
    wd, ws, wc = orc.moe_init_routing(expert_idx, e)
    wq, wsc = orc.dyn_quant_i8_rows(xb, wd, topk)
    assert np.array_equal(q.cpu().numpy(), wq) and np.array_equal(s.cpu().numpy(), wsc)
    # rows in expert order are the tokens themselves here; un-permute with the inverse map sums each token topk times
    permuted = x[(d2s // topk).long()]
    back = cc.moe_token_unpermute(permuted, s2d, None, topk)
    torch.cuda.synchronize()
    want = orc.f32_to_bf16(orc.bf16_to_f32(xb) * np.float32(topk))
    assert np.array_equal(back.view(torch.int16).cpu().numpy().view(np.uint16), want)
