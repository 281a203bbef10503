"""The MoE FFN chain of the reference's Ascend950 dispatch-FFN-combine example on one rank, every stage a call
of this library, against the same chain of oracle routines (the structure of the reference's golden,
examples/utils/gen_data_moe.py:460-620, with ep = 1):

    bf16 tokens -> routing sort -> MXFP8 quantise and scatter (packed rows) -> GMM1 + SwiGLU + MXFP8 quantise
    (one kernel, reading the packed rows) -> GMM2 -> weighted un-permute -> bf16 tokens

Stage by stage the device results equal the oracle's to the bit where the stage is byte or index work, and
feed the next device stage; the final tensor is compared with the all-oracle chain."""
import numpy as np
import pytest
import torch

import oracle as orc
import catccos_amd as cc

pytestmark = pytest.mark.gpu


def bf16_dev(bits):
    return torch.from_numpy(bits.view(np.int16)).cuda().view(torch.bfloat16)


def bits(t):
    torch.cuda.synchronize()
    return t.view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("cfg", [(96, 512, 1024, 8, 2), (300, 1024, 512, 16, 6), (64, 256, 512, 4, 1)],
                         ids=["m96-top2", "m300-top6-16experts", "m64-top1"])
def test_ffn_chain_against_oracle_chain(cfg):
    m, k, n, e, topk = cfg
    rng = np.random.default_rng(m + k + e)
    x = orc.f32_to_bf16(rng.standard_normal((m, k)).astype(np.float32))
    expert_idx = np.argsort(rng.random((m, e)), axis=1)[:, :topk].astype(np.int32)
    logits = rng.standard_normal((m, topk)).astype(np.float32)
    probs = (np.exp(logits) / np.exp(logits).sum(1, keepdims=True)).astype(np.float32)
    h = n // 2
    w1 = [orc.f32_to_bf16((rng.standard_normal((k, n)) / np.sqrt(k)).astype(np.float32)) for _ in range(e)]
    w2 = [orc.f32_to_bf16((rng.standard_normal((h, k)) / np.sqrt(h)).astype(np.float32)) for _ in range(e)]
    b1, sb1 = map(np.stack, zip(*[orc.mx_quant_b(w, orc.E4M3, orc.RNE, 0) for w in w1]))      # [E, K, N], scales [E, K/64, N, 2]
    b2, sb2 = map(np.stack, zip(*[orc.mx_quant_b(w, orc.E4M3, orc.RNE, 1) for w in w2]))      # [E, N2 = k, K2 = h] as the golden stores it
    rows = m * topk

    # ---- oracle chain
    d2s_o, s2d_o, cnt_o = orc.moe_init_routing(expert_idx, e)
    packed_o = orc.mx_quant_scatter_packed(x, s2d_o, rows, topk, orc.E4M3)
    a1_o, sa1_o = packed_o[:, :k], packed_o[:, k:]
    _, c1_o = orc.mx_gmm(a1_o, sa1_o, b1, sb1, n, k, orc.E4M3, 0, group_sizes=cnt_o, want_bf16=True)
    act_o = orc.swiglu_bf16(c1_o)
    a2_o, sa2_o = orc.mx_quant_rows(act_o, orc.E4M3)
    _, y_o = orc.mx_gmm(a2_o, sa2_o, b2, sb2, k, h, orc.E4M3, 1, group_sizes=cnt_o, want_bf16=True)
    out_o = orc.moe_token_unpermute(y_o, s2d_o, probs, topk)

    # ---- device chain
    cc.set_option("require_tiled_gemm", 1)
    try:
        d2s, s2d, cnt = cc.moe_init_routing(torch.from_numpy(expert_idx).cuda(), e)
        packed = torch.empty((rows, cc.packed_row_bytes(k)), dtype=torch.uint8, device="cuda")
        cc.mx_quant_scatter_packed(bf16_dev(x), s2d, packed, topk)
        tb1 = (torch.from_numpy(b1).cuda(), torch.from_numpy(sb1).cuda())
        a2, sa2 = cc.mx_grouped_matmul_swiglu_packed(packed, k, tb1[0], tb1[1], cnt, "e4m3", 0, "e4m3")
        y = cc.mx_grouped_matmul(a2, sa2, torch.from_numpy(b2).cuda(), torch.from_numpy(sb2).cuda(), cnt, "e4m3", 1)
        out = cc.moe_token_unpermute(y, s2d, torch.from_numpy(probs).cuda(), topk)
        # the up projection from separate arrays gives the same bytes as from the packed rows
        a2b, sa2b = cc.mx_grouped_matmul_swiglu(packed[:, :k].contiguous(), packed[:, k:].contiguous(), tb1[0], tb1[1], cnt, "e4m3", 0, out_fmt="e4m3")
    finally:
        cc.set_option("require_tiled_gemm", 0)
    torch.cuda.synchronize()

    # index and byte stages: to the bit
    assert np.array_equal(s2d.cpu().numpy(), s2d_o) and np.array_equal(d2s.cpu().numpy(), d2s_o) and np.array_equal(cnt.cpu().numpy(), cnt_o)
    assert np.array_equal(packed.cpu().numpy(), packed_o)
    assert torch.equal(a2, a2b) and torch.equal(sa2, sa2b)
    # the quantised activation: codes within one step of the oracle chain's on nearly all elements (a bf16 step of a
    # GEMM result moves a code at most one step; scales move only where a block maximum crosses a power of two)
    deq = orc.mx_dequant_rows(a2.cpu().numpy(), sa2.cpu().numpy(), h, orc.E4M3)
    deq_o = orc.mx_dequant_rows(a2_o, sa2_o, h, orc.E4M3)
    m1 = orc.compare(deq, deq_o)
    assert m1["max_rel_floor_rms"] <= 0.15 and np.mean(sa2.cpu().numpy() == sa2_o) > 0.995, m1
    assert np.mean(a2.cpu().numpy() == a2_o) > 0.97
    # GMM2 and the un-permute, given the device's own quantised activation: the GEMM gate
    _, y_d = orc.mx_gmm(a2.cpu().numpy(), sa2.cpu().numpy(), b2, sb2, k, h, orc.E4M3, 1, group_sizes=cnt_o, want_bf16=True)
    m2 = orc.compare(y.float().cpu().numpy(), orc.bf16_to_f32(y_d))
    assert m2["max_rel_floor1"] <= 1e-2 and m2["max_rel_floor_rms"] <= 1e-2 and abs(m2["eb"]) <= 2.0 ** -7, m2
    assert np.array_equal(bits(out), orc.moe_token_unpermute(bits(y), s2d_o, probs, topk))
    # the chain's output against the all-oracle chain: a code of the quantised activation that lands one E4M3 step
    # away (3 % of them do, above) moves an output by a few tenths of a percent of the tensor's rms, so the two chains
    # agree to about 1 % rms and a few percent at the worst element - what any two implementations of this chain do
    got, want = out.float().cpu().numpy(), orc.bf16_to_f32(out_o)
    rms = np.sqrt(np.mean(want ** 2))
    assert np.sqrt(np.mean((got - want) ** 2)) <= 2e-2 * rms and np.abs(got - want).max() <= 0.12 * rms


def test_ffn_takes_up_projections_of_any_one_byte_type():
    """The up projection's payload and scales are bytes whatever their element type is called, as in mx_grouped_matmul_swiglu_packed."""
    m, k, n, e = 20, 128, 128, 3
    g = torch.Generator(device="cuda").manual_seed(9)
    x, idx = torch.randn(m, k, device="cuda", generator=g).bfloat16(), torch.randint(0, e, (m, 2), device="cuda", generator=g, dtype=torch.int32)
    probs = torch.rand(m, 2, device="cuda", generator=g)
    w1, sw1, w2, sw2 = (torch.stack([cc.mx_quant(torch.randn(r, c, device="cuda", generator=g).bfloat16())[i] for _ in range(e)])
                        for r, c in ((n, k), (k, n // 2)) for i in (0, 1))
    want = cc.moe_ffn_mxfp8(x, idx, probs, w1, sw1, w2, sw2)
    got = cc.moe_ffn_mxfp8(x, idx, probs, w1.view(torch.float8_e4m3fn), sw1.view(torch.int8), w2, sw2)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    with pytest.raises(ValueError, match="uint8"):
        cc.moe_ffn_mxfp8(x, idx, probs, w1, sw1, w2.view(torch.int8), sw2)


@pytest.mark.parametrize("n,k,note", [
    (96, 128, "MX-quantised output"),     # the up projection alone: 48 columns are no whole MX blocks
    (128, 132, "16-byte stores"),         # both: K of the up projection, and columns of the down projection, whose note is the later one
    (128, 128, ""),
])
def test_ffn_reports_a_projection_on_the_generic_kernels(n, k, note):
    """cch_last_error() names the precondition when either projection of the call ran on the one-thread-per-element kernels, and nothing of older calls."""
    L = cc._abi.lib()
    m, e, h = 8, 2, n // 2
    g = torch.Generator(device="cuda").manual_seed(n + k)
    x, idx = torch.randn(m, k, device="cuda", generator=g).bfloat16(), torch.randint(0, e, (m, 2), device="cuda", generator=g, dtype=torch.int32)
    probs = torch.rand(m, 2, device="cuda", generator=g)
    w1, sw1, w2, sw2 = (torch.stack([cc.mx_quant(torch.randn(r, c, device="cuda", generator=g).bfloat16())[i] for _ in range(e)])
                        for r, c in ((n, k), (k, h)) for i in (0, 1))
    cc.mx_matmul(*cc.mx_quant(torch.randn(4, 40, device="cuda").bfloat16()), *cc.mx_quant(torch.randn(16, 40, device="cuda").bfloat16()), trans_b=1)
    assert b"generic" in L.cch_last_error() or b"note" in L.cch_last_error()
    cc.moe_ffn_mxfp8(x[:0], idx[:0], probs[:0], w1, sw1, w2, sw2)     # no tokens: nothing ran, and no note of the call before is left
    assert L.cch_last_error() == b""
    out = cc.moe_ffn_mxfp8(x, idx, probs, w1, sw1, w2, sw2)
    got = L.cch_last_error().decode()
    assert torch.isfinite(out.float()).all() and (note in got if note else got == ""), got


@pytest.mark.parametrize("m,k,n,e,topk,dropped", [
    (1, 64, 128, 1, 1, False),         # one route, one piece of one pair of blocks
    (37, 960, 256, 3, 2, True),        # K an odd multiple of 64, dropped entries of either sign
    (129, 1984, 128, 8, 8, True),      # 1032 routes: two groups of keys per wave; eight tokens per workgroup
    (300, 1088, 256, 256, 7, False),   # 2100 routes, as many experts as one launch takes
    (515, 512, 128, 5, 8, True),       # 4120 routes, sixteen tokens and all 128 route places of a workgroup
    (1024, 64, 128, 4, 8, False),      # 8192 routes: the most that one launch takes
    (1025, 192, 128, 4, 8, True),      # one token more: the sort's own launches
    (8192, 64, 128, 5, 1, True),       # 8192 routes to one expert each
    (5016, 4160, 128, 5, 1, True),     # 1672 workgroups of three tokens of five pieces look at 5016 routes: 2^23 in all but for some
    (5019, 4160, 128, 5, 1, True),     # and 1673 at 5019, more: two launches
    (70, 2048, 1024, 96, 4, True),     # more weights than the caches hold: rows of whole pieces are stored with the non-temporal hint
    (70, 1984, 1024, 96, 4, True),     # and of partial ones
    (5, 17472, 128, 2, 2, False),      # 18 pieces a token, more than a workgroup's waves
    (6, 512, 128, 257, 3, True),       # more experts than MAX: refused
])
def test_whole_ffn_is_its_stages(m, k, n, e, topk, dropped):
    """moe_ffn_mxfp8 against its stages called one by one on rows that were gathered instead of scattered: the same bytes."""
    g = torch.Generator(device="cuda").manual_seed(m + k + e)
    x = (torch.randn(m, k, device="cuda", generator=g) * 2).bfloat16()
    idx = torch.randint(-2 if dropped else 0, e + (3 if dropped else 0), (m, topk), device="cuda", generator=g, dtype=torch.int32)
    probs = torch.rand(m, topk, device="cuda", generator=g)
    w1 = [cc.mx_quant_b(torch.randn(k, n, device="cuda", generator=g).bfloat16() * k ** -0.5, trans_b=1) for _ in range(min(e, 8))]
    w2 = [cc.mx_quant_b(torch.randn(n // 2, k, device="cuda", generator=g).bfloat16() * n ** -0.5, trans_b=1) for _ in range(min(e, 8))]
    w1, sw1, w2, sw2 = (torch.stack([w[i % len(w)][h] for i in range(e)]) for w in (w1, w2) for h in (0, 1))
    if e > 256:
        with pytest.raises(cc.CatccosError, match="num_experts"):
            cc.moe_ffn_mxfp8(x, idx, probs, w1, sw1, w2, sw2)
        return
    d2s, s2d, cnt = cc.moe_init_routing(idx, e)
    a, sa = cc.mx_quant(x)
    token = (d2s.clamp(min=0) // topk).long()
    cc.set_option("require_tiled_gemm", 1)
    try:
        out = cc.moe_ffn_mxfp8(x, idx, probs, w1, sw1, w2, sw2)
        act, act_scales = cc.mx_grouped_matmul_swiglu(a[token], sa[token], w1, sw1, cnt, "e4m3", 1, out_fmt="e4m3")
        y = cc.mx_grouped_matmul(act, act_scales, w2, sw2, cnt, "e4m3", 1)
    finally:
        cc.set_option("require_tiled_gemm", 0)
    want = cc.moe_token_unpermute(y, s2d, probs, topk)
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert torch.isfinite(want.float()).all() and want.float().abs().max() > 0
