"""The work whose speed this repository answers for: what a serving program has this package do, through its tensor-level
entry points, from one decode step to a long prefill.

Six kinds of pass, each written as a user's program writes it:

    quant      MX quantisation of an activation tensor on its own (what a rank sends instead of bf16)
    mx_linear  a linear layer with MX weights: quantise the activations, multiply
    w8a8       a linear layer with int8 weights: per-token dynamic quantisation, multiply, dequantise
    moe_ffn    the MXFP8 mixture-of-experts feed-forward, routing to combine
    moe_w8a8   the int8 expert up projection: routing, gather + quantise, grouped matmul + dequant + SwiGLU
    mx_gmm     the grouped matmul over tokens that arrived quantised and sorted by expert

Token counts are whatever the batch holds (odd as a rule); the sizes of the layers are those of this repository's
configurations and shape lists, and in draw() others of the same kind.  Weights are quantised once, as a program does when it
loads them; the layouts are the two that the entry points take (trans_b = 0: [K, N], 1: [N, K])."""
import math

import numpy as np
import torch

import catccos_amd as cc


def listed():
    return [
        # a decode step's activations (64 sequences) on their way to the other ranks: the smallest call there is
        {"name": "quant-decode", "kind": "quant", "m": 64, "k": 7168, "fmt": "e4m3", "half": False},
        # a prefill chunk's activations
        {"name": "quant-prefill", "kind": "quant", "m": 4096, "k": 7168, "fmt": "e4m3", "half": False},
        # one decode step of 16 sequences through a dense MXFP8 layer (the weights of the prefill case below)
        {"name": "mx-linear-decode", "kind": "mx_linear", "m": 16, "k": 2048, "n": 7168, "fmt": "e4m3", "trans_b": 0, "half": False},
        # a layer none of whose sizes is a power of two, with [N, K] weights and half output: the shape list's largest
        {"name": "mx-linear-ragged", "kind": "mx_linear", "m": 3000, "k": 1984, "n": 3000, "fmt": "e4m3", "trans_b": 1, "half": True},
        # a prefill chunk through the dense MXFP8 layer
        {"name": "mx-linear-prefill", "kind": "mx_linear", "m": 4096, "k": 2048, "n": 7168, "fmt": "e4m3", "trans_b": 0, "half": False},
        # a decode step of 64 sequences through a dense int8 layer, [N, K] weights
        {"name": "w8a8-decode", "kind": "w8a8", "m": 64, "k": 4096, "n": 8192, "trans_b": 1, "half": False},
        # a long prefill through the same layer, [K, N] weights
        {"name": "w8a8-prefill", "kind": "w8a8", "m": 8192, "k": 4096, "n": 8192, "trans_b": 0, "half": False},
        # the mixture-of-experts block at a decode step of 64 sequences, 6 of 16 experts each
        {"name": "moe-ffn-decode", "kind": "moe_ffn", "m": 64, "k": 7168, "n": 4096, "e": 16, "top_k": 6, "trans_b": 1},
        # the same block with 512 tokens: the largest size of its own shape list
        {"name": "moe-ffn-512", "kind": "moe_ffn", "m": 512, "k": 7168, "n": 4096, "e": 16, "top_k": 6, "trans_b": 1},
        # the int8 expert up projection for 4096 tokens, 2 of 16 experts each, skewed
        {"name": "moe-w8a8-up", "kind": "moe_w8a8", "m": 4096, "k": 7168, "n": 4096, "e": 16, "top_k": 2, "trans_b": 0},
        # 16384 received tokens over 32 local experts, Zipf-sized groups, MXFP4 and MXFP8
        {"name": "mx-gmm-fp4", "kind": "mx_gmm", "m": 16384, "k": 7168, "n": 4096, "e": 32, "fmt": "e2m1", "trans_b": 0},
        {"name": "mx-gmm-fp8", "kind": "mx_gmm", "m": 16384, "k": 7168, "n": 4096, "e": 32, "fmt": "e4m3", "trans_b": 0},
    ]


def _log(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dim(rng, lo, hi, unit):
    """A layer's size: half of them a multiple of 1024 (where the range has one), the others a multiple of 128 or of `unit`."""
    v = _log(rng, lo, hi)
    u = rng.choice([1024, 1024, 128, unit])
    return max(v // u * u, lo if u > v else u)


_FLOPS, _WEIGHTS = 9.0e11, 0.9e9   # no drawn case is larger than mx-gmm-fp8


def draw(rng):
    while True:
        kind = rng.choice(["quant", "mx_linear", "mx_linear", "w8a8", "moe_ffn", "moe_ffn", "moe_w8a8", "mx_gmm", "mx_gmm"])
        c = {"kind": kind}
        if kind == "quant":
            c.update(m=_log(rng, 1, 16384), k=_dim(rng, 512, 8192, 32), fmt=rng.choice(["e4m3", "e4m3", "e5m2", "e2m1"]), half=rng.random() < 0.25)
            if c["m"] * c["k"] <= 1 << 26:
                return c
            continue
        c.update(m=_log(rng, 1, 16384), k=_dim(rng, 512, 8192, 64), n=_dim(rng, 512, 8192, 8))
        if kind in ("mx_linear", "mx_gmm"):
            c["fmt"] = rng.choice(["e4m3", "e4m3", "e2m1", "e5m2"])
        if kind in ("mx_linear", "w8a8"):
            c["half"] = rng.random() < 0.25
            e = rows = 1
        else:
            e = c["e"] = rng.choice([4, 8, 16, 32, 64])
            rows = 1
        if kind in ("moe_ffn", "moe_w8a8"):
            c["n"] = max(512, c["n"] // 64 * 64)          # gate and up halves, each a whole number of MX blocks
            c["top_k"] = rows = rng.choice([t for t in (1, 2, 4, 6, 8) if t <= c["e"]])
        if kind == "moe_ffn":
            c["n"] = max(512, c["n"] // 128 * 128)        # the down projection's K
        c["trans_b"] = rng.choice([0, 1])
        if kind not in ("w8a8", "moe_w8a8") and (c["k"] % 128 or (kind == "moe_ffn" and c["n"] % 256)):
            # Scale rows of an odd number of byte pairs: with an odd number of rows the last row's last scales were dropped
            # when this file was written, so that such a pass has no earlier result to be compared with.
            c["m"] += c["m"] % 2
        up = 1.5 if kind == "moe_ffn" else 1.0
        if 2.0 * c["m"] * rows * c["k"] * c["n"] * up <= _FLOPS and 1.0 * e * c["k"] * c["n"] * up <= _WEIGHTS:
            return c


def _weights(gen, e, k, n, fmt, trans_b):
    """MX weights of e matrices [k, n] of variance 1/k, quantised down K: payload and scales, stacked."""
    ws = [cc.mx_quant_b((torch.randn(k, n, device="cuda", generator=gen) * k ** -0.5).to(torch.bfloat16), fmt, trans_b=trans_b) for _ in range(e)]
    return torch.stack([w[0] for w in ws]), torch.stack([w[1] for w in ws])


def _activations(gen, m, k, dtype=torch.bfloat16):
    """Activations as a normalisation leaves them: unit variance, a few channels an order of magnitude larger."""
    gain = torch.exp(0.5 * torch.randn(k, device="cuda", generator=gen))
    return (torch.randn(m, k, device="cuda", generator=gen) * gain).to(dtype)


def _routes(gen, m, e, top_k, skew):
    """Each token's top_k distinct experts, drawn with probabilities ~ rank^-skew over shuffled experts."""
    rank = torch.randperm(e, device="cuda", generator=gen) + 1
    u = torch.rand(m, e, device="cuda", generator=gen).clamp_(1e-6, 1 - 1e-6)
    score = -skew * torch.log(rank.float()) - torch.log(-torch.log(u))
    return score.topk(top_k, dim=1).indices.to(torch.int32).contiguous()


def _groups(seed, t, e):
    """Rows per expert: multinomial over shuffled Zipf(1.1) shares, one expert with none."""
    rng = np.random.default_rng(seed)
    p = (np.arange(e) + 1.0) ** -1.1
    gs = rng.multinomial(t, rng.permutation(p / p.sum())).astype(np.int32)
    i, j = int(gs.argmin()), int(gs.argmax())
    if gs[i] > 0:
        gs[j] += gs[i]
        gs[i] = 0
    return torch.from_numpy(gs).cuda()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    c = dict(case)
    kind, m, k = c["kind"], c["m"], c["k"]
    s = {"case": c, "kind": kind}
    if kind == "quant":
        s["x"] = _activations(gen, m, k, torch.float16 if c["half"] else torch.bfloat16)
        return s
    n, tb = c["n"], c["trans_b"] if "trans_b" in c else 0
    s["out_dtype"] = torch.float16 if c.get("half") else torch.bfloat16
    if kind == "mx_linear":
        b, sb = _weights(gen, 1, k, n, c["fmt"], tb)
        s.update(x=_activations(gen, m, k), b=b[0], sb=sb[0])
    elif kind == "w8a8":
        shape = (n, k) if tb else (k, n)
        s.update(x=_activations(gen, m, k), b=torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=gen),
                 per_ch=(torch.rand(n, device="cuda", generator=gen) + 0.5) / (73.0 * k ** 0.5))
    elif kind == "moe_ffn":
        e, h = c["e"], n // 2
        s["w1"], s["sw1"] = _weights(gen, e, k, n, "e4m3", tb)
        s["w2"], s["sw2"] = _weights(gen, e, h, k, "e4m3", tb)
        s.update(x=_activations(gen, m, k), idx=_routes(gen, m, e, c["top_k"], 0.5),
                 probs=torch.softmax(torch.randn(m, c["top_k"], device="cuda", generator=gen), dim=1))
    elif kind == "moe_w8a8":
        e = c["e"]
        shape = (e, n, k) if tb else (e, k, n)
        s.update(x=_activations(gen, m, k), idx=_routes(gen, m, e, c["top_k"], 1.1),
                 w=torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=gen),
                 per_ch=(torch.rand(e, n, device="cuda", generator=gen) + 0.5) / (73.0 * k ** 0.5))
    else:
        s["b"], s["sb"] = _weights(gen, c["e"], k, n, c["fmt"], tb)
        s["a"], s["sa"] = cc.mx_quant(_activations(gen, m, k), c["fmt"])
        s["groups"] = _groups(seed, m, c["e"])
    return s


def run(s):
    c, kind = s["case"], s["kind"]
    if kind == "quant":
        return cc.mx_quant(s["x"], c["fmt"])
    if kind == "mx_linear":
        a, sa = cc.mx_quant(s["x"], c["fmt"])
        return cc.mx_matmul(a, sa, s["b"], s["sb"], c["fmt"], c["trans_b"], s["out_dtype"])
    if kind == "w8a8":
        q, per_tok = cc.dynamic_quant_i8(s["x"])
        return cc.w8a8_matmul_dequant(q, s["b"], per_tok, s["per_ch"], c["trans_b"], s["out_dtype"])
    if kind == "moe_ffn":
        return cc.moe_ffn_mxfp8(s["x"], s["idx"], s["probs"], s["w1"], s["sw1"], s["w2"], s["sw2"], c["trans_b"])
    if kind == "moe_w8a8":
        d2s, s2d, cnt = cc.moe_init_routing(s["idx"], c["e"])
        q, per_tok = cc.dynamic_quant_i8(s["x"], d2s, c["top_k"])
        out = cc.gmm_dequant_swiglu(q, s["w"], cnt, per_tok, s["per_ch"], c["trans_b"])
        return out, s2d, cnt
    return cc.mx_grouped_matmul(s["a"], s["sa"], s["b"], s["sb"], s["groups"], c["fmt"], c["trans_b"])


def _mx_bytes(elements, fmt):
    return elements * (0.5 if fmt == "e2m1" else 1.0) + elements / 32.0


def work(case):
    kind, m, k = case["kind"], case["m"], case["k"]
    if kind == "quant":
        return {"bytes": 2.0 * m * k + _mx_bytes(m * k, case["fmt"]), "flops": 0.0}
    n = case["n"]
    if kind == "mx_linear":
        return {"bytes": 2.0 * m * (k + n) + _mx_bytes(k * n, case["fmt"]), "flops": 2.0 * m * k * n}
    if kind == "w8a8":
        return {"bytes": 2.0 * m * (k + n) + k * n + 4.0 * n, "flops": 2.0 * m * k * n}
    e = case["e"]
    if kind == "mx_gmm":
        # every expert but the empty one is read (or as many as there are rows)
        return {"bytes": _mx_bytes(m * k + min(e - 1, m) * k * n, case["fmt"]) + 2.0 * m * n, "flops": 2.0 * m * k * n}
    rows = m * case["top_k"]
    used = e * (1.0 - (1.0 - case["top_k"] / e) ** m)      # experts that some token names, were all equally likely
    if kind == "moe_ffn":
        return {"bytes": 4.0 * m * k + 8.0 * rows + _mx_bytes(used * 1.5 * k * n, "e4m3"), "flops": 3.0 * rows * k * n}
    return {"bytes": 2.0 * m * k + 8.0 * rows + used * (k * n + 4.0 * n) + 1.0 * rows * n, "flops": 2.0 * rows * k * n}


def tolerance(case):
    """Four times what the path differs from the same pass in 64 bits: the rounding of its output, once, is all of that."""
    kind = case["kind"]
    if kind == "quant":
        return "exact"                                   # bytes
    if kind == "moe_ffn":
        # a sum that falls on the other side of a bf16 step between the two products moves a code of the quantised
        # activation: 0.2 % of the result's size in all, 5 % at the worst element
        return {"rel": 8.5e-3, "max": 0.2}
    if case.get("half"):
        return {"rel": 8.5e-4, "max": 2.4e-3}            # measured 2.1e-4 and 5.8e-4
    return {"rel": 6.6e-3, "max": 1.6e-2}                # measured 1.66e-3 and 3.9e-3
