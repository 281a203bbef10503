"""The native forms of the entry points (csrc/torch/direct_calls.cpp) against the general path they stand in front of: the same
outputs for every form that the entry points accept, the same errors for what they refuse, and no effect where they decline."""
import pytest
import torch

import catccos_amd as cc
from catccos_amd import ops


class _Declines:
    def __getattr__(self, name):
        return lambda *a: NotImplemented


def _names():
    return ["mx_quant", "dynamic_quant_i8", "moe_init_routing", "w8a8_matmul_dequant", "gmm_i8", "mx_matmul", "mx_grouped_matmul", "moe_ffn_mxfp8"]


def test_host_tensors_and_odd_arguments_are_declined():
    x = torch.zeros(2, 64, dtype=torch.bfloat16)
    for name in _names():
        f = getattr(ops._direct, name)
        for args in ((), (x,), (x, "e4m3", 0), (x, None, 1, 0), (x, 4, False), (x, x, x, x, 0, torch.bfloat16), (None,) * 7, (x,) * 8, (1, 2, 3)):
            assert f(*args) is NotImplemented
    with pytest.raises(ValueError):
        cc.mx_quant(x)


def _without_module(monkeypatch):
    def fails(name, package=None):
        raise ImportError("libtorch_python.so: cannot open shared object file")
    monkeypatch.setattr(ops._importlib, "import_module", fails)
    monkeypatch.setattr(ops, "_direct", ops._Direct())


def test_host_tensors_are_refused_as_such_without_the_native_module(monkeypatch):
    _without_module(monkeypatch)
    with pytest.warns(RuntimeWarning, match="does not load"):
        with pytest.raises(ValueError, match="GPU tensors only"):
            cc.mx_quant(torch.zeros(2, 64, dtype=torch.bfloat16))


@pytest.mark.gpu
def test_calls_are_served_without_the_native_module(monkeypatch):
    calls = _calls()
    want = [_flat(f(*a, **kw)) for f, a, kw in calls]
    _without_module(monkeypatch)
    with pytest.warns(RuntimeWarning, match="does not load"):
        got = [_flat(f(*a, **kw)) for f, a, kw in calls]
    for w, g in zip(want, got):
        for x, y in zip(w, g):
            assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))


def _calls(dev="cuda"):
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    m, k, n, e = 37, 256, 512, 4
    x = torch.randn(m, k, device=dev, generator=g).bfloat16()
    idx = torch.randint(0, e, (m, 2), device=dev, generator=g, dtype=torch.int32)
    probs = torch.rand(m, 2, device=dev, generator=g)
    gs = torch.tensor([10, 0, 20, 5], dtype=torch.int32, device=dev)
    out = []
    for fmt in ("e4m3", "e5m2", "e2m1", cc.FMT_E4M3, "fp8", "E4M3"):
        out.append((cc.mx_quant, (x, fmt), {}))
        out.append((cc.mx_quant, (x.half(), fmt, cc.ROUND_LUT), {}))
        a, sa = cc.mx_quant(x, fmt)
        for tb in (0, 1, False, True):
            w = [cc.mx_quant_b(torch.randn(k, n, device=dev, generator=g).bfloat16(), fmt, trans_b=tb) for _ in range(e)]
            b, sb = torch.stack([v[0] for v in w]), torch.stack([v[1] for v in w])
            for dt in (torch.bfloat16, torch.float16):
                out.append((cc.mx_matmul, (a, sa, b[0], sb[0], fmt, tb, dt), {}))
                out.append((cc.mx_grouped_matmul, (a, sa, b, sb, gs, fmt, tb), {"out_dtype": dt}))
    for mode in (cc.DQ_DEVICE, cc.DQ_GOLDEN):
        out.append((cc.dynamic_quant_i8, (x,), {"mode": mode}))
        out.append((cc.dynamic_quant_i8, (x, idx.reshape(-1), 2, mode), {}))
    for cumsum in (False, True):
        out.append((cc.moe_init_routing, (idx, e, cumsum), {}))
    out.append((cc.moe_init_routing, (torch.randint(0, e, (40000,), device=dev, generator=g, dtype=torch.int32), e), {}))
    q, pt = cc.dynamic_quant_i8(x)
    for tb in (0, 1):
        wi = torch.randint(-127, 128, (e, n, k) if tb else (e, k, n), dtype=torch.int8, device=dev, generator=g)
        pc = torch.rand(e, n, device=dev, generator=g) * 1e-3
        for dt in (torch.bfloat16, torch.float16):
            out.append((cc.w8a8_matmul_dequant, (q, wi[0], pt, pc[0], tb, dt), {}))
            out.append((cc.gmm_dequant, (q, wi, gs, pt, pc, tb, dt), {}))
            out.append((cc.gmm_dequant_swiglu, (q, wi, gs, pt, pc, tb, dt), {}))
        w1 = [cc.mx_quant_b(torch.randn(k, n, device=dev, generator=g).bfloat16(), trans_b=tb) for _ in range(e)]
        w2 = [cc.mx_quant_b(torch.randn(n // 2, k, device=dev, generator=g).bfloat16(), trans_b=tb) for _ in range(e)]
        out.append((cc.moe_ffn_mxfp8, (x, idx, probs) + tuple(torch.stack([v[i] for v in w]) for w in (w1, w2) for i in (0, 1)) + (tb,), {}))
    return out


def _flat(r):
    return r if isinstance(r, tuple) else (r,)


def _strided(t):
    """The same values with other strides (every second column of a wider tensor)."""
    if not isinstance(t, torch.Tensor) or t.dim() == 0:
        return t
    wide = torch.zeros(t.shape[:-1] + (2 * t.shape[-1],), dtype=t.dtype, device=t.device)
    wide[..., ::2] = t
    return wide[..., ::2]


@pytest.mark.gpu
def test_native_and_general_forms_give_the_same(monkeypatch):
    calls = _calls()
    native = [_flat(f(*a, **kw)) for f, a, kw in calls]
    strided = [_flat(f(*[_strided(v) for v in a], **kw)) for f, a, kw in calls]
    with torch.inference_mode():
        inference = [_flat(f(*a, **kw)) for f, a, kw in calls]
    monkeypatch.setattr(ops, "_direct", _Declines())
    for (f, a, kw), nat, st, inf in zip(calls, native, strided, inference):
        want = _flat(f(*a, **kw))
        for got in (nat, st, inf):
            assert len(got) == len(want)
            for x, y in zip(got, want):
                assert x.dtype == y.dtype and x.shape == y.shape and x.is_contiguous() and not x.requires_grad
                assert x.untyped_storage().nbytes() == y.untyped_storage().nbytes()
                # (rows past the groups are zeros; NaN compares by its bytes)
                assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)), f.__name__


@pytest.mark.gpu
def test_plain_calls_take_the_native_form(monkeypatch):
    calls, took = _calls(), []
    native = ops._direct

    class Counts:
        def __getattr__(self, name):
            def f(*a):
                r = getattr(native, name)(*a)
                took.append((name, r is not NotImplemented))
                return r
            return f
    monkeypatch.setattr(ops, "_direct", Counts())
    for f, a, kw in calls:
        del took[:]
        f(*a, **kw)
        assert took and took[0][1] == (not any(isinstance(v, str) and v in ("fp8", "E4M3") for v in a)), f.__name__


@pytest.mark.gpu
def test_what_was_refused_stays_refused(monkeypatch):
    bad = []
    for f, a, kw in _calls()[::3]:
        for i, v in enumerate(a):
            if isinstance(v, torch.Tensor):
                for other in (v.cpu(), v[:0], v.to(torch.float64), v[None], torch.cat([v, v[:1]]), None):
                    bad.append((f, a[:i] + (other,) + a[i + 1:], kw))
            else:
                bad.append((f, a[:i] + ("nonsense",) + a[i + 1:], kw))

    def outcome(f, a, kw):
        try:
            return [tuple(t.shape) for t in _flat(f(*a, **kw))]
        except Exception as e:
            return type(e), str(e)
    # (a route table longer or shorter than the rows, group sizes past them and the like stay calls the kernels are made for)
    got = [outcome(*c) for c in bad]
    monkeypatch.setattr(ops, "_direct", _Declines())
    for c, g in zip(bad, got):
        assert outcome(*c) == g, c[0].__name__


@pytest.mark.gpu
def test_on_another_stream_and_in_a_graph():
    calls = _calls()[:12]
    want = [_flat(f(*a, **kw)) for f, a, kw in calls]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = [_flat(f(*a, **kw)) for f, a, kw in calls]
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = [_flat(f(*a, **kw)) for f, a, kw in calls]
    for _ in range(3):
        for h in held:
            for t in h:
                t.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for w, g, h in zip(want, got, held):
            for x, y, z in zip(w, g, h):
                assert torch.equal(x.view(torch.uint8), y.view(torch.uint8)) and torch.equal(x.view(torch.uint8), z.view(torch.uint8))
