"""f3s_linear_f16 at the edges of its tiles against float64: every output
within one rounding to binary16 (2^-11 of it, or half the smallest subnormal)
plus the float32 sum's error bound, K * 2^-24 * sum |x w|; and the layer's use
of it, which leaves hooked or subclassed projections to their own call."""
from __future__ import annotations

import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,M,bias", [
    (1, 8, 32, True), (15, 64, 96, False), (16, 72, 192, True), (17, 128, 416, True),
    (65, 136, 64, True), (1000, 256, 1536, False), (333, 120, 2048, True),
    (65535, 128, 192, True), (65536, 128, 384, True), (65553, 64, 800, False),
    (70001, 256, 416, True), (49151, 96, 224, True), (49152, 96, 224, False),   # 4 and 16 waves
    (33, 64, 2080, True), (5, 8, 12_320, False), (17, 256, 32_768, True), (49_160, 40, 4128, True),
])
def test_linear(gpu, n, K, M, bias):
    from fused3s_amd import _lib
    gen = torch.Generator(device="cuda").manual_seed(n + K + M)
    rand = lambda *s: torch.randn(*s, generator=gen, device="cuda", dtype=torch.float32)
    x, w = rand(n, K).half(), (rand(M, K) * 0.2).half()
    b = rand(M).half() if bias else None
    y = torch.full((n + 1, M), 7.0, dtype=torch.float16, device="cuda")   # one row past the end
    status = _lib.hip().f3s_linear_f16(x.data_ptr(), w.data_ptr(), b.data_ptr() if bias else None,
                                       y.data_ptr(), n, K, M,
                                       torch.cuda.current_stream().cuda_stream)
    assert status == 0
    assert (y[n] == 7.0).all()
    want = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    size = x.double().abs() @ w.double().abs().t() + (b.double().abs() if bias else 0.0)
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -25 + size * ((K + 1) * 2.0 ** -24)
    assert bool(((y[:n].double() - want).abs() <= bound).all())


def test_linear_rejects(gpu):
    from fused3s_amd import _lib
    x = torch.zeros(64, 256, dtype=torch.float16, device="cuda")
    f = _lib.hip().f3s_linear_f16
    assert f(x.data_ptr(), x.data_ptr(), None, x.data_ptr(), 4, 12, 32, None) == 5
    assert f(x.data_ptr(), x.data_ptr(), None, x.data_ptr(), 4, 264, 32, None) == 5
    assert f(x.data_ptr(), x.data_ptr(), None, x.data_ptr(), 4, 64, 48, None) == 5
    assert f(x.data_ptr() + 2, x.data_ptr(), None, x.data_ptr(), 4, 64, 32, None) == 1
    assert f(None, x.data_ptr(), None, x.data_ptr(), 4, 64, 32, None) == 1
    assert f(None, None, None, None, 0, 64, 32, None) == 0


def test_layer_projections(gpu):
    from fused3s_amd import torch_ops
    rp, ci = random_csr(700, 6, 4)
    graph = torch_ops.TorchGraph(rp, ci, heads=2)
    torch.manual_seed(1)
    layer = torch_ops.GraphTransformerLayer(96, heads=2).cuda().half()
    x = torch.randn(700, 96, device="cuda").half()
    y = layer(x, graph)
    seen = []
    hooks = [m.register_forward_hook(lambda *a: seen.append(1)) for m in (layer.qkv, layer.proj)]
    z = layer(x, graph)              # hooked: torch's own product
    assert len(seen) == 2
    for h in hooks:
        h.remove()
    assert (y - z).abs().max() <= 2e-3 * z.abs().max()
    assert len(seen) == 2 and torch.equal(layer(x, graph), y) and len(seen) == 2
    odd = torch_ops.GraphTransformerLayer(100, heads=2, out_dim=40).cuda().half()   # K % 8, M % 32
    assert odd(torch.randn(700, 100, device="cuda").half(), graph).shape == (700, 40)
    wide = torch_ops.GraphTransformerLayer(96, heads=2).cuda()                      # float32 module
    assert wide(x.float(), graph).dtype == torch.float32


def test_layer_yields_to_overrides(gpu):
    """A dispatch mode sees the layer's products, and a graph that brings its
    own attention has it called."""
    from torch.utils.flop_counter import FlopCounterMode

    from fused3s_amd import torch_ops
    rp, ci = random_csr(100, 4, 3)
    graph = torch_ops.TorchGraph(rp, ci, heads=1)
    layer = torch_ops.GraphTransformerLayer(64, heads=1).cuda().half()
    x = torch.randn(100, 64, dtype=torch.float16, device="cuda")
    with FlopCounterMode(display=False) as counter:
        layer(x, graph)
    assert counter.get_total_flops() == 2 * 100 * 64 * (192 + 64)

    calls = []

    class Own(torch_ops.TorchGraph):
        def attention(self, *args, **kwargs):
            calls.append(1)
            return super().attention(*args, **kwargs)

    layer(x, Own(rp, ci, heads=1))
    assert calls


def test_layer_calls_a_replaced_attention(gpu, monkeypatch):
    """One assigned on a graph, and one assigned on TorchGraph itself."""
    from fused3s_amd import torch_ops
    rp, ci = random_csr(100, 4, 3)
    graph = torch_ops.TorchGraph(rp, ci, heads=1)
    layer = torch_ops.GraphTransformerLayer(64, heads=1).cuda().half()
    x = torch.randn(100, 64, dtype=torch.float16, device="cuda")
    calls = []
    attention = torch_ops.TorchGraph.attention

    def own(self, *args, **kwargs):
        calls.append(1)
        return attention(self, *args, **kwargs)

    graph.attention = own.__get__(graph)
    layer(x, graph)
    assert len(calls) == 1
    del graph.attention
    monkeypatch.setattr(torch_ops.TorchGraph, "attention", own)
    layer(x, graph)
    assert len(calls) == 2


class _OwnAttention:
    """A program's own attention in the place of a TorchGraph: each node's v."""

    heads = 1

    def attention(self, q, k, v, scale=1.0):
        return v.float()


def test_layer_yields_to_watchers(gpu):
    """The layer's products are torch's own where a function mode, a functorch
    transform, forward-mode differentiation or a replaced torch.nn.functional.
    linear is there to see them."""
    import torch.autograd.forward_ad as forward_ad
    from torch.overrides import TorchFunctionMode

    from fused3s_amd import torch_ops
    layer = torch_ops.GraphTransformerLayer(64, heads=1).cuda().half()
    graph = _OwnAttention()
    x = torch.randn(100, 64, dtype=torch.float16, device="cuda")
    own = layer(x, graph)
    seen = []

    class Count(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Count():
        y = layer(x, graph)
    assert seen.count(torch.nn.functional.linear) == 2
    bound = 2e-3 * own.abs().max()
    assert (y - own).abs().max() <= bound

    with torch.device("cuda"):   # a function mode too, but it sees no products
        assert torch.equal(layer(x, graph), own)

    z = torch.func.vmap(lambda t: layer(t, graph))(torch.stack([x, -x]))
    assert (z[0] - own).abs().max() <= bound

    with forward_ad.dual_level():
        dual = layer(forward_ad.make_dual(x, x), graph)
        tangent = forward_ad.unpack_dual(dual).tangent
    assert tangent is not None   # the layer is affine here: J x = f(x) - f(0)
    assert (tangent - (own - layer(torch.zeros_like(x), graph))).abs().max() <= 2 * bound

    product = torch.nn.functional.linear
    calls = []
    torch.nn.functional.linear = lambda *a: calls.append(1) or product(*a)
    try:
        layer(x, graph)
    finally:
        torch.nn.functional.linear = product
    assert len(calls) == 2
