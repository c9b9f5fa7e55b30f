"""f3s_attention_fwd_packed: the compiled plan's pass on one [n][3][H][64]
tensor gives the bits of the planned pass on copies of its thirds (float32),
and those rounded once (binary16), for every launch shape of a masked plan:
teams, one-wave workgroups, four-wave workgroups and split windows."""
from __future__ import annotations

import numpy as np
import pytest
import torch  # noqa: F401  (torch's HIP runtime first)

from conftest import random_csr, rng

pytestmark = pytest.mark.gpu


def star_csr(n: int, hubs: int, seed: int):
    r = rng(seed)
    rows = np.concatenate([np.repeat(np.arange(hubs), n // 2), np.arange(n)])
    cols = np.concatenate([r.integers(0, n, hubs * (n // 2)), np.arange(n)])
    keys = np.unique(rows.astype(np.int64) * n + cols)
    rp = np.searchsorted(keys // n, np.arange(n + 1)).astype(np.int32)
    return rp, (keys % n).astype(np.int32)


@pytest.mark.parametrize("graph,n,H", [
    ("random", 1, 1), ("random", 45, 3), ("random", 3000, 1),   # teams
    ("random", 17_001, 1), ("random", 20_000, 5),               # one- and four-wave workgroups
    ("star", 30_000, 2),                                        # split windows
    ("random", 700, 64),                                        # the most heads
])
def test_packed_is_planned(gpu, graph, n, H):
    from fused3s_amd import torch_ops
    rp, ci = random_csr(n, 9, n + H) if graph == "random" else star_csr(n, 3, n)
    g = torch_ops.TorchGraph(rp, ci, heads=H)
    if graph == "star":
        assert g.plan.num_split > 0
    gen = torch.Generator().manual_seed(n)
    qkv = torch.randn(n, 3 * H * 64, generator=gen).half().cuda()
    q, k, v = (t.contiguous() for t in qkv.view(n, 3, H, 64).unbind(1))
    want = g.attention(q, k, v, scale=0.125)
    assert torch.equal(g.attention_packed(qkv, 0.125), want)
    half = g.attention_packed(qkv, 0.125, torch.float16)
    assert half.dtype == torch.float16 and torch.equal(half, want.half())


def test_packed_rejects(gpu):
    from fused3s_amd import torch_ops
    rp, ci = random_csr(64, 3, 5)
    g = torch_ops.TorchGraph(rp, ci, heads=1)
    qkv = torch.zeros(64, 192, dtype=torch.float16, device="cuda")
    for bad in (qkv[:, :128], qkv.float(), qkv.cpu(), qkv[:63]):
        with pytest.raises(ValueError):
            g.attention_packed(bad)
    with pytest.raises(ValueError):
        g.attention_packed(qkv, dtype=torch.bfloat16)
    dense = torch_ops.TorchGraph(rp, ci, heads=1, masked=False)
    assert not dense.takes_packed()
    with pytest.raises(gpu.F3SError) as e:   # the plan holds no lists
        dense.attention_packed(qkv)
    assert e.value.name == "F3S_EINVAL"


@pytest.mark.parametrize("dtype", ["int32", "int64"])
def test_graph_from_device_tensors(gpu, dtype):
    """A graph prepared from CUDA index tensors (copied device to device, on
    a side stream too) is the one prepared from host arrays, and keeps its own
    copy of them."""
    from fused3s_amd import torch_ops
    rp, ci = random_csr(1500, 7, 8)
    want = torch_ops.TorchGraph(rp, ci, heads=2)
    drp, dci = (torch.as_tensor(a).to(getattr(torch, dtype)).cuda() for a in (rp, ci))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = torch_ops.TorchGraph(drp, dci, heads=2)
        drp.zero_(), dci.zero_()
    s.synchronize()
    assert np.array_equal(got.csr.row_ptr.numpy(), rp) and np.array_equal(got.csr.col_idx.numpy(), ci)
    assert (got.n, got.nnz) == (want.n, want.nnz)
    q, k, v = torch.randn(3, 1500, 2, 64).half().cuda().unbind(0)
    assert torch.equal(got.attention(q, k, v), want.attention(q, k, v))


def test_graph_refuses_device_tensors_as_host_ones(gpu):
    """Types that numpy does not take are no index types on the device either;
    the other ones are converted as on the host."""
    from fused3s_amd import torch_ops
    rp, ci = (torch.from_numpy(a) for a in random_csr(60, 4, 9))
    for device in ("cpu", "cuda"):
        with pytest.raises(TypeError):
            torch_ops.TorchGraph(rp.to(device), ci.bfloat16().to(device))
        g = torch_ops.TorchGraph(rp.short().to(device), ci.double().to(device))
        assert np.array_equal(g.csr.col_idx.numpy(), ci) and g.n == 60


@pytest.mark.parametrize("n,H", [(11_184_682, 1), (174_760, 64)])
def test_packed_at_its_limit(gpu, n, H):
    """The largest packed tensors taken, within 384 bytes a head of 4 GiB less
    48 KiB, give the planned pass's bits in every row; one node more is refused."""
    from fused3s_amd import torch_ops
    assert 3 * n * H * 128 <= 0xffff4000 < 3 * (n + 1) * H * 128

    def graph(nodes):
        i = torch.arange(nodes, device="cuda")
        pair = torch.stack([i, torch.where(i % 3 == 0, nodes - 1 - i // 64, (i * 7919 + 13) % nodes)])
        return torch_ops.TorchGraph((torch.arange(nodes + 1, device="cuda") * 2).int(),
                                    pair.sort(0).values.t().flatten().int(), heads=H)

    g = graph(n)
    assert g.takes_packed()
    gen = torch.Generator(device="cuda").manual_seed(n)
    qkv = torch.empty(n, 3 * H * 64, dtype=torch.float16, device="cuda")
    qkv.normal_(generator=gen)
    got = g.attention_packed(qkv, 0.125)
    half = g.attention_packed(qkv, 0.125, torch.float16)
    q, k, v = (t.contiguous() for t in qkv.view(n, 3, H, 64).unbind(1))
    del qkv
    want = g.attention(q, k, v, scale=0.125)
    assert torch.equal(got, want) and torch.equal(half, want.half())
    del q, k, v, want, got, half, g
    more = graph(n + 1)
    assert not more.takes_packed()
    with pytest.raises(gpu.F3SError) as e:
        more.attention_packed(torch.empty(n + 1, 3 * H * 64, dtype=torch.float16, device="cuda"))
    assert e.value.name == "F3S_EUNSUPPORTED"
