"""The drop-in launch's heavy windows on teams: at the edges of what is heavy
(1,024 tiles on graphs of few tiles), where the heaviest makes the first of
them run apart (few other tiles) and where it does not (many), in natural and
descending order and in orders that put them past the 512 and 64 entries
looked at; every row against the planned pass, which cuts windows elsewhere
(bound: the parity tests' 2e-3), and on one graph of each kind against the
oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import rng

pytestmark = pytest.mark.gpu


def star(W: int, hubs: dict[int, int]):
    """A self-loop per node; hubs[w] = tiles of window w, spread over 16 rows."""
    n = 16 * W - 3
    r = rng(W)
    rows, cols = [np.arange(n)], [np.arange(n)]
    for w, tiles in hubs.items():
        c = r.choice(np.delete(np.arange(W), w), tiles - 1, replace=False)
        rows.append(16 * w + r.integers(0, min(16, n - 16 * w), len(c)))
        cols.append(np.minimum(16 * c + r.integers(0, 16, len(c)), n - 1))
    key = np.unique(np.concatenate(rows).astype(np.int64) * n + np.concatenate(cols))
    rp = np.searchsorted(key, np.arange(n + 1, dtype=np.int64) * n).astype(np.int32)
    return torch.from_numpy(rp).cuda(), torch.from_numpy((key % n).astype(np.int32)).cuda()


@pytest.mark.parametrize("W,hubs,H", [
    (1025, {0: 1024, 3: 1025, 1024: 1025}, 1),
    (1100, {7: 1030, 1099: 1100}, 3),
    (6000, {w: 1026 + w for w in range(0, 520)}, 1),   # more than the team list takes
    (1100, {w: 1026 + w for w in range(0, 40)}, 1),    # more than the entries that run apart
    (16_384, {5: 16_384, 900: 1500}, 1),
    (16_500, {9: 16_384, 40: 16_390, 16_000: 16_500, 77: 2000}, 2),
])
@pytest.mark.parametrize("masked", [True, False])
def test_heavy_windows(gpu, W, hubs, H, masked):
    from fused3s_amd import torch_ops
    rp, ci = star(W, hubs)
    n = rp.numel() - 1
    gen = torch.Generator(device="cuda").manual_seed(W)
    q, k, v = (torch.randn(n, H, 64, device="cuda", generator=gen, dtype=torch.float16)
               for _ in range(3))
    want = torch_ops.TorchGraph(rp, ci, heads=H, masked=masked).attention(q, k, v, scale=0.25)
    offs, bcol, mask = torch_ops.to_block_sparse(rp, ci)
    down = torch.sort(offs[1:] - offs[:-1], descending=True, stable=True).indices.to(torch.int32)
    past = torch.cat([down[600:664], down[:64], down[64:600], down[664:]])   # from entry 64 on
    for order in (None, down, past, down.flip(0).contiguous()):
        got = torch.ops.fused3s.attention_fwd(q, k, v, offs, bcol, mask if masked else None,
                                              order, 0.25)
        assert torch.isfinite(got).all()
        assert (got - want).abs().max() <= 2e-3
        again = torch.ops.fused3s.attention_fwd(q, k, v, offs, bcol, mask if masked else None,
                                                order, 0.25)
        assert torch.equal(got, again)


@pytest.mark.parametrize("W,hubs", [(1100, {7: 1030, 1099: 1100}),                       # apart
                                    (1300, {w: 1025 + 7 * w for w in range(0, 30, 2)})])
@pytest.mark.parametrize("masked", [True, False])
def test_heavy_windows_oracle(gpu, W, hubs, masked):
    import _oracle as orc

    from fused3s_amd import torch_ops
    rp, ci = star(W, hubs)
    n = rp.numel() - 1
    gen = torch.Generator(device="cuda").manual_seed(W + 1)
    q, k, v = (torch.randn(n, 1, 64, device="cuda", generator=gen, dtype=torch.float16)
               for _ in range(3))
    offs, bcol, mask = torch_ops.to_block_sparse(rp, ci)
    down = torch.sort(offs[1:] - offs[:-1], descending=True, stable=True).indices.to(torch.int32)
    host = [t.float().cpu().numpy().reshape(n, 64) for t in (q, k, v)]
    if masked:
        want = orc.masked_attention(n, 64, 1, *host, rp.cpu().numpy(), ci.cpu().numpy(), scale=0.25)
    else:
        want = orc.tile_dense_attention(n, 64, 1, *host, offs.cpu().numpy(), bcol.cpu().numpy(),
                                        scale=0.25)
    for order in (None, down):
        got = torch.ops.fused3s.attention_fwd(q, k, v, offs, bcol, mask if masked else None,
                                              order, 0.25)
        assert np.abs(got.cpu().numpy().reshape(want.shape) - want).max() <= 2e-3


@pytest.mark.parametrize("masked", [True, False])
def test_one_node_joined_to_all(gpu, masked):
    """The hub window of such a graph is most of the pass.  Past the entries
    looked at it is one wave's; in descending order it has 16 waves (1 / 7 to 1 / 9
    of the time), not 4 (1 / 3.5)."""
    from fused3s_amd import torch_ops
    n = 131_000
    i = torch.arange(n, device="cuda")
    key = torch.unique(torch.cat([i * n + i, i * n + 7, 7 * n + i]))
    rp = torch.searchsorted(key, torch.arange(n + 1, device="cuda") * n).int()
    offs, bcol, mask = torch_ops.to_block_sparse(rp, (key % n).int())
    q, k, v = (torch.randn(n, 1, 64, device="cuda", dtype=torch.float16) for _ in range(3))
    down = torch.sort(offs[1:] - offs[:-1], descending=True, stable=True).indices.int()

    def us(order):
        def run():
            return torch.ops.fused3s.attention_fwd(q, k, v, offs, bcol, mask if masked else None,
                                                   order, 0.125)
        out = run()
        best = float("inf")
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            run()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best, out

    team, got = us(down)
    wave, want = us(down.flip(0).contiguous())
    assert (got - want).abs().max() <= 2e-3
    assert team < wave / 5
