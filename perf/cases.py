"""Performance cases of the fused sparse graph attention path.

Each case is one call (or the short sequence of calls) that a program using
the PyTorch binding makes: the planned attention pass on a graph prepared
once, the stateless operator on block-sparse tensors, the CSR -> block-sparse
converter, the graph-transformer layer, and the whole preparation plus layer
that a mini-batch loop pays on every batch.  Graphs are made on the GPU from
the case and the seed alone, of the two families the package's workloads use: power-law
degrees on random node ids, and communities of consecutive node ids.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from fused3s_amd import torch_ops

D = 64   # feature dim per head

# path: planned  TorchGraph.attention on q, k, v [n, H, 64] fp16
#       operator torch.ops.fused3s.attention_fwd on to_block_sparse's tensors
#       blocks   to_block_sparse on int32 CSR tensors
#       layer    GraphTransformerLayer on a prepared TorchGraph
#       batch    TorchGraph from host CSR arrays, then GraphTransformerLayer
# graph: powerlaw (gamma, max_degree) or community (community, p_intra)


def _case(name, path, graph, n, degree, heads=1, masked=True, ordered=False, scale=1.0, loops=True,
          gamma=2.2, max_degree=16384, community=4096, p_intra=0.8, dim=128):
    return {"name": name, "path": path, "graph": graph, "n": n, "degree": degree, "heads": heads,
            "masked": masked, "ordered": ordered, "scale": scale, "loops": loops, "gamma": gamma,
            "max_degree": max_degree, "community": community, "p_intra": p_intra, "dim": dim}


def listed():
    return [
        # a citation-sized graph, attended again and again (one call is one
        # launch): latency
        _case("planned_small", "planned", "powerlaw", 2708, 3.9, gamma=2.5, max_degree=170),
        # the package's headline workload: a large graph of random node ids,
        # one head, edge-exact
        _case("planned_1m", "planned", "powerlaw", 1_000_000, 16),
        # the largest workload: community-ordered ids, four heads
        _case("planned_community_h4", "planned", "community", 2_400_000, 50, heads=4),
        # the reference's own semantics (every column of an active tile) on a
        # small sparse graph
        _case("dense_small", "planned", "powerlaw", 3327, 2.74, masked=False, gamma=2.8,
              max_degree=99),
        # and on the headline graph
        _case("dense_1m", "planned", "powerlaw", 1_000_000, 16, masked=False),
        # the reference's launch shape without a plan: descending window
        # order, headline graph
        _case("operator_1m", "operator", "powerlaw", 1_000_000, 16, ordered=True),
        # the same operator inside a model without an order: mid-sized graph
        # of odd size, three heads, scaled logits
        _case("operator_mid_h3", "operator", "community", 50_001, 20, heads=3, scale=0.125,
              community=1000),
        # conversion of a small graph: launches and host round trips
        _case("blocks_small", "blocks", "powerlaw", 2708, 3.9, gamma=2.5, max_degree=170),
        # conversion of the headline graph, with hub windows
        _case("blocks_1m", "blocks", "powerlaw", 1_000_000, 16),
        # conversion of the community graph: many edges per window
        _case("blocks_community", "blocks", "community", 2_400_000, 50),
        # a mini-batch step: a sampled subgraph arrives from the loader, is
        # prepared and goes through a layer once
        _case("batch_layer", "batch", "powerlaw", 20_011, 14, heads=4, loops=False, gamma=2.5,
              max_degree=500),
        # full-graph inference with a graph-transformer layer
        _case("layer_large_h2", "layer", "powerlaw", 500_000, 12, heads=2, gamma=2.5,
              max_degree=4096),
    ]


def draw(rng):
    path = rng.choice(["planned", "planned", "operator", "operator", "blocks", "blocks", "layer",
                       "batch"])
    masked = path in ("blocks", "layer", "batch") or rng.random() < 0.65
    top = {"planned": 1_000_000, "operator": 1_000_000, "blocks": 1_500_000, "layer": 500_000,
           "batch": 60_000}[path]
    n = int(round(math.exp(rng.uniform(math.log(1000), math.log(top)))))
    degree = round(math.exp(rng.uniform(math.log(3), math.log(50))), 2)
    heads = rng.choice([1, 1, 2, 3, 4, 8])
    # no dearer than the largest listed cases
    most = 40e6 if masked else 12e6
    while heads > 1 and n * (degree + 1) * heads > most:
        heads -= 1
    degree = min(degree, max(3.0, round(most / (n * heads) - 1, 2)))
    graph = rng.choice(["powerlaw", "community"])
    return {"path": path, "graph": graph, "n": n, "degree": degree, "heads": heads,
            "masked": masked, "ordered": rng.random() < 0.5, "scale": rng.choice([1.0, 0.125]),
            "loops": rng.random() < 0.7, "gamma": round(rng.uniform(2.1, 2.9), 2),
            "max_degree": int(min(16384, max(64, n // 16))),
            "community": rng.choice([512, 1000, 4096]), "p_intra": round(rng.uniform(0.6, 0.9), 2),
            "dim": rng.choice([64, 100, 128])}


# ------------------------------------------------------------------ inputs

def _generator(seed, salt):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + salt) % (1 << 62))


def _relabel(case, gen):
    """New node ids, drawn from `gen`: the nodes of each window of 16 in a
    random order, and the windows too -- among all of them, or on a graph of
    communities among 32 neighbours, which keeps its locality.  Every window
    keeps its number of active tiles, so another seed gives another graph of
    the same sizes."""
    n = case["n"]
    W = n // 16   # whole windows; the nodes after them stay
    win = torch.arange(W, device="cuda")
    if case["graph"] == "powerlaw":
        win = torch.randperm(W, device="cuda", generator=gen)
    else:
        g = W // 32
        part = torch.argsort(torch.rand(g, 32, device="cuda", generator=gen), dim=1)
        win[:32 * g] = (part + 32 * torch.arange(g, device="cuda")[:, None]).flatten()
    inner = torch.argsort(torch.rand(W, 16, device="cuda", generator=gen), dim=1)
    ids = torch.arange(n, device="cuda")
    ids[:16 * W] = (win[:, None] * 16 + inner).flatten()
    return ids


def _graph(case, seed):
    """Symmetric CSR (row_ptr, col_idx) of int32 CUDA tensors, columns
    ascending and unique in each row.  The case decides which nodes are
    joined, the seed what their ids are."""
    n, gen = case["n"], _generator(20, 0)
    pairs = max(1, int(n * case["degree"] / 2))
    if case["graph"] == "powerlaw":
        w = np.arange(1, n + 1, dtype=np.float64) ** (-1.0 / (case["gamma"] - 1.0))
        mean = w.sum() / n
        w = np.minimum(w, mean * max(2.0, case["max_degree"] / case["degree"]))
        cdf = torch.from_numpy(np.cumsum(w) / w.sum()).cuda()
        x = torch.rand(2, pairs, dtype=torch.float64, device="cuda", generator=gen)
        ends = torch.searchsorted(cdf, x).clamp_(max=n - 1)
        del x
        ends = torch.randperm(n, device="cuda", generator=gen)[ends]   # no order by degree
        u, v = ends[0], ends[1]
    else:
        c = case["community"]
        u = torch.randint(n, (pairs,), device="cuda", generator=gen)
        intra = torch.rand(pairs, device="cuda", generator=gen) < case["p_intra"]
        base = u // c * c
        size = torch.clamp(n - base, max=c)
        x = torch.rand(pairs, dtype=torch.float64, device="cuda", generator=gen)
        v = torch.where(intra, base + (x * size).long(), (x * n).long())
        del x, base, size, intra
    ids = _relabel(case, _generator(seed, 1))
    keep = u != v
    u, v = ids[u[keep]], ids[v[keep]]
    keys = [u * n + v, v * n + u]
    if case["loops"]:
        i = torch.arange(n, device="cuda")
        keys.append(i * n + i)
    del u, v, keep
    keys = torch.unique(torch.cat(keys))
    row_ptr = torch.searchsorted(keys, torch.arange(n + 1, device="cuda") * n)
    return row_ptr.to(torch.int32), (keys % n).to(torch.int32)


def _features(case, seed):
    """q, k, v ~ N(0, 1) in fp16, [n, H, 64]."""
    gen = _generator(seed, 2)
    return [torch.randn(case["n"], case["heads"], D, device="cuda", generator=gen,
                        dtype=torch.float16) for _ in range(3)]


def _layer(case, seed):
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(int(seed) % (1 << 62))
        layer = torch_ops.GraphTransformerLayer(case["dim"], heads=case["heads"])
    return layer.cuda().half()


def _nodes(case, seed):
    return torch.randn(case["n"], case["dim"], device="cuda", generator=_generator(seed, 3),
                       dtype=torch.float16)


def prepare(case, seed):
    row_ptr, col_idx = _graph(case, seed)
    path = case["path"]
    if path == "planned":
        q, k, v = _features(case, seed)
        graph = torch_ops.TorchGraph(row_ptr, col_idx, heads=case["heads"], masked=case["masked"])
        return {"case": case, "graph": graph, "q": q, "k": k, "v": v}
    if path == "operator":
        q, k, v = _features(case, seed)
        offs, bcol, mask = torch_ops.to_block_sparse(row_ptr, col_idx)
        order = None
        if case["ordered"]:
            # the reference's descending workload order
            order = torch.sort(offs[1:] - offs[:-1], descending=True,
                               stable=True).indices.to(torch.int32)
        return {"case": case, "q": q, "k": k, "v": v, "offs": offs, "bcol": bcol,
                "mask": mask if case["masked"] else None, "order": order}
    if path == "blocks":
        return {"case": case, "row_ptr": row_ptr, "col_idx": col_idx}
    layer, x = _layer(case, seed), _nodes(case, seed)
    if path == "layer":
        graph = torch_ops.TorchGraph(row_ptr, col_idx, heads=case["heads"])
        return {"case": case, "layer": layer, "x": x, "graph": graph}
    return {"case": case, "layer": layer, "x": x, "row_ptr": row_ptr.cpu().numpy(),
            "col_idx": col_idx.cpu().numpy()}


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "planned":
        return state["graph"].attention(state["q"], state["k"], state["v"], scale=case["scale"])
    if path == "operator":
        return torch.ops.fused3s.attention_fwd(state["q"], state["k"], state["v"], state["offs"],
                                               state["bcol"], state["mask"], state["order"],
                                               case["scale"])
    if path == "blocks":
        return torch_ops.to_block_sparse(state["row_ptr"], state["col_idx"])
    if path == "layer":
        return state["layer"](state["x"], state["graph"])
    graph = torch_ops.TorchGraph(state["row_ptr"], state["col_idx"], heads=case["heads"])
    return state["layer"](state["x"], graph)


# ------------------------------------------------------------- work, tolerance

def _sizes(case):
    """Expected edges and active tiles."""
    n, W = case["n"], (case["n"] + 15) // 16
    edges = n * (case["degree"] + (1 if case["loops"] else 0))
    per = 16.0 * edges / n   # a window's edges

    def hit(balls, bins):
        return bins * (1.0 - math.exp(-balls / bins))

    if case["graph"] == "community":
        bins = min(W, max(1, case["community"] // 16))
        tiles = W * min(W, hit(per * case["p_intra"], bins) + hit(per * (1 - case["p_intra"]), W))
    else:
        tiles = W * hit(per, W)
    return edges, tiles


def work(case):
    n, H = case["n"], case["heads"]
    edges, tiles = _sizes(case)
    csr = 4.0 * edges + 4.0 * n
    path = case["path"]
    if path == "blocks":
        return {"bytes": csr + 36.0 * tiles + 4.0 * (n / 16), "flops": 0.0}
    attn = 4.0 * D * H * (edges if case["masked"] else 256.0 * tiles)
    feats = n * H * D * (3 * 2 + 4.0)
    if path in ("planned", "operator"):
        return {"bytes": feats + (csr if case["masked"] else 4.0 * tiles), "flops": attn}
    weights = 4 * H * D * case["dim"]
    return {"bytes": csr + 2.0 * (2 * n * case["dim"] + weights),
            "flops": attn + 2.0 * n * weights}


def tolerance(case):
    if case["path"] == "blocks":
        return "exact"
    if case["path"] in ("planned", "operator"):
        # weights and inputs of the second product in fp16, sums in fp32
        # (2.1e-4 against 64 bits at most over the ranges)
        return {"rel": 8e-4}
    # and fp16 projections, in and out (3.8e-4)
    return {"rel": 1.6e-3}


# ------------------------------------------------------------------ 64 bits

def _masked64(row_ptr, col_idx, q, k, v, scale):
    n, H = q.shape[0], q.shape[1]
    out = torch.zeros(n, H, D, dtype=torch.float64, device="cuda")
    host = row_ptr.cpu().numpy().astype(np.int64)
    step = max(1, (1 << 20) // H)
    r0 = 0
    while r0 < n:
        r1 = int(np.searchsorted(host, host[r0] + step, side="right")) - 1
        r1 = min(n, max(r1, r0 + 1))
        e0, e1 = int(host[r0]), int(host[r1])
        if e1 > e0:
            deg = (row_ptr[r0 + 1:r1 + 1] - row_ptr[r0:r1]).long()
            idx = torch.repeat_interleave(torch.arange(r1 - r0, device="cuda"), deg)
            col = col_idx[e0:e1].long()
            s = (q[r0 + idx].double() * k[col].double()).sum(-1) * scale
            m = torch.full((r1 - r0, H), -math.inf, dtype=torch.float64, device="cuda")
            m.scatter_reduce_(0, idx[:, None].expand(-1, H), s, "amax")
            p = torch.exp(s - m[idx])
            total = torch.zeros_like(m).index_add_(0, idx, p)
            acc = torch.zeros(r1 - r0, H, D, dtype=torch.float64, device="cuda")
            acc.index_add_(0, idx, p[..., None] * v[col].double())
            out[r0:r1] = torch.where(total[..., None] > 0, acc / total[..., None], 0.0)
        r0 = r1
    return out


def _tiles(case, row_ptr, col_idx):
    """Ascending unique (window, block column) keys, W * window + column."""
    n, W = case["n"], (case["n"] + 15) // 16
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"),
                                   (row_ptr[1:] - row_ptr[:-1]).long())
    keys, edge_tile = torch.unique(rows // 16 * W + col_idx.long() // 16, return_inverse=True)
    return W, rows, keys, edge_tile


def _dense64(case, row_ptr, col_idx, q, k, v, scale):
    n, H = q.shape[0], q.shape[1]
    W, rows, keys, edge_tile = _tiles(case, row_ptr, col_idx)
    del rows, edge_tile
    win, bcol = keys // W, keys % W
    offs = torch.searchsorted(win, torch.arange(W + 1, device="cuda")).cpu().numpy()
    lane = torch.arange(16, device="cuda")
    out = torch.zeros(W * 16, H, D, dtype=torch.float64, device="cuda")
    w0 = 0
    while w0 < W:
        w1 = int(np.searchsorted(offs, offs[w0] + 32768, side="right")) - 1
        w1 = min(W, max(w1, w0 + 1))
        t0, t1 = int(offs[w0]), int(offs[w1])
        if t1 > t0:
            wt = win[t0:t1]
            qrow = (wt[:, None] * 16 + lane).clamp_(max=n - 1)
            col = bcol[t0:t1, None] * 16 + lane
            there = col < n
            col = col.clamp_(max=n - 1)
            loc = wt - w0
            for h in range(H):
                kt = k[col, h].double().transpose(1, 2).contiguous()
                s = torch.bmm(q[qrow, h].double(), kt) * scale
                s.masked_fill_(~there[:, None, :], -math.inf)
                m = torch.full((w1 - w0, 16), -math.inf, dtype=torch.float64, device="cuda")
                m.scatter_reduce_(0, loc[:, None].expand(-1, 16), s.amax(-1), "amax")
                p = torch.exp(s - m[loc][..., None])
                total = torch.zeros_like(m).index_add_(0, loc, p.sum(-1))
                acc = torch.zeros(w1 - w0, 16, D, dtype=torch.float64, device="cuda")
                acc.index_add_(0, loc, torch.bmm(p, v[col, h].double()))
                o = torch.where(total[..., None] > 0, acc / total[..., None], 0.0)
                out[w0 * 16:w1 * 16, h] = o.reshape(-1, D)
        w0 = w1
    return out[:n]


def exact(case, seed):
    row_ptr, col_idx = _graph(case, seed)
    path = case["path"]
    if path == "blocks":
        W, rows, keys, edge_tile = _tiles(case, row_ptr, col_idx)
        offs = torch.searchsorted(keys, torch.arange(W + 1, device="cuda") * W).to(torch.int32)
        mask = torch.zeros(keys.numel() * 16, dtype=torch.int32, device="cuda")
        mask.index_add_(0, edge_tile * 16 + rows % 16,
                        torch.bitwise_left_shift(torch.ones_like(col_idx), col_idx % 16))
        return offs, (keys % W).to(torch.int32), mask.to(torch.int16).view(-1, 16)
    if path in ("planned", "operator"):
        q, k, v = _features(case, seed)
        if case["masked"]:
            return _masked64(row_ptr, col_idx, q, k, v, case["scale"])
        return _dense64(case, row_ptr, col_idx, q, k, v, case["scale"])
    layer, x = _layer(case, seed), _nodes(case, seed)
    lin = torch.nn.functional.linear
    n, H = case["n"], case["heads"]
    qkv = lin(x.double(), layer.qkv.weight.double(), layer.qkv.bias.double()).view(n, 3, H, D)
    o = _masked64(row_ptr, col_idx, qkv[:, 0], qkv[:, 1], qkv[:, 2], D ** -0.5)
    return lin(o.view(n, H * D), layer.proj.weight.double(), layer.proj.bias.double())
