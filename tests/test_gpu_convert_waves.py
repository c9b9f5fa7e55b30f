"""The converter's main launch at the sizes where its branches meet, bit for
bit against the oracle: windows around one wave's 1,024 edges, a hub
workgroup's one chunk of 4,096 edges and the heavier hubs' two ways out (few
tiles for their edges: staged beside the bitmap; many: atomics on the zeroed
output), windows around a stage of 160 tiles, rows in any order, empty rows,
and the lists without masks."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as orc
from conftest import rng

pytestmark = pytest.mark.gpu


def window_graph(windows: dict[int, np.ndarray], n: int, sort: bool, seed: int):
    """CSR of n nodes; windows[w] = columns dealt at random to the 16 rows of
    window w (some rows get none)."""
    r = rng(seed)
    rows, cols = [], []
    for w, c in windows.items():
        used = r.choice(16, size=int(r.integers(1, 17)), replace=False)
        rows.append(16 * w + r.choice(used, len(c)))
        cols.append(c)
    rr = np.concatenate(rows).astype(np.int64)
    cc = np.concatenate(cols).astype(np.int64)
    order = np.lexsort((cc, rr)) if sort else np.argsort(rr, kind="stable")
    rr, cc = rr[order], cc[order]
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rr + 1, 1)
    return np.cumsum(rp).astype(np.int32), cc.astype(np.int32)


def check(gpu, rp, ci, masks=True):
    n = len(rp) - 1
    offs, bcol, mask = orc.convert(n, rp, ci)
    bsf = gpu.convert_device(gpu.DeviceCSR(rp, ci), masks=masks)
    assert np.array_equal(bsf.window_offsets.numpy(), offs)
    assert np.array_equal(bsf.block_col.numpy(), bcol)
    if masks:
        assert np.array_equal(bsf.tile_mask.numpy().reshape(-1, 16), mask)


@pytest.mark.parametrize("n", [16 * 1023 + 5, 16 * 1024, 16 * 2050, 70_001])
@pytest.mark.parametrize("sort", [True, False])
def test_window_sizes(gpu, n, sort):
    r = rng(n + sort)
    W = (n + 15) // 16
    edges = (1, 63, 64, 65, 127, 128, 129, 1023, 1024, 1025, 4095, 4096, 4097, 8200)
    windows = {}
    for k, E in enumerate(edges):
        windows[3 + 5 * k] = r.integers(0, n, E)               # columns anywhere
        windows[5 + 5 * k] = 16 * 7 + r.integers(0, 16 * 40, E)   # within 40 block columns
    windows[W - 1] = r.integers(0, n, 300)
    last = n - 16 * (W - 1)   # rows of the last window
    rp, ci = window_graph(windows, 16 * W, sort, 5)
    if last < 16:             # its edges move to the rows it has
        e0 = rp[16 * (W - 1)]
        rp = np.concatenate([rp[:16 * (W - 1) + 1], np.full(last, rp[-1], np.int32)])
        ci[e0:] = np.sort(ci[e0:]) if sort else ci[e0:]
    check(gpu, rp, ci)


@pytest.mark.parametrize("tiles", [159, 160, 161, 320, 321, 1000])
def test_stage_rounds(gpu, tiles):
    # every block column once, in one wave's window and in a hub window
    n = 16 * 1100
    r = rng(tiles)
    c = 16 * np.arange(tiles) + r.integers(0, 16, tiles)
    windows = {0: c, 9: np.concatenate([c, r.choice(c, 1100), r.choice(c, 100)])}
    rp, ci = window_graph(windows, n, True, 6)
    check(gpu, rp, ci)


def test_many_hubs_and_lists_without_masks(gpu):
    # more hub windows than one list block's share, light ones between them
    n = 16 * 2100
    r = rng(3)
    windows = {w: r.integers(0, n, int(r.integers(1000, 1200)) if w % 3 else 5000)
               for w in range(0, 2100, 2)}
    rp, ci = window_graph(windows, n, True, 7)
    check(gpu, rp, ci)
    check(gpu, rp, ci, masks=False)


def one_row(cols, n):
    """Node 7's row is `cols`; every other node has an edge to itself."""
    rows = np.arange(n)
    counts = np.ones(n, np.int64)
    counts[7] = len(cols)
    ci = np.empty(int(counts.sum()), np.int32)
    rp = np.concatenate([[0], np.cumsum(counts)])
    ci[rp[:-1]] = rows
    ci[rp[7]:rp[8]] = cols
    return rp.astype(np.int32), ci


@pytest.mark.parametrize("order", ["ascending", "repeated", "pairs", "shuffled"])
def test_shared_mask_words(gpu, order):
    """A heavy hub of more tiles than are staged, whose neighbouring edges
    share words of the masks: runs of 16, runs longer than a wave (columns
    repeated), runs that come back to a word, none."""
    n = 16 * 3000
    c = np.arange(n)
    if order == "repeated":
        c = np.repeat(c, 5)
    elif order == "pairs":   # two edges of one tile, two of the next, two of the first ...
        c = c.reshape(-1, 2, 8, 2).transpose(0, 2, 1, 3).ravel()
    elif order == "shuffled":
        c = rng(4).permutation(c)
    rp, ci = one_row(c, n)
    check(gpu, rp, ci)
    rp, ci = window_graph({5: np.tile(np.arange(n), 16), 6: np.arange(n)}, n, order != "shuffled", 8)
    check(gpu, rp, ci)


def test_masks_of_one_node_joined_to_all(gpu):
    """A word's 16 edges are ORed at once: the masks add a tenth to a quarter to
    the conversion's time (with an atomic for every edge, 1.1 times as much again)."""
    import torch

    from fused3s_amd import torch_ops
    rp, ci = (torch.from_numpy(a).cuda() for a in one_row(np.arange(300_000), 300_000))

    def us(masks):
        best = float("inf")
        for _ in range(8):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            torch_ops.to_block_sparse(rp, ci, masks=masks)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3)
        return best

    assert us(True) < 1.7 * us(False)


def test_more_hubs_than_workgroups(gpu):
    """2,600 hub windows, 2,300 of them heavy: each of the launch's 2,048 hub
    workgroups takes a second window after a staged, few-tile or many-tile one."""
    W, n = 2600, 16 * 2600
    r = rng(12)
    windows = {}
    for w in range(W):
        kind = w % 4 if w % 26 < 23 else 4
        if kind == 0:     # heavy, a tile for nearly every edge
            c = r.integers(0, n, 4200)
        elif kind == 1:   # heavy, 20 tiles
            c = (r.integers(0, n - 320) + r.integers(0, 320, 4800)).astype(np.int64)
        elif kind == 2:   # heavy, a row of consecutive columns of more tiles than are staged
            c = np.arange(n) if w % 400 == 2 else np.arange(5000) + int(r.integers(0, n - 5000))
        elif kind == 3:   # heavy by one edge
            c = r.integers(0, n, 4097)
        else:             # staged
            c = r.integers(0, n, int(r.integers(1025, 4097)))
        windows[w] = c
    rp, ci = window_graph(windows, n, True, 13)
    check(gpu, rp, ci)
    check(gpu, rp, ci, masks=False)
