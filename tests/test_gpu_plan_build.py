"""Building a plan at the sizes where its launches change: the window order
ranked in one launch up to 4,096 windows and sorted past that, and the plan's
scans over one block of 1,024 positions, a few, and with hub windows split on
both sides of a block's edge."""
from __future__ import annotations

import numpy as np
import pytest

import _oracle as orc
from conftest import rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [1, 2, 63, 64, 65, 4095, 4096, 4097, 9000])
def test_window_order(gpu, W):
    # many equal counts (stable: ascending window), zeros, one window of W tiles
    r = rng(W)
    counts = r.integers(0, min(W, 5) + 1, W)
    counts[W // 2] = W
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    bsf = gpu.DeviceBSF(16 * W, W, int(offs[-1]), gpu.DeviceArray.from_numpy(offs), None, None)
    got = gpu.window_order_device(bsf).numpy()
    assert np.array_equal(got, orc.window_order(offs))


@pytest.mark.parametrize("W", [1023, 1024, 1025, 2500])
@pytest.mark.parametrize("seg", [0, 3])
def test_plan_positions(gpu, W, seg):
    n, r = 16 * W - 3, rng(W + seg)
    deg = r.integers(0, 4, n)
    for w in (0, 5, 1022, 1023, 1024, W - 1):   # windows of many tiles, split with seg = 3
        if w < W:
            deg[16 * w] = 40
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    ci = r.integers(0, n, int(rp[-1])).astype(np.int32)
    keys = np.unique(np.repeat(np.arange(n), deg).astype(np.int64) * n + ci)   # no repeats
    rp = np.searchsorted(keys // n, np.arange(n + 1)).astype(np.int32)
    ci = (keys % n).astype(np.int32)
    bsf = gpu.convert_device(gpu.DeviceCSR(rp, ci))
    order = gpu.window_order_device(bsf)
    q, k, v = (r.standard_normal((n, 1, 64)).astype(np.float16) for _ in range(3))
    dq, dk, dv = (gpu.DeviceArray.from_numpy(x.view(np.uint16)) for x in (q, k, v))
    f = [x.astype(np.float32) for x in (q, k, v)]
    want = orc.masked_attention(n, 64, 1, *f, rp, ci, 0.125)
    dense = orc.tile_dense_attention(n, 64, 1, *f, bsf.window_offsets.numpy(),
                                     bsf.block_col.numpy(), 0.125)
    for o in (order, None):
        plan = gpu.Plan(bsf, o, H=1, seg_tiles=seg)
        tiles = np.diff(bsf.window_offsets.numpy())
        if seg:
            assert plan.num_items == int(np.maximum(1, -(-tiles // seg)).sum())
            assert plan.num_split == int((tiles > seg).sum())
        for compiled in (False, True):
            if compiled:
                plan.compile()
            for _ in range(2):   # the arrival counts are left at zero
                out = gpu.DeviceArray((n, 1, 64), np.float32)
                out.fill_bytes(0xff)
                plan.forward(dq, dk, dv, out, masked=True, scale=0.125)
                gpu.synchronize()
                assert np.abs(out.numpy() - want).max() <= 2e-3
        out = gpu.DeviceArray((n, 1, 64), np.float32)
        out.fill_bytes(0xff)
        plan.forward(dq, dk, dv, out, masked=False, scale=0.125)
        gpu.synchronize()
        assert np.abs(out.numpy() - dense).max() <= 2e-3


@pytest.mark.parametrize("W", [513, 1024, 1025, 2049, 4095, 4096, 4097])
@pytest.mark.parametrize("masked", [True, False])
def test_natural_order_schedule(gpu, W, masked):
    # the drop-in launch without an order, whose schedule is built by one
    # workgroup up to 4,096 windows: hub windows of every block column (heavy
    # past 1,024), windows without edges, a short last window
    n, r = 16 * W - 7, rng(W)
    keys = [np.arange(0, n, 3, dtype=np.int64) * (n + 1)]
    for w in (0, 7, 1000, W - 1):
        if w < W:
            u = 16 * w + int(r.integers(0, 9))
            keys.append(u * np.int64(n) + np.arange(0, n, 16))
    u = r.integers(0, n, 6 * n)
    u = u[u // 16 % 50 != 13]
    keys.append(u * np.int64(n) + r.integers(0, n, len(u)))
    keys = np.unique(np.concatenate(keys))
    rp = np.searchsorted(keys // n, np.arange(n + 1)).astype(np.int32)
    ci = (keys % n).astype(np.int32)
    bsf = gpu.convert_device(gpu.DeviceCSR(rp, ci))
    q, k, v = (r.standard_normal((n, 1, 64)).astype(np.float16) for _ in range(3))
    dev = [gpu.DeviceArray.from_numpy(x.view(np.uint16)) for x in (q, k, v)]
    out = gpu.DeviceArray((n, 1, 64), np.float32)
    out.fill_bytes(0xff)   # NaN: a row no window writes fails
    gpu.attention_fwd(*dev, out, bsf, masked=masked, scale=0.125)
    gpu.synchronize()
    f = [x.astype(np.float32) for x in (q, k, v)]
    want = (orc.masked_attention(n, 64, 1, *f, rp, ci, 0.125) if masked else
            orc.tile_dense_attention(n, 64, 1, *f, bsf.window_offsets.numpy(),
                                     bsf.block_col.numpy(), 0.125))
    assert np.abs(out.numpy() - want).max() <= 2e-3
