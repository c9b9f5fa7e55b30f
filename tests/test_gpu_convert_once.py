"""f3s_convert_csr_to_bsf_once against the oracle and against the count and
fill calls it stands for: the smallest graphs, graphs with and without listed
hub windows, no masks, and invalid CSRs, whose offsets may add up to more than
the lists hold (nothing is written past them)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import _oracle as orc
from conftest import random_csr, rng

pytestmark = pytest.mark.gpu

GUARD = 64   # tiles past the lists' end, filled with 0x5a


def most(n: int, nnz: int) -> int:
    return min(nnz, ((n + 15) // 16) ** 2)


def once(gpu, rp, ci, masks=True):
    """(status, T, offsets, block_col, tile_mask): both lists `most` + GUARD long."""
    from fused3s_amd import _lib
    n, nnz = len(rp) - 1, len(ci)
    csr = gpu.DeviceCSR(rp, ci)
    offs = gpu.DeviceArray((n + 15) // 16 + 1, np.int32)
    bcol = gpu.DeviceArray(most(n, nnz) + GUARD, np.int32)
    mask = gpu.DeviceArray((most(n, nnz) + GUARD) * 16, np.uint16)
    bcol.fill_bytes(0x5a)
    mask.fill_bytes(0x5a)
    T = C.c_int64(-1)
    status = _lib.hip().f3s_convert_csr_to_bsf_once(
        csr.row_ptr.ptr, csr.col_idx.ptr, n, nnz, offs.ptr, bcol.ptr, mask.ptr if masks else None,
        C.byref(T), None)
    gpu.synchronize()
    return status, T.value, offs.numpy(), bcol.numpy(), mask.numpy().reshape(-1, 16)


def two_calls(gpu, rp, ci):
    from fused3s_amd import _lib
    n, nnz = len(rp) - 1, len(ci)
    csr = gpu.DeviceCSR(rp, ci)
    offs = gpu.DeviceArray((n + 15) // 16 + 1, np.int32)
    T = C.c_int64(-1)
    f = _lib.hip().f3s_convert_csr_to_bsf
    assert f(csr.row_ptr.ptr, csr.col_idx.ptr, n, nnz, offs.ptr, None, None, C.byref(T), None) == 0
    bcol, mask = gpu.DeviceArray(T.value, np.int32), gpu.DeviceArray(T.value * 16, np.uint16)
    assert f(csr.row_ptr.ptr, csr.col_idx.ptr, n, nnz, offs.ptr, bcol.ptr, mask.ptr, C.byref(T),
             None) == 0
    return offs.numpy(), bcol.numpy(), mask.numpy().reshape(-1, 16)


def hubs(n: int, seed: int):
    """Windows of 1,025 to 9,000 edges among ones of a few."""
    r = rng(seed)
    deg = r.integers(0, 4, n)
    for u, d in ((3, 1025), (40, 4096), (77, 4097), (n - 1, 9000 if n > 9000 else n)):
        deg[u] = min(d, n)
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    ci = np.concatenate([np.sort(r.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    return rp, ci


@pytest.mark.parametrize("graph,n", [("random", 1), ("random", 16), ("random", 17),
                                     ("random", 2708), ("random", 40_001),
                                     ("full", 16), ("full", 200), ("full", 700),
                                     ("hubs", 20_000), ("hubs", 33_003)])
def test_once_is_two_calls(gpu, graph, n):
    rp, ci = (random_csr(n, min(n, 7), n) if graph == "random" else hubs(n, n) if graph == "hubs"
              else (np.arange(n + 1, dtype=np.int32) * n, np.tile(np.arange(n, dtype=np.int32), n)))
    if graph == "full":   # every tile there is
        assert len(orc.convert(n, rp, ci)[1]) == most(n, n * n) < n * n
    offs, bcol, mask = orc.convert(n, rp, ci)
    T = len(bcol)
    for want in ((offs, bcol, mask), two_calls(gpu, rp, ci)):
        status, t, o, b, m = once(gpu, rp, ci)
        assert status == 0 and t == T
        assert np.array_equal(o, want[0]) and np.array_equal(b[:T], want[1])
        assert np.array_equal(m[:T], want[2])
        assert (b[T:] == 0x5a5a5a5a).all() and (m[T:] == 0x5a5a).all()
    status, t, o, b, m = once(gpu, rp, ci, masks=False)
    assert status == 0 and t == T and np.array_equal(b[:T], bcol) and (m == 0x5a5a).all()


@pytest.mark.parametrize("hub", [False, True])
def test_once_invalid(gpu, hub):
    """A row pointer that goes back makes later windows count the same edges
    again; a column past n is left out.  Both are EDATA, and the lists' guards
    stay as they were."""
    W, E = 200, 1500 if hub else 600
    n = 16 * W
    ci = (np.arange(E) * 7 % n).astype(np.int32)
    rp = np.zeros(n + 1, np.int32)
    for w in range(W):   # odd windows go back to 0, even ones have E edges and W tiles
        rp[16 * w:16 * w + 16] = np.linspace(0, E, 17)[:16].astype(np.int32) if w % 2 == 0 else 0
        if w % 2:
            rp[16 * w] = E
    rp[n] = 0
    status, _, _, b, m = once(gpu, rp, ci)
    assert status != 0
    assert (b[E:] == 0x5a5a5a5a).all() and (m[E:] == 0x5a5a).all()   # (E < W * W)
    rp, ci = random_csr(300, 5, 2)
    ci = ci.copy()
    ci[7] = 300
    status, _, _, b, m = once(gpu, rp, ci)
    end = most(300, len(ci))
    assert status != 0 and (b[end:] == 0x5a5a5a5a).all() and (m[end:] == 0x5a5a).all()
    with pytest.raises(gpu.F3SError) as e:
        gpu.convert_device(gpu.DeviceCSR(rp, ci))
    assert e.value.name == "F3S_EDATA"


@pytest.mark.parametrize("n,degree,copied", [(20_000, 25, True), (4000, 100, False), (700, 90, False)])
def test_lists_keep_no_more_than_four_times_their_size(gpu, n, degree, copied):
    """Clustered graphs, 25, 100 and 90 edges a node in groups of 160: the
    tensors are copies of their own size where the lists they were found in are
    far longer; contents as the oracle's, in a DeviceBSF too."""
    torch = pytest.importorskip("torch")
    from fused3s_amd import torch_ops
    r = rng(n + degree)
    rows = np.repeat(np.arange(n), degree)
    key = np.unique(rows * n + np.minimum(rows // 160 * 160 + r.integers(0, 160, len(rows)), n - 1))
    rp = np.searchsorted(key, np.arange(n + 1) * n).astype(np.int32)
    ci = (key % n).astype(np.int32)
    offs, bcol, mask = orc.convert(n, rp, ci)
    T, nnz = len(bcol), len(ci)
    o, b, m = torch_ops.to_block_sparse(rp, ci)
    assert np.array_equal(o.cpu().numpy(), offs) and np.array_equal(b.cpu().numpy(), bcol)
    assert np.array_equal(m.cpu().numpy().view(np.uint16), mask)
    kept = T if copied else most(n, nnz)
    assert b.untyped_storage().nbytes() == 4 * kept and m.untyped_storage().nbytes() == 32 * kept
    assert kept <= 4 * T or 36 * (kept - T) < 2**22
    assert torch_ops.to_block_sparse(rp, ci, masks=False)[1].untyped_storage().nbytes() == 4 * kept
    h = gpu.convert_device(gpu.DeviceCSR(rp, ci)).to_host()
    assert np.array_equal(h.window_offsets, offs) and np.array_equal(h.block_col_indices, bcol)
    assert np.array_equal(h.tile_masks, mask)


def test_failed_call_leaves_the_next_its_status(gpu):
    """A call that fails after its first launch (here on an error that another
    library's HIP call left pending on the thread) waits for its kernels: one
    that finds a bad column then does not write it into the next call's status
    words, which are the thread's."""
    torch = pytest.importorskip("torch")
    from fused3s_amd import _lib
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = C.CDLL(path)
    f = _lib.hip().f3s_convert_csr_to_bsf
    n = 4_000_000
    rp = torch.arange(n + 1, dtype=torch.int32, device="cuda") * 16
    ci = torch.randint(n, (16 * n,), dtype=torch.int32, device="cuda")
    offs = torch.empty(n // 16 + 1, dtype=torch.int32, device="cuda")
    small_rp, small_ci = (torch.from_numpy(a).cuda() for a in random_csr(2000, 5, 6))
    small_offs = torch.empty(126, dtype=torch.int32, device="cuda")
    T = C.c_int64(-1)

    def big():
        return f(rp.data_ptr(), ci.data_ptr(), n, 16 * n, offs.data_ptr(), None, None, C.byref(T),
                 None)

    def small():
        return f(small_rp.data_ptr(), small_ci.data_ptr(), 2000, small_ci.numel(),
                 small_offs.data_ptr(), None, None, C.byref(T), None)

    assert big() == 0 and small() == 0   # (the scratch of both is cached now)
    ci[-1] = n                           # outside [0, n)
    torch.cuda.synchronize()
    assert hip.hipSetDevice(10_000) != 0
    failed = big()
    status = small()
    assert failed == 4 and status == 0   # F3S_ENODEV (the pending error), F3S_OK
    assert small_offs[125].item() == T.value
    torch.cuda.synchronize()
