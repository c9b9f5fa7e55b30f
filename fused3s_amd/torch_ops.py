"""PyTorch-ROCm binding of the fused pass, for a graph-transformer layer.

The reference has no framework binding; its natural caller is a graph
attention layer: a QKV projection GEMM, the fused sparse attention over the
graph's edges, and an output projection.  Here torch supplies the device
memory and the stream; the attention is the HIP library's planned pass
(f3s_attention_fwd_planned), called on torch's current stream with the
tensors' device pointers, and the layer's projections are its f3s_linear_f16
(torch.nn.Linear's own product where that kernel is not the better one).  There is no CPU fallback and no autograd: the
fused pass is forward-only, so calling it on tensors that require grad
raises.

    graph = TorchGraph(row_ptr, col_idx, heads=4)      # convert + plan + compile once
    o = graph.attention(q, k, v)                       # q/k/v [n, H, 64] fp16 -> fp32
    layer = GraphTransformerLayer(in_dim, heads=4).cuda().half()
    y = layer(x, graph)                                # x [n, in_dim] fp16

The drop-in launch is also a registered torch operator, on the block-sparse
form held in torch tensors (no plan, no state between calls):

    offs, bcol, mask = to_block_sparse(row_ptr, col_idx)        # GPU converter
    o = torch.ops.fused3s.attention_fwd(q, k, v, offs, bcol, mask, order, scale)
"""
from __future__ import annotations

import numpy as np
import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

# torch ships its own HIP runtime (torch/lib/libamdhip64.so, soname
# libamdhip64.so.7).  libf3s_hip.so binds to whichever libamdhip64.so.7 the
# process loaded first, so torch must be imported before the library's first
# GPU call; loaded the other way round, the process holds two HIP runtimes
# and torch sees no device.  Refuse that state with a clear message.


def _hip_runtimes() -> set[str]:
    try:
        with open("/proc/self/maps") as f:
            return {line.split()[-1] for line in f if "libamdhip64" in line}
    except OSError:
        return set()


if len(_hip_runtimes()) > 1:
    raise ImportError("two HIP runtimes are loaded (" + ", ".join(sorted(_hip_runtimes())) +
                      "): import torch before the first fused3s_amd GPU call")

import ctypes as C

from . import _lib
from .attention import Plan
from .device import DeviceArray, Stream, check
from .graph import (DeviceBSF, DeviceCSR, convert_device, converts_once, lists_oversized,
                    most_tiles, window_order_device)

HEAD_DIM = 64


class _TorchStream(Stream):
    """torch's current HIP stream, viewed as a library Stream (not owned)."""

    def __init__(self, handle: int):   # noqa: D107 -- no stream is created
        self.handle = handle

    def __del__(self):
        pass


def current_stream() -> Stream:
    return _TorchStream(torch.cuda.current_stream().cuda_stream)


def _on_device(t, s: Stream) -> DeviceArray:
    """An int32 copy of an index array in library memory: from host memory, or
    device to device when it is a tensor of an index type on the current device
    already."""
    if torch.is_tensor(t):
        if (t.is_cuda and t.device.index == torch.cuda.current_device()
                and t.dtype in (torch.int32, torch.int64)):
            t = t.to(torch.int32).contiguous()
            a = DeviceArray(tuple(t.shape), np.int32)
            if a.nbytes:
                check(_lib.hip().f3s_memcpy_d2d(a.ptr, t.data_ptr(), a.nbytes, s.handle),
                      "f3s_memcpy_d2d")
            return a
        t = t.cpu().numpy()
    return DeviceArray.from_numpy(np.ascontiguousarray(t, np.int32), s)


def _device_csr(row_ptr, col_idx, s: Stream) -> DeviceCSR:
    csr = DeviceCSR.__new__(DeviceCSR)
    csr.row_ptr, csr.col_idx = _on_device(row_ptr, s), _on_device(col_idx, s)
    csr.n = csr.row_ptr.shape[0] - 1
    csr.nnz = csr.col_idx.shape[0]
    return csr


class TorchGraph:
    """A graph prepared once for repeated fused passes: CSR on the device,
    block-sparse form with row masks (GPU converter), descending-workload
    window order, and a compiled plan for `heads` heads of 64 dims.  A small
    graph's block-sparse lists keep the memory of a tile per edge (19 MB at most)."""

    def __init__(self, row_ptr, col_idx, heads: int = 1, masked: bool = True):
        if not torch.cuda.is_available():
            raise RuntimeError("TorchGraph needs a ROCm device (no CPU fallback)")
        s = current_stream()
        self.csr = _device_csr(row_ptr, col_idx, s)
        self.n = self.csr.n
        self.nnz = self.csr.nnz
        self.heads = heads
        self.masked = masked
        self.bsf: DeviceBSF = convert_device(self.csr, masks=True, stream=s)
        self.order = window_order_device(self.bsf, s)
        self.plan = Plan(self.bsf, self.order, H=heads, stream=s)
        if masked:
            self.plan.compile(s)

    def attention(self, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                  scale: float = 1.0, out: torch.Tensor | None = None) -> torch.Tensor:
        """softmax over each node's neighbours of scale * q.k, weights applied
        to v; [n, H, 64] fp16 contiguous CUDA tensors in, [n, H, 64] fp32 out.
        masked=False gives the reference's tile-dense semantics instead."""
        n, H = self.n, self.heads
        shape = (n, H, HEAD_DIM)
        for name, t in (("q", q), ("k", k), ("v", v)):
            if t.requires_grad:
                raise RuntimeError("the fused pass is forward-only (no autograd)")
            if t.dtype is not torch.float16 or not t.is_cuda or not t.is_contiguous():
                raise ValueError(f"{name} must be a contiguous float16 CUDA tensor")
            if t.shape != shape and t.shape != (n, H * HEAD_DIM):   # (a Size is a tuple)
                raise ValueError(f"{name} must have shape {shape}, got {tuple(t.shape)}")
        if out is None:
            out = torch.empty(shape, dtype=torch.float32, device=q.device)
        elif (out.dtype != torch.float32 or not out.is_contiguous()
              or out.numel() != n * H * HEAD_DIM):
            raise ValueError("out must be a contiguous float32 tensor of n * H * 64 elements")
        # Plan.forward without its wrappers: a small graph's pass is shorter
        # than the Python around it
        bsf = self.bsf
        check(_lib.hip().f3s_attention_fwd_planned(
            self.plan.handle, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
            bsf.block_col.ptr, bsf.tile_mask.ptr if self.masked else None, n, HEAD_DIM, H, scale,
            torch.cuda.current_stream().cuda_stream), "f3s_attention_fwd_planned")
        return out

    def takes_packed(self) -> bool:
        """Whether attention_packed takes this graph: masked semantics, and
        the packed tensor within the 32-bit offsets of its launch."""
        return self.masked and 3 * self.n * self.heads * 2 * HEAD_DIM <= 0xffff4000

    def attention_packed(self, qkv: torch.Tensor, scale: float = 1.0,
                         dtype: torch.dtype = torch.float32) -> torch.Tensor:
        """attention() on the [n, 3 * H * 64] fp16 output of one projection
        (q, k and v side by side in each row, no copies made), O [n, H, 64]
        in float32 or float16 (f3s_attention_fwd_packed)."""
        if qkv.requires_grad:
            raise RuntimeError("the fused pass is forward-only (no autograd)")
        if qkv.dtype != torch.float16 or not qkv.is_cuda or not qkv.is_contiguous():
            raise ValueError("qkv must be a contiguous float16 CUDA tensor")
        if tuple(qkv.shape) != (self.n, 3 * self.heads * HEAD_DIM):
            raise ValueError(f"qkv must have shape {(self.n, 3 * self.heads * HEAD_DIM)}, "
                             f"got {tuple(qkv.shape)}")
        if dtype not in (torch.float32, torch.float16):
            raise ValueError("dtype must be float32 or float16")
        out = torch.empty((self.n, self.heads, HEAD_DIM), dtype=dtype, device=qkv.device)
        if self.n:
            check(_lib.hip().f3s_attention_fwd_packed(
                self.plan.handle, qkv.data_ptr(), out.data_ptr(), int(dtype == torch.float16),
                self.n, HEAD_DIM, self.heads, float(scale),
                torch.cuda.current_stream().cuda_stream), "f3s_attention_fwd_packed")
        return out


_LINEAR_FORWARD, _LINEAR = torch.nn.Linear.forward, torch.nn.functional.linear


def _watched() -> bool:
    """Whether something sees, replaces or transforms torch's calls: compilation
    and tracing, autocast, dispatch modes, function modes (torch.device's own
    does neither), functorch's transforms, forward-mode differentiation (which
    no_grad leaves on)."""
    if torch.compiler.is_compiling():
        return True
    c = torch._C
    modes = c._len_torch_function_stack()
    return (c._len_torch_dispatch_stack() > 0
            or modes > 0 and any(type(c._get_function_stack_at(i)) is not DeviceContext
                                 for i in range(modes))
            or torch.is_autocast_enabled() or forward_ad._current_level >= 0
            or c._functorch.peek_interpreter_stack() is not None or torch.jit.is_tracing())


def _is_plain_linear(m: torch.nn.Module) -> bool:
    """A torch.nn.Linear whose call is its product and nothing else."""
    hooks = torch.nn.modules.module
    return (type(m) is torch.nn.Linear and "forward" not in m.__dict__
            and torch.nn.Linear.forward is _LINEAR_FORWARD
            and torch.nn.functional.linear is _LINEAR
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks
                     or m._backward_pre_hooks or hooks._global_forward_hooks
                     or hooks._global_forward_pre_hooks or hooks._global_backward_hooks
                     or hooks._global_backward_pre_hooks))


def _project(m: torch.nn.Module, x: torch.Tensor, watched: bool) -> torch.Tensor:
    """m(x), by f3s_linear_f16 where that is the same thing: a plain fp16
    Linear of a contiguous fp16 matrix on its own device, in sizes the kernel
    takes, where nothing watches the call (_watched).  (Called without autograd.)  Below
    64 K rows of more than 128 inputs and outputs the library's tiles are the
    better ones (20,011 x 256 -> 768: 17 against 28 us; -> 128: 8 against 9,
    and half the call's host time)."""
    if (not watched and type(x) is torch.Tensor and x.dim() == 2 and x.is_cuda
            and x.dtype is torch.float16 and x.is_contiguous() and x.shape[0] > 0
            and _is_plain_linear(m)):
        w, b = m.weight, m.bias
        M, K = w.shape
        if (K % 8 == 0 and K <= 256 and M % 32 == 0 and M <= 32768 and x.shape[1] == K
                and (K <= 128 or M <= 128 or x.shape[0] >= 65536)
                and w.dtype is torch.float16 and w.device == x.device and w.is_contiguous()
                and type(w) is torch.nn.Parameter
                and (b is None or (b.dtype is torch.float16 and b.device == x.device
                                   and b.is_contiguous()))
                and (x.data_ptr() | w.data_ptr()) % 16 == 0
                and x.device.index == torch.cuda.current_device()):
            y = torch.empty((x.shape[0], M), dtype=torch.float16, device=x.device)
            check(_lib.hip().f3s_linear_f16(
                x.data_ptr(), w.data_ptr(), b.data_ptr() if b is not None else None,
                y.data_ptr(), x.shape[0], K, M, torch.cuda.current_stream().cuda_stream),
                "f3s_linear_f16")
            return y
    return m(x)


_ATTENTION = TorchGraph.attention


def _is_plain_graph(graph) -> bool:
    """Whether attention_packed stands for graph.attention: not where a
    program brings an attention of its own, in a subclass, on the graph or in
    the place of TorchGraph's."""
    return (isinstance(graph, TorchGraph) and type(graph).attention is _ATTENTION
            and "attention" not in graph.__dict__)


class GraphTransformerLayer(torch.nn.Module):
    """x -> [Q K V] = x W_qkv -> fused edge attention per head -> concat ->
    W_o, forward only.  Compute dtype of the projections is the module's
    (fp16 after .half()); attention accumulates and returns fp32, which is
    cast back to the projection dtype before W_o."""

    def __init__(self, in_dim: int, heads: int = 1, out_dim: int | None = None,
                 bias: bool = True):
        super().__init__()
        self.heads = heads
        self.qkv = torch.nn.Linear(in_dim, 3 * heads * HEAD_DIM, bias=bias)
        self.proj = torch.nn.Linear(heads * HEAD_DIM, out_dim or in_dim, bias=bias)
        self.scale = HEAD_DIM ** -0.5

    @torch.no_grad()
    def forward(self, x: torch.Tensor, graph: TorchGraph) -> torch.Tensor:
        if graph.heads != self.heads:
            raise ValueError("graph was planned for a different head count")
        n = x.shape[0]
        watched = _watched()
        qkv = _project(self.qkv, x, watched).to(torch.float16)
        dtype = self.proj.weight.dtype
        if _is_plain_graph(graph) and graph.takes_packed() and qkv.dim() == 2 \
                and qkv.is_contiguous():
            # the pass reads q, k and v where the projection wrote them, and
            # writes O in the dtype the output projection takes
            o = graph.attention_packed(qkv, self.scale,
                                       dtype if dtype == torch.float16 else torch.float32)
        else:
            qkv = qkv.view(n, 3, self.heads, HEAD_DIM)
            q, k, v = (qkv[:, i].contiguous() for i in range(3))
            o = graph.attention(q, k, v, scale=self.scale)
        return _project(self.proj, o.view(n, self.heads * HEAD_DIM).to(dtype), watched)


# ------------------------------------------------------------------ operator

def _cuda_i32(t, what: str) -> torch.Tensor:
    """An int32 CUDA copy (or view) of an integer array; int64 input (the
    usual index type of torch graph code) is narrowed after a range check."""
    t = torch.as_tensor(t)
    if t.dtype == torch.int64:
        if t.numel() and (int(t.min()) < -2**31 or int(t.max()) >= 2**31):
            raise ValueError(f"{what} holds values outside the int32 range")
        t = t.to(torch.int32)
    elif t.dtype != torch.int32:
        raise ValueError(f"{what} must hold int32 (or int64) values")
    if not t.is_cuda:
        t = t.to("cuda")
    return t.contiguous()


def to_block_sparse(row_ptr, col_idx, masks: bool = True):
    """convert_csr_to_block_sparse (src/converter.cu:13-44) on the GPU into
    torch tensors: (window_offsets int32 [W + 1], block_col_indices int32
    [T], tile_mask int16 [T, 16] -- bit c of row r of a tile set iff that
    edge exists -- or None).  Two calls of f3s_convert_csr_to_bsf on torch's
    current stream, the count (one host round trip for T), then the fill; or,
    on small graphs, one call for both, whose lists are then views of storage
    for at most four times their entries, or 4 MB more (lists_oversized)."""
    rp = _cuda_i32(row_ptr, "row_ptr")
    ci = _cuda_i32(col_idx, "col_idx")
    n = rp.numel() - 1
    if n < 0:
        raise ValueError("row_ptr must hold n + 1 entries")
    W = (n + 15) // 16
    lib = _lib.hip()
    s = torch.cuda.current_stream().cuda_stream
    offs = torch.empty(W + 1, dtype=torch.int32, device=rp.device)
    T = C.c_int64(0)
    cptr = ci.data_ptr() if ci.numel() else None
    if converts_once(n, ci.numel()):
        most = most_tiles(n, ci.numel())
        bcol = torch.empty(most, dtype=torch.int32, device=rp.device)
        mask = torch.empty((most, 16), dtype=torch.int16, device=rp.device) if masks else None
        check(lib.f3s_convert_csr_to_bsf_once(
            rp.data_ptr(), cptr, n, ci.numel(), offs.data_ptr(), bcol.data_ptr(),
            mask.data_ptr() if masks else None, C.byref(T), s), "f3s_convert_csr_to_bsf_once")
        t = int(T.value)
        bcol, mask = bcol[:t], (mask[:t] if masks else None)
        if lists_oversized(t, most):
            bcol, mask = bcol.clone(), (mask.clone() if masks else None)
        return offs, bcol, mask
    check(lib.f3s_convert_csr_to_bsf(rp.data_ptr(), cptr, n, ci.numel(), offs.data_ptr(), None,
                                     None, C.byref(T), s), "f3s_convert_csr_to_bsf(count)")
    t = int(T.value)
    # at least one element each, so the fill call gets real pointers
    bcol = torch.empty(max(t, 1), dtype=torch.int32, device=rp.device)
    mask = torch.empty((max(t, 1), 16), dtype=torch.int16, device=rp.device) if masks else None
    T2 = C.c_int64(0)
    check(lib.f3s_convert_csr_to_bsf(rp.data_ptr(), cptr, n, ci.numel(), offs.data_ptr(),
                                     bcol.data_ptr(), mask.data_ptr() if masks else None,
                                     C.byref(T2), s), "f3s_convert_csr_to_bsf(fill)")
    return offs, bcol[:t], (mask[:t] if masks else None)


def _check_operands(q, k, v, window_offsets, block_col, tile_mask, window_order):
    if q.dim() != 3 or q.shape[2] != HEAD_DIM:
        raise ValueError(f"q must be [n, H, {HEAD_DIM}]")
    n, H = q.shape[0], q.shape[1]
    for name, t in (("q", q), ("k", k), ("v", v)):
        if t.dtype != torch.float16 or not t.is_cuda or not t.is_contiguous():
            raise ValueError(f"{name} must be a contiguous float16 CUDA tensor")
        if tuple(t.shape) != (n, H, HEAD_DIM):
            raise ValueError(f"{name} must have shape {(n, H, HEAD_DIM)}, got {tuple(t.shape)}")
    W = (n + 15) // 16
    for name, t, shape in (("window_offsets", window_offsets, (W + 1,)),
                           ("block_col", block_col, None),
                           ("window_order", window_order, (W,))):
        if t is None:
            if name != "window_order":
                raise ValueError(f"{name} is required")
            continue
        if t.dtype != torch.int32 or not t.is_cuda or not t.is_contiguous() or t.dim() != 1:
            raise ValueError(f"{name} must be a contiguous 1-d int32 CUDA tensor")
        if shape is not None and tuple(t.shape) != shape:
            raise ValueError(f"{name} must have shape {shape}, got {tuple(t.shape)}")
    if tile_mask is not None:
        if (tile_mask.dtype not in (torch.int16, torch.uint16) or not tile_mask.is_cuda
                or not tile_mask.is_contiguous()
                or tuple(tile_mask.shape) != (block_col.shape[0], 16)):
            raise ValueError("tile_mask must be a contiguous [T, 16] int16 CUDA tensor")
    return n, H, W


@torch.library.custom_op("fused3s::attention_fwd", mutates_args=())
def attention_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor,
                  window_offsets: torch.Tensor, block_col: torch.Tensor,
                  tile_mask: torch.Tensor | None, window_order: torch.Tensor | None,
                  scale: float = 1.0) -> torch.Tensor:
    """f3s_attention_fwd (the reference's launch, tests/test_fused_3s_v2.cu:
    124-131, every window whole) on torch tensors and torch's current
    stream: q/k/v [n, H, 64] float16, the block-sparse form of
    to_block_sparse, window_order int32 [W] or None (natural order); a
    tile_mask gives the masked (edge-exact) semantics, None the reference's
    tile-dense one.  Returns O [n, H, 64] float32."""
    if q.requires_grad or k.requires_grad or v.requires_grad:
        raise RuntimeError("the fused pass is forward-only (no autograd)")
    n, H, W = _check_operands(q, k, v, window_offsets, block_col, tile_mask, window_order)
    out = torch.empty((n, H, HEAD_DIM), dtype=torch.float32, device=q.device)
    if n == 0:
        return out
    s = torch.cuda.current_stream(q.device).cuda_stream
    # an empty block_col tensor may have no storage: the C-ABI wants a pointer
    # whenever W > 0, and with T = 0 no tile is read through it
    bptr = block_col.data_ptr() or window_offsets.data_ptr()
    mptr = None
    if tile_mask is not None:
        mptr = tile_mask.data_ptr() or out.data_ptr()
    check(_lib.hip().f3s_attention_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
                                       window_offsets.data_ptr(), bptr, mptr,
                                       window_order.data_ptr() if window_order is not None
                                       else None, W, n, HEAD_DIM, H, float(scale), s),
          "f3s_attention_fwd")
    return out


@attention_fwd.register_fake
def _attention_fwd_fake(q, k, v, window_offsets, block_col, tile_mask, window_order, scale=1.0):
    return torch.empty(q.shape, dtype=torch.float32, device=q.device)
