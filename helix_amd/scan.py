"""Torch-facing SSD scan operator over the HELIX C ABI.

The host-side mirror of what the reference's ggml bridge does for llama.cpp
(integration/ggml/ggml-helix.cpp:157-361): map tensors (sizes and element
strides) onto a helix_scan_desc, keep a context and a scratch buffer, and
enqueue on the caller's stream. PyTorch provides device memory and the stream
only; all arithmetic runs in the HIP kernels of libhelix.so.
"""
from __future__ import annotations

import contextlib
import math
import threading
from collections import OrderedDict
from ctypes import c_float

import torch

from .abi import ARGS_STRUCT, DESC_STRUCT, Context, HelixError
from .desc import (HELIX_A_SCALAR_PER_HEAD, HELIX_BACKEND_AUTO, HELIX_BACKEND_MPP, HELIX_BACKEND_SGMMA, HELIX_BF16,
                   HELIX_ERR_SCRATCH_TOO_SMALL, HELIX_ERR_UNSUPPORTED_SHAPE, HELIX_F16, HELIX_F32, HELIX_OK,
                   HELIX_TENSOR_NULL, HelixScanDesc, HelixTensor)

BACKENDS = {"auto": HELIX_BACKEND_AUTO, "fp32": HELIX_BACKEND_SGMMA, "sgmma": HELIX_BACKEND_SGMMA,
            "bf16": HELIX_BACKEND_MPP, "mpp": HELIX_BACKEND_MPP}
# Storage type of x, B, C and y (helix_scan_desc.io_dtype).
IO_DTYPES = {torch.float32: HELIX_F32, torch.bfloat16: HELIX_BF16, torch.float16: HELIX_F16}

_ctx_lock = threading.Lock()
_contexts: dict[int, Context] = {}
# Scratch is kept per thread, device and stream (the last SCRATCH_STREAMS that
# a thread used), grown monotonically: scans that may run at the same time must
# not share one. Each buffer is allocated under its own stream, so one that is
# replaced or dropped goes back to the allocator for later work of that stream
# only.
SCRATCH_STREAMS = 8
_scratch = threading.local()


def context(device: int) -> Context:
    with _ctx_lock:
        ctx = _contexts.get(device)
        if ctx is None:
            ctx = Context(device)
            _contexts[device] = ctx
        return ctx


def tensor_arg(t: torch.Tensor | None) -> HelixTensor:
    if t is None:
        return HELIX_TENSOR_NULL
    return HelixTensor(t.data_ptr(), 0)


def _scratch_for(device: int, st: int, nbytes: int, stream: torch.cuda.Stream | None = None) -> torch.Tensor | None:
    """This thread's scratch on the device for the stream of handle st, grown to nbytes (0: as it is). stream: the
    stream object where it may not be the current one."""
    pool = getattr(_scratch, "pool", None)
    if pool is None:
        pool = _scratch.pool = OrderedDict()
    key = (device, st)
    buf = pool.get(key)
    if buf is not None:
        pool.move_to_end(key)
    if nbytes and (buf is None or buf.numel() < nbytes):
        with _under(device, st, stream):
            buf = torch.empty(nbytes, dtype=torch.uint8, device=f"cuda:{device}")
        pool[key] = buf
        if len(pool) > SCRATCH_STREAMS:
            pool.popitem(last=False)
    return buf


def _capturing(device: int, st: int, stream) -> bool:
    with _under(device, st, stream):
        return torch.cuda.is_current_stream_capturing()


def _under(device: int, st: int, stream):
    """The context in which torch allocates for the stream."""
    if stream is None:
        return contextlib.nullcontext()
    if not isinstance(stream, torch.cuda.Stream):
        stream = torch.cuda.ExternalStream(st, device=device) if st else torch.cuda.default_stream(device)
    return torch.cuda.stream(stream)


def make_desc(x: torch.Tensor, dt: torch.Tensor, B: torch.Tensor, C: torch.Tensor,
              s: torch.Tensor, y: torch.Tensor, A: torch.Tensor, *, backend: str = "auto",
              multipass: bool = True, dt_min: float = 0.0, dt_max: float = math.inf) -> HelixScanDesc:
    """Descriptor from tensor shapes and element strides:
    x, y [S, L, H, P]; dt [S, L, H]; B, C [S, L, G, N]; s [S, H, P, N]; A [H]."""
    S, L, H, P = x.shape
    G, N = B.shape[2], B.shape[3]
    d = HelixScanDesc()
    d.n_tok, d.n_seq, d.n_head, d.head_dim, d.d_state, d.n_group = L, S, H, P, N, G
    sx, sy, sb, sc, sdt, ss = x.stride(), y.stride(), B.stride(), C.stride(), dt.stride(), s.stride()
    d.s_x[0], d.s_x[1], d.s_x[2], d.seq_x = sx[1], sx[2], sx[3], sx[0]
    d.s_y[0], d.s_y[1], d.s_y[2], d.seq_y = sy[1], sy[2], sy[3], sy[0]
    d.s_b[0], d.s_b[1], d.s_b[2], d.seq_b = sb[1], sb[2], sb[3], sb[0]
    d.s_c[0], d.s_c[1], d.s_c[2], d.seq_c = sc[1], sc[2], sc[3], sc[0]
    d.s_dt[0], d.s_dt[1], d.seq_dt = sdt[1], sdt[2], sdt[0]
    d.s_s[0], d.s_s[1], d.s_s[2], d.seq_s = ss[1], ss[2], ss[3], ss[0]
    d.s_a = A.stride(0)
    d.io_dtype = IO_DTYPES[x.dtype]
    d.chunk = 0
    d.backend = BACKENDS[backend]
    d.multipass = multipass
    d.dt_min = dt_min
    d.dt_max = dt_max
    return d


def ssd_scan(x: torch.Tensor, dt: torch.Tensor, A: torch.Tensor, B: torch.Tensor, C: torch.Tensor,
             s0: torch.Tensor | None = None, ids: torch.Tensor | None = None, *,
             backend: str = "auto", dt_min: float = 0.0, dt_max: float = math.inf,
             multipass: bool = True,
             y: torch.Tensor | None = None, s1: torch.Tensor | None = None,
             scratch: torch.Tensor | None = None, stream: torch.cuda.Stream | None = None):
    """Chunked SSD prefill scan on the MI355X kernels. Returns (y, s1).

    x [S,L,H,P], dt [S,L,H] (pre-softplus), A [H], B/C [S,L,G,N], s0 [S,H,P,N]
    (zeros when None), ids int32 [S] (source state row per sequence), on one
    gfx950 device. x, B, C and y are float32, bfloat16 or float16 (one type);
    dt, A and the states are float32. multipass=False runs the single-pass kernel (fp32,
    no scratch; backend "bf16" is then declined). Raises HelixError when the
    shape is declined.
    """
    dev = x.device
    if dev.type != "cuda":
        raise ValueError("ssd_scan runs on a HIP device; got " + str(dev))
    # x, B, C (and y) share one storage type: float32, bfloat16 or float16;
    # dt, A and the states are float32.
    if x.dtype not in IO_DTYPES:
        raise ValueError(f"x must be float32, bfloat16 or float16; got {x.dtype}")
    for name, t, want in (("x", x, x.dtype), ("dt", dt, torch.float32), ("A", A, torch.float32),
                          ("B", B, x.dtype), ("C", C, x.dtype)):
        if t.dtype != want or t.device != dev:
            raise ValueError(f"{name} must be {want} on {dev}")
    S, L, H, P = x.shape
    G, N = B.shape[2], B.shape[3]
    if y is None:
        y = torch.empty((S, L, H, P), dtype=x.dtype, device=dev)
    elif y.dtype != x.dtype:
        raise ValueError(f"y must be {x.dtype}")
    if s1 is None:
        s1 = torch.empty((S, H, P, N), dtype=torch.float32, device=dev)
    if ids is not None and (ids.dtype != torch.int32 or not ids.is_contiguous()):
        raise ValueError("ids must be a contiguous int32 tensor")
    # No s0: a zero state, of the dense strides, without a tensor of zeros.
    ss = s0.stride() if s0 is not None else (H * P * N, P * N, N, 1)
    if s1.stride() != ss:
        raise ValueError("s0 and s1 must share strides")
    sx, sy, sb, sc, sdt = x.stride(), y.stride(), B.stride(), C.stride(), dt.stride()
    fields = (L, S, H, P, N, G, sx[1], sx[2], sx[3], sb[1], sb[2], sb[3], sc[1], sc[2], sc[3], sdt[1], sdt[2],
              ss[1], ss[2], ss[3], sy[1], sy[2], sy[3], A.stride(0), sx[0], sb[0], sc[0], sdt[0], ss[0], sy[0],
              0, HELIX_A_SCALAR_PER_HEAD, IO_DTYPES[x.dtype], HELIX_F32, BACKENDS[backend], bool(multipass))
    try:
        d = DESC_STRUCT.pack(*fields, dt_min, dt_max)
    except OverflowError:   # a bound past float32's range
        d = DESC_STRUCT.pack(*fields, c_float(dt_min).value, c_float(dt_max).value)
    index = dev.index if dev.index is not None else torch.cuda.current_device()
    ctx = _contexts.get(index) or context(index)
    st = stream.cuda_stream if stream is not None else torch._C._cuda_getCurrentRawStream(index)
    lent = scratch
    # Work under capture gets memory of the graph's own, which no later call touches.
    capturing = lent is None and (torch.cuda.is_current_stream_capturing() if stream is None
                                  else _capturing(index, st, stream))
    if lent is None and not capturing:
        scratch = _scratch_for(index, st, 0)
    ptrs = (0 if s0 is None else s0.data_ptr(), x.data_ptr(), dt.data_ptr(), A.data_ptr(), B.data_ptr(), C.data_ptr(),
            0 if ids is None else ids.data_ptr(), y.data_ptr(), s1.data_ptr())
    while True:
        have = 0 if scratch is None else scratch.numel() * scratch.element_size()
        rc, need = ctx.run(st, d, ARGS_STRUCT.pack(*ptrs, 0 if scratch is None else scratch.data_ptr(), have))
        if rc != HELIX_ERR_SCRATCH_TOO_SMALL or have >= need:
            break
        if lent is not None:
            # 16-bit storage on the fp32 path does without where it is lent too little.
            rc, _ = ctx.run(st, d, ARGS_STRUCT.pack(*ptrs, 0, need))
            if rc == HELIX_ERR_SCRATCH_TOO_SMALL:
                raise ValueError(f"scratch needs {need} bytes")
            break
        if capturing:
            with _under(index, st, stream):
                scratch = torch.empty(need, dtype=torch.uint8, device=dev)
        else:
            scratch = _scratch_for(index, st, need, stream)
    if rc == HELIX_ERR_UNSUPPORTED_SHAPE:
        raise HelixError(1, f"shape declined: {ctx.backend_desc(HelixScanDesc.from_buffer_copy(d))}")
    if rc != HELIX_OK:
        raise HelixError(rc, ctx.last_error())
    return y, s1
