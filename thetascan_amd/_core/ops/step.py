"""A decode step of the depth-1 kernel memory with the plain sum.

``kernel_step`` continues a carried state by at most eight tokens per
sequence in three launches: the stacked projections (ts_skinny_linear for few
bf16 rows, else library GEMMs), everything between the projections
(ts_memory_step: features, recurrence, read, output gate) and the output
projection.  Same mathematics as the multi-view path that longer
continuations take (block.py:595-618, engine.py:117-158, 426-544).
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn.functional as F

from ... import _lib
from . import fused, stream
from .linear import keeps_dtype

MAX_TOKENS = 8
WIDTHS = (16, 32, 64, 128)
SKINNY_ROWS = 64


def eligible(x: torch.Tensor, spec, head_dim: int, params) -> bool:
    """Whether ts_memory_step takes this continuation: few tokens, widths of
    the kernel, the input as wide as the projection's rows (``params[0]``; any
    other width is refused by the multi-view path's product), and every
    parameter a contiguous tensor beside the input and of its dtype, which the
    projections keep (the kernel's rows are of one dtype: under an autocast to
    another the multi-view path follows the projection)."""
    dtype, device = x.dtype, x.get_device()
    _, T, D = x.shape
    if not (x.is_cuda and (dtype == torch.bfloat16 or dtype == torch.float32) and 1 <= T <= MAX_TOKENS
            and spec.m in WIDTHS and head_dim in WIDTHS and spec.m >= head_dim and D == params[0].shape[1]
            and keeps_dtype(dtype)):
        return False
    for p in params:
        if p is not None and not (p.dtype == dtype and p.get_device() == device and p.is_contiguous()
                                  and p.data_ptr() % 16 == 0):
            return False
    return True


def _linear(x2: torch.Tensor, wa: torch.Tensor, wb: torch.Tensor | None) -> torch.Tensor:
    """x2 [n,k] times [wa; wb]^T.  Up to 64 bf16 rows take ts_skinny_linear:
    a library GEMM of so few rows is all latency (B8, 512 -> 1536 and 512:
    4.8 us each against 3.7 us for both, with no concatenated weight)."""
    n, k = x2.shape
    row, col = x2.stride()
    na, ka = wa.shape
    nb, kb = (0, k) if wb is None else wb.shape
    # (a weight of another row length is the library product's to refuse: the
    # kernel reads k elements of every row; rows of other strides, which a
    # reshape leaves as they are, are its to read)
    if not (x2.dtype == torch.bfloat16 and n <= SKINNY_ROWS and ka == k and kb == k and k % 32 == 0 and na % 16 == 0
            and nb % 16 == 0 and col == 1 and row % 8 == 0 and x2.data_ptr() % 16 == 0):
        parts = [F.linear(x2, w) for w in (wa, wb) if w is not None]
        return parts[0] if wb is None else torch.cat(parts, dim=1)
    y = torch.empty(n, na + nb, dtype=x2.dtype, device=x2.device)
    status = _lib.load().ts_skinny_linear(x2.data_ptr(), n, k, row, wa.data_ptr(), na, _lib.ptr(wb), nb, y.data_ptr(),
                                          na + nb, _lib.stream_handle(x2.device))
    _lib.check(status, "ts_skinny_linear")
    return y


def kernel_step(x: torch.Tensor, w_qkv, w_g, b_g, w1, w2, tau, w_out, spec, normalize: bool, heads: int) -> torch.Tensor:
    """``y`` [B,T,D] of the next T tokens; the active carry's state is read and
    its successor left on the carry (in place for a captured step)."""
    carry = stream.active()
    B, T, D = x.shape
    H = heads
    d = w_qkv.shape[0] // (3 * H)
    dev, dt = x.device, x.dtype
    blocks = carry.take()
    cols = d + int(normalize)
    init = None
    if blocks is not None:
        # (as scan_launch takes a carried state)
        if (len(blocks) != 1 or blocks[0].shape[-2:] != (spec.m, cols)
                or blocks[0].numel() != B * H * spec.m * cols):
            raise ValueError("streaming state does not match this scan's widths")
        init = blocks[0].detach().to(device=dev, dtype=torch.float32).contiguous()
    if blocks is not None and stream.updates_in_place():
        fin = blocks[0]
        if fin.dtype != torch.float32 or not fin.is_contiguous() or fin.device != dev:
            raise ValueError("a state updated in place must be a contiguous fp32 tensor beside the input")
    else:
        fin = torch.empty(B, H, spec.m, cols, dtype=torch.float32, device=dev)
    proj = _linear(x.reshape(B * T, D), w_qkv, w_g)
    P = proj.shape[1]
    y = torch.empty(B * T, H * d, dtype=dt, device=dev)
    view = lambda t, col, width: _lib.Strided(t.data_ptr() + col * t.element_size(), T * width, d, width)  # noqa: E731
    hd = H * d
    pos = stream.device_position()
    inv = [fused.inverse_frequencies(rot, spec.rope_base, dev) if rot else None for rot in (spec.in_rot, spec.feat_rot)]
    code = _lib.dtype_code(dt)
    desc = _lib.MemoryStepDesc(B, H, T, d, spec.m, code, code, spec.kind, spec.in_rot, spec.feat_rot, int(normalize),
                               int(w_g is not None), float(spec.gain), float(spec.resid_scale), float(spec.eps),
                               0 if pos is not None else carry.position)
    io = _lib.MemoryStepIO(
        view(proj, 0, P), view(proj, hd, P), view(proj, 2 * hd, P),
        view(proj, 3 * hd, P) if w_g is not None else _lib.strided(None), view(y, 0, hd),
        w1.data_ptr(), w2.data_ptr(), _lib.ptr(tau), _lib.ptr(b_g), _lib.ptr(inv[0]), _lib.ptr(inv[1]), _lib.ptr(pos),
        _lib.ptr(init), fin.data_ptr())
    lib = _lib.load()
    with _lib.timed("ts_memory_step", lambda: _lib.nbytes(proj, y, w1, w2, init, fin)):
        status = lib.ts_memory_step(ctypes.byref(desc), ctypes.byref(io), _lib.stream_handle(dev))
    _lib.check(status, "ts_memory_step")
    carry.put([fin])
    return _linear(y, w_out, None).view(B, T, w_out.shape[0])
