"""Causal softmax attention without a backward (ts_causal_attention_fwd).

The hybrid language model's softmax layers are torch's fused attention in
training; where nothing is recorded (evaluation, generation) heads of 64 in
bf16 run one HIP launch that reads grouped key/value heads and the
projections' token-major rows in place.
"""
from __future__ import annotations

import ctypes

import torch

from ... import _lib
from . import rownorm


def supported(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> bool:
    """Whether :func:`causal_attention` takes these (a host query): bf16
    [B,H,T,64] queries and [B,Hkv,T,64] keys and values on one GPU with
    16-byte aligned rows, Hkv dividing H, and no gradient to record."""
    tensors = (q, k, v)
    if torch.compiler.is_compiling() or (torch.is_grad_enabled() and any(t.requires_grad for t in tensors)):
        return False
    if not all(t.is_cuda and t.device == q.device and t.ndim == 4 and t.dtype == torch.bfloat16 for t in tensors):
        return False
    B, H, T, d = q.shape
    if d != 64 or k.shape != v.shape or k.shape[0] != B or k.shape[2:] != (T, d) or q.numel() == 0 or k.numel() == 0:
        return False
    return H % k.shape[1] == 0 and T <= 65535 * 128 and all(
        t.stride(-1) == 1 and t.data_ptr() % 16 == 0 and all(s % 8 == 0 for s in t.stride()[:3]) for t in tensors)


def causal_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """softmax(q k^T / 8, causal) v, [B,H,T,64] in the query's memory order."""
    lib = _lib.load()
    B, H, T, d = q.shape
    out = rownorm._like(q)
    desc = _lib.AttentionDesc(B, H, k.shape[1], T, d, _lib.dtype_code(q.dtype), d ** -0.5)
    with _lib.timed("ts_causal_attention_fwd", lambda: _lib.nbytes(q, k, v, out)):
        status = lib.ts_causal_attention_fwd(ctypes.byref(desc), _lib.strided(q), _lib.strided(k), _lib.strided(v),
                                             _lib.strided(out), _lib.stream_handle(q.device))
    _lib.check(status, "ts_causal_attention_fwd")
    return out
