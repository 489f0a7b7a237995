"""A temporal bank's reads, blend and output gate as one autograd node.

``bank_read(nums, masses, resids, coef, gate, gate_bias)`` returns

    y = (sum_j coef[j,h] (resid_j + s num_j / (mass_j + eps))) * silu(gate + gate_bias)

(engine.py:440-442, 526-528; block.py:683-722; gates.py:34-40) from
ts_bank_read_fwd, written token-major: a [B,H,T,d] view of [B,T,H,d] memory,
which the output projection reads as [B,T,H*d] without a copy.  The backward
is one ts_bank_read_bwd launch for every gradient.
"""
from __future__ import annotations

import ctypes

import torch

from ... import _lib
from .dispatch import HipOp
from .linear import slot_sum


def eligible(nums, masses, resids, heads: int) -> bool:
    """Whether ts_bank_read takes these views: 1 to 8 of them, of one shape
    and dtype (bf16 or fp32) on the GPU, in rows of at most 512 bytes, with
    one residual of that dtype for all of them or one each."""
    n, first = len(nums), nums[0]
    if not 1 <= n <= _lib.BANK_MAX or not first.is_cuda or first.ndim != 4:
        return False
    if first.dtype not in (torch.bfloat16, torch.float32) or len(resids) not in (1, n):
        return False
    B, H, _, d = first.shape
    row = d * first.element_size()
    if H != heads or row % 16 or row > 512 or B * H > 65535:
        return False
    return (all(t.shape == first.shape and t.dtype == first.dtype for t in (*nums, *resids))
            and all((m is None) == (masses[0] is None) for m in masses))


def check_gate(gate: torch.Tensor | None, num: torch.Tensor) -> None:
    """Raise unless ``gate`` has the rows that a read epilogue of ``num`` reads."""
    if gate is not None and (gate.dtype != num.dtype or gate.shape != num.shape or gate.device != num.device):
        raise ValueError(f"the output gate's pre-activation ({gate.dtype}, {tuple(gate.shape)}, {gate.device}) does not "
                         f"match the reads ({num.dtype}, {tuple(num.shape)}, {num.device})")


def _rows(t: torch.Tensor) -> torch.Tensor:
    vec = 16 // t.element_size()
    ok = t.stride(-1) == 1 and t.data_ptr() % 16 == 0 and all(s % vec == 0 for s in t.stride()[:3])
    return t if ok else t.contiguous()


def _strides(ts):
    return (_lib.Strided * _lib.BANK_MAX)(*[_lib.strided(t) for t in ts])


def _call(nums, masses, resids, coef, gate, gate_bias, s, eps):
    """(desc, io, the tensors the io points at)."""
    B, H, T, d = nums[0].shape
    nk, rk = [_rows(t) for t in nums], [_rows(t) for t in resids]
    mk = [m.detach().to(torch.float32) for m in masses]
    cf = coef.detach().to(torch.float32).contiguous()
    gk = None if gate is None else _rows(gate)
    gb = None if gate_bias is None else gate_bias.detach().to(torch.float32).contiguous()
    desc = _lib.BankReadDesc(B, H, T, d, len(nk), len(rk), _lib.dtype_code(nk[0].dtype), int(bool(mk)),
                             int(gk is not None), float(s), float(eps))
    io = _lib.BankReadIO(_strides(nk), _strides(mk), _strides(rk), _lib.strided(gk), cf.data_ptr(), _lib.ptr(gb))
    return desc, io, (nk, mk, rk, cf, gk, gb)


def _forward(nums: list[torch.Tensor], masses: list[torch.Tensor], resids: list[torch.Tensor], coef: torch.Tensor,
             gate: torch.Tensor | None, gate_bias: torch.Tensor | None, s: float, eps: float) -> torch.Tensor:
    lib = _lib.load()
    # (every converted operand stays bound until the launch: a dropped one's
    # memory could become y's)
    desc, io, kept = _call(nums, masses, resids, coef, gate, gate_bias, s, eps)
    nk, mk, rk, _, gk, _ = kept
    B, H, T, d = nk[0].shape
    y = torch.empty(B, T, H, d, dtype=nk[0].dtype, device=nk[0].device).transpose(1, 2)
    with _lib.timed("ts_bank_read_fwd", lambda: _lib.nbytes(*nk, *mk, *rk, gk, y)):
        status = lib.ts_bank_read_fwd(ctypes.byref(desc), ctypes.byref(io), _lib.strided(y),
                                      _lib.stream_handle(y.device))
    _lib.check(status, "ts_bank_read_fwd")
    return y


def _fake(nums, masses, resids, coef, gate, gate_bias, s, eps):
    B, H, T, d = nums[0].shape
    return nums[0].new_empty(B, T, H, d).transpose(1, 2)


def _backward_impl(dy: torch.Tensor, nums: list[torch.Tensor], masses: list[torch.Tensor],
                   resids: list[torch.Tensor], coef: torch.Tensor, gate: torch.Tensor | None,
                   gate_bias: torch.Tensor | None, s: float, eps: float, need: list[bool]) -> list[torch.Tensor]:
    lib = _lib.load()
    desc, io, (nk, mk, rk, cf, gk, gb) = _call(nums, masses, resids, coef, gate, gate_bias, s, eps)
    B, H, T, d = nk[0].shape
    n, dev, dt = len(nk), nk[0].device, nk[0].dtype
    need_resid, need_coef, need_bias = need
    g = _rows(dy.to(dt))
    dnum = [torch.empty(B, H, T, d, dtype=dt, device=dev) for _ in nk]
    dmass = [torch.empty(B, H, T, dtype=torch.float32, device=dev) for _ in mk]
    dres = [torch.empty(B, H, T, d, dtype=dt, device=dev) for _ in rk] if need_resid else []
    dg = None if gk is None else torch.empty(B, T, H, d, dtype=dt, device=dev).transpose(1, 2)
    parts = ctypes.c_int32()
    _lib.check(lib.ts_bank_read_parts(ctypes.byref(desc), ctypes.byref(parts)), "ts_bank_read_parts")
    cpart = torch.empty(parts.value, n, H, dtype=torch.float32, device=dev) if need_coef else None
    bpart = torch.empty(parts.value, H * d, dtype=torch.float32, device=dev) if need_bias else None
    grads = _lib.BankReadGrads(_lib.strided(g), _strides(dnum), _strides(dmass), _strides(dres), _lib.strided(dg),
                               _lib.ptr(cpart), _lib.ptr(bpart))
    with _lib.timed("ts_bank_read_bwd", lambda: _lib.nbytes(*nk, *mk, *rk, gk, g, *dnum, *dmass, *dres, dg)):
        status = lib.ts_bank_read_bwd(ctypes.byref(desc), ctypes.byref(io), ctypes.byref(grads),
                                      _lib.stream_handle(dev))
    _lib.check(status, "ts_bank_read_bwd")
    # absent gradients travel as placeholders (each its own: outputs of a custom op must not alias)
    dcoef = slot_sum(cpart, torch.float32, (n, H)).to(coef.dtype) if need_coef else dy.new_empty(0)
    dbias = slot_sum(bpart, gate_bias.dtype, gate_bias.shape) if need_bias else dy.new_empty(0)
    return (dnum + [x.to(m.dtype) for x, m in zip(dmass, masses)] + dres
            + [dcoef, dy.new_empty(0) if dg is None else dg, dbias])


def _backward_fake(dy, nums, masses, resids, coef, gate, gate_bias, s, eps, need):
    B, H, T, d = nums[0].shape
    return ([t.new_empty(t.shape) for t in nums] + [m.new_empty(m.shape) for m in masses]
            + ([t.new_empty(t.shape) for t in resids] if need[0] else [])
            + [coef.new_empty(coef.shape) if need[1] else dy.new_empty(0),
               dy.new_empty(0) if gate is None else dy.new_empty(B, T, H, d).transpose(1, 2),
               gate_bias.new_empty(gate_bias.shape) if need[2] else dy.new_empty(0)])


def _setup(ctx, inputs, output):
    nums, masses, resids, coef, gate, gate_bias, s, eps = inputs
    ctx.counts, ctx.args = (len(nums), len(masses), len(resids)), (s, eps)
    ctx.need = [any(r.requires_grad for r in resids), coef.requires_grad,
                gate is not None and gate_bias is not None and gate_bias.requires_grad]
    ctx.save_for_backward(*nums, *masses, *resids, coef, gate, gate_bias)


def _backward(ctx, dy, bwd):
    n, m, r = ctx.counts
    saved = list(ctx.saved_tensors)
    nums, masses, resids, (coef, gate, gate_bias) = saved[:n], saved[n:n + m], saved[n + m:n + m + r], saved[n + m + r:]
    need_resid, need_coef, need_bias = ctx.need
    res = list(bwd(dy, nums, masses, resids, coef, gate, gate_bias, *ctx.args, ctx.need))
    dnum, dmass, rest = res[:n], res[n:n + m], res[n + m:]
    dres = rest[:r] if need_resid else [None] * r
    dcoef, dg, db = rest[-3:]
    return (dnum, dmass, dres, dcoef if need_coef else None, None if gate is None else dg,
            db if need_bias else None, None, None)


_bank_read_op = HipOp("bank_read", forward=_forward, forward_fake=_fake, backward_impl=_backward_impl,
                      backward_fake=_backward_fake, setup=_setup, backward=_backward)


def bank_read(nums, masses, resids, coef: torch.Tensor, *, s: float = 1.0, eps: float = 1e-6,
              gate: torch.Tensor | None = None, gate_bias: torch.Tensor | None = None) -> torch.Tensor:
    """``nums`` [B,H,T,d] per view, ``masses`` fp32 [B,H,T] per view (None:
    an unnormalized read), ``resids`` one tensor for every view or one each,
    ``coef`` [n,H]; with ``gate`` (the [B,H,T,d] view of x W_g^T, the dtype of
    ``nums``) the output gate is applied too."""
    mass = [] if masses[0] is None else list(masses)
    check_gate(gate, nums[0])
    return _bank_read_op(list(nums), mass, list(resids), coef, gate, gate_bias, float(s), float(eps))


# ------------------------------------------------------------------ parameters

def params_eligible(alpha: torch.Tensor, eta: torch.Tensor, x_dtype: torch.dtype) -> bool:
    """Whether ts_bank_params forms this bank's retentions and blend."""
    return (alpha.is_cuda and alpha.shape == eta.shape and alpha.ndim == 2 and alpha.dtype == eta.dtype
            and alpha.dtype in (torch.bfloat16, torch.float32) and x_dtype in (torch.bfloat16, torch.float32)
            and 1 <= alpha.shape[0] < _lib.BANK_MAX)


def _params_desc(alpha, tanh_eta, stream_code):
    return _lib.BankParamsDesc(alpha.shape[0], alpha.shape[1], int(tanh_eta), _lib.dtype_code(alpha.dtype), stream_code)


def _ptrs(ts):
    return (ctypes.c_void_p * len(ts))(*[_lib.ptr(t) for t in ts])


def _params_forward(alpha: torch.Tensor, eta: torch.Tensor, tanh_eta: bool, stream_code: int) -> list[torch.Tensor]:
    lib = _lib.load()
    n, H = alpha.shape
    a, e = alpha.detach().contiguous(), eta.detach().contiguous()
    las = [torch.empty(H, dtype=torch.float32, device=a.device) for _ in range(n)]
    coef = torch.empty(n + 1, H, dtype=torch.float32, device=a.device)
    status = lib.ts_bank_params_fwd(ctypes.byref(_params_desc(a, tanh_eta, stream_code)), a.data_ptr(), e.data_ptr(),
                                    _ptrs(las), coef.data_ptr(), _lib.stream_handle(a.device))
    _lib.check(status, "ts_bank_params_fwd")
    return las + [coef]


def _params_fake(alpha, eta, tanh_eta, stream_code):
    n, H = alpha.shape
    return [alpha.new_empty(H, dtype=torch.float32) for _ in range(n)] + [
        alpha.new_empty(n + 1, H, dtype=torch.float32)]


def _params_backward_impl(grads: list[torch.Tensor], alpha: torch.Tensor, eta: torch.Tensor, tanh_eta: bool,
                          stream_code: int) -> list[torch.Tensor]:
    lib = _lib.load()
    a, e = alpha.detach().contiguous(), eta.detach().contiguous()
    # absent gradients travel as empty placeholders
    gs = [None if g.numel() == 0 else g.to(torch.float32).contiguous() for g in grads]
    da, de = torch.empty_like(a), torch.empty_like(e)
    status = lib.ts_bank_params_bwd(ctypes.byref(_params_desc(a, tanh_eta, stream_code)), a.data_ptr(), e.data_ptr(),
                                    _ptrs(gs[:-1]), _lib.ptr(gs[-1]), da.data_ptr(), de.data_ptr(),
                                    _lib.stream_handle(a.device))
    _lib.check(status, "ts_bank_params_bwd")
    return [da, de]


def _params_backward_fake(grads, alpha, eta, tanh_eta, stream_code):
    return [torch.empty_like(alpha), torch.empty_like(eta)]


def _params_setup(ctx, inputs, output):
    alpha, eta, *ctx.args = inputs
    ctx.save_for_backward(alpha, eta)


def _params_backward(ctx, grads, bwd):
    alpha, eta = ctx.saved_tensors
    da, de = bwd([alpha.new_empty(0) if g is None else g for g in grads], alpha, eta, *ctx.args)
    return da, de, None, None


_bank_params_op = HipOp("bank_params", forward=_params_forward, forward_fake=_params_fake,
                        backward_impl=_params_backward_impl, backward_fake=_params_backward_fake,
                        setup=_params_setup, backward=_params_backward)


def bank_params(alpha: torch.Tensor, eta: torch.Tensor, tanh_eta: bool, x_dtype: torch.dtype):
    """(log retentions [H] fp32 per branch, blend coefficients [n+1, H]) of a
    fast bank with parameters alpha, eta [n, H] (block.py:647-695) for streams
    of ``x_dtype``: one launch each way."""
    *las, coef = _bank_params_op(alpha, eta, bool(tanh_eta), _lib.dtype_code(x_dtype))
    return las, coef
