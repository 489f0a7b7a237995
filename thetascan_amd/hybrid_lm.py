"""A ~17M-parameter hybrid language model around two ThetaScan mixers, and
the per-row symmetric int8 round trip of its weights.

This is the host model of the reference's language-model benchmark harness
(benchmarks/parameter-golf/prepare_harness.py:613-741 patches it into an
upstream training script that is not part of the reference): a 9-layer
decoder, d_model 512, vocabulary 1024, tied embeddings with a tanh logit
soft-cap, U-net skip connections between the first and last blocks, and
blocks that mix the running residual with the embedding (``resid_mix``)
before an attention (or ThetaScan) mixer and a ReLU^2 MLP.  The attention
layers are grouped-query (8 query heads, 4 key/value heads) with RMS-normed
queries and keys, RoPE and a per-head query gain.  Layers 4 and 5 swap
attention for ThetaScan-Kernel memories (the ReLU^2 ridge of
``kernel_expanded_reference_v0_1`` at m = 128 = 2 x 64 by random feature
expansion, grouped key/value projections), and their FFNs are trimmed so that
the parameter count follows the count contract of
tests/test_projection_layouts.py:101-113 (baseline 17,059,912 parameters,
attention mixer 786,440, FFN hidden 1024).

The upstream script is not available, so this model is defined here from
those facts; its int8 round trip has no reference numbers to match.
"""
from __future__ import annotations

import dataclasses

import torch
import torch.nn as nn
import torch.nn.functional as F

from ._core.ops import attention as hip_attention, rowglue, rownorm
from .api import ThetaScan
from .config import ThetaScanConfig

VOCAB = 1024
D_MODEL = 512
LAYERS = 9
HEADS = 8
KV_HEADS = 4
FFN_HIDDEN = 1024
THETA_LAYERS = (4, 5)
# FFN hidden width of the two ThetaScan blocks: the mixer has 852,008
# parameters against attention's 786,440, so 960 = 1024 - 64 keeps the model
# within 64 parameters of the baseline (17,059,976 = 17,059,912 + 2 (65,568 - 65,536))
THETA_FFN_HIDDEN = 960
LOGIT_SOFTCAP = 30.0
ROPE_BASE = 10_000.0


def theta_config() -> ThetaScanConfig:
    """The ThetaScan-Kernel layer: the kernel_expanded_reference_v0_1 recipe
    (ReLU^2 ridge with a learned per-head threshold, key-mass read, a fast
    two-rate bank, partial input RoPE) at memory_multiplier 2 (m = 128 by 2x
    expansion of a 64-wide base) with grouped key/value heads."""
    cfg = ThetaScanConfig.kernel_expanded_reference_v0_1(d_model=D_MODEL, n_heads=HEADS)
    return dataclasses.replace(cfg, memory_multiplier=2, share_key_query=False, key_value_heads=KV_HEADS)


def _rms(x: torch.Tensor) -> torch.Tensor:
    """RMS norm of the last axis (F.rms_norm's eps): one ts_rownorm launch per
    direction for [B,T,D] activations on the GPU."""
    if x.ndim == 3 and rownorm.supported(x.unsqueeze(1)):
        return rownorm.rms_rows(x.unsqueeze(1)).squeeze(1)
    return F.rms_norm(x, (x.shape[-1],))


def _add_rms(x: torch.Tensor, u: torch.Tensor, a: torch.Tensor | None,
             b: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """``y = a x + b u`` and its RMS norm: one row-glue launch on the GPU."""
    if x.ndim == 3 and rowglue.add_norm_supported(x, u, a, b):
        return rowglue.scale_add_norm(x, u, a, b)
    y = rowglue.scale_add(x, u, a, b)
    return y, _rms(y)


class Rotary(nn.Module):
    def __init__(self, dim: int, base: float = ROPE_BASE):
        super().__init__()
        self.register_buffer("inv_freq", 1.0 / (base ** (torch.arange(0, dim, 2, dtype=torch.float32) / dim)),
                             persistent=False)

    def forward(self, T: int, device):
        return rownorm.rotary_tables(self.inv_freq.to(device), T)


def _rotate(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """Rotate halves (x1, x2) of the last axis by the position's phases."""
    h = x.shape[-1] // 2
    x1, x2 = x[..., :h].float(), x[..., h:].float()
    c, s = cos[None, None], sin[None, None]
    return torch.cat([x1 * c + x2 * s, x2 * c - x1 * s], -1).to(x.dtype)


class CausalSelfAttention(nn.Module):
    def __init__(self, dim: int = D_MODEL, heads: int = HEADS, kv_heads: int = KV_HEADS, q_gain: float = 1.5):
        super().__init__()
        self.heads, self.kv_heads, self.hd = heads, kv_heads, dim // heads
        self.c_q = nn.Linear(dim, dim, bias=False)
        self.c_k = nn.Linear(dim, kv_heads * self.hd, bias=False)
        self.c_v = nn.Linear(dim, kv_heads * self.hd, bias=False)
        self.proj = nn.Linear(dim, dim, bias=False)
        nn.init.zeros_(self.proj.weight)
        self.q_gain = nn.Parameter(torch.full((heads,), q_gain))
        self.rotary = Rotary(self.hd)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        B, T, D = x.shape
        q = self.c_q(x).view(B, T, self.heads, self.hd).transpose(1, 2)
        k = self.c_k(x).view(B, T, self.kv_heads, self.hd).transpose(1, 2)
        v = self.c_v(x).view(B, T, self.kv_heads, self.hd).transpose(1, 2)
        cos, sin = self.rotary(T, x.device)
        if rownorm.supported(q, rope=True) and rownorm.supported(k, rope=True):
            # norm, rotary turn and query gain in one launch per stream
            q = rownorm.rms_rows(q, cos, sin, self.q_gain)
            k = rownorm.rms_rows(k, cos, sin)
        else:
            q, k = _rotate(_rms(q), cos, sin), _rotate(_rms(k), cos, sin)
            q = q * self.q_gain.to(q.dtype)[None, :, None, None]
        y = attention(q, k, v)
        return self.proj(y.transpose(1, 2).reshape(B, T, D))


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> torch.Tensor:
    """Causal softmax attention of q [B,H,T,d] against k, v [B,Hkv,T,d]
    (Hkv divides H: grouped key/value heads): the HIP kernel for bf16 heads
    of 64 where nothing is recorded for a backward, the fused (flash /
    memory-efficient) kernels for bf16 on the GPU, which read the grouped
    heads in place, the math form in fp32 elsewhere (the bf16 math form
    multiplies by a transposed operand)."""
    # (the fused kernels take the projections' token-major heads in place and
    # return theirs in the query's order, which reshapes to rows without a copy)
    if hip_attention.supported(q, k, v):
        return hip_attention.causal_attention(q, k, v)
    grouped = k.shape[1] != q.shape[1]
    if q.is_cuda and q.dtype == torch.bfloat16:
        from torch.nn.attention import SDPBackend, sdpa_kernel

        with sdpa_kernel([SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]):
            return F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=grouped)
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    if grouped:
        rep = q.shape[1] // k.shape[1]
        k, v = k.repeat_interleave(rep, dim=1), v.repeat_interleave(rep, dim=1)
    out = F.scaled_dot_product_attention(q.float(), k.float(), v.float(), is_causal=True)
    return out.to(q.dtype)


class MLP(nn.Module):
    def __init__(self, dim: int, hidden: int):
        super().__init__()
        self.fc = nn.Linear(dim, hidden, bias=False)
        self.proj = nn.Linear(hidden, dim, bias=False)
        nn.init.zeros_(self.proj.weight)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.proj(rowglue.relu2(self.fc(x)))


class Block(nn.Module):
    def __init__(self, theta: bool):
        super().__init__()
        self.theta = theta
        self.attn = ThetaScan(theta_config()) if theta else CausalSelfAttention()
        if theta:
            # the recipe's memory starts near identity; its projections start
            # like attention's (the output projection at zero)
            nn.init.zeros_(self.attn._core.proj_out.weight)
        self.mlp = MLP(D_MODEL, THETA_FFN_HIDDEN if theta else FFN_HIDDEN)
        self.attn_scale = nn.Parameter(torch.ones(D_MODEL))
        self.mlp_scale = nn.Parameter(torch.ones(D_MODEL))
        self.resid_mix = nn.Parameter(torch.stack((torch.ones(D_MODEL), torch.zeros(D_MODEL))))

    def forward(self, x: torch.Tensor, x0: torch.Tensor) -> torch.Tensor:
        # mix0 x + mix1 x0, then x + scale * f(x) per sublayer: one row-glue
        # launch each on the GPU, with the norm that the sublayer reads
        x, n = _add_rms(x, x0, self.resid_mix[0], self.resid_mix[1])
        x, n = _add_rms(x, self.attn(n), None, self.attn_scale)
        return rowglue.scale_add(x, self.mlp(n), None, self.mlp_scale)


class HybridLM(nn.Module):
    """Token ids [B,T] -> mean next-token cross-entropy (or logits)."""

    def __init__(self):
        super().__init__()
        self.tok_emb = nn.Embedding(VOCAB, D_MODEL)
        nn.init.normal_(self.tok_emb.weight, std=0.005)
        self.blocks = nn.ModuleList([Block(i in THETA_LAYERS) for i in range(LAYERS)])
        self.n_enc = LAYERS // 2
        self.skip_weights = nn.Parameter(torch.ones(min(self.n_enc, LAYERS - self.n_enc), D_MODEL))

    def forward(self, idx: torch.Tensor, targets: torch.Tensor | None = None) -> torch.Tensor:
        x = _rms(self.tok_emb(idx))
        x0 = x
        skips = []
        for i, block in enumerate(self.blocks):
            if i >= self.n_enc and skips:
                x = rowglue.scale_add(x, skips.pop(), None, self.skip_weights[i - self.n_enc])
            x = block(x, x0)
            if i < self.n_enc:
                skips.append(x)
        x = _rms(x)
        logits = F.linear(x, self.tok_emb.weight.to(x.dtype))
        if targets is None:
            return LOGIT_SOFTCAP * torch.tanh(logits.float() / LOGIT_SOFTCAP)
        # the soft-capped logits' cross entropy: one HIP launch per direction
        # on the GPU (the fp32 capped logits are never stored)
        return rowglue.softcap_cross_entropy(logits.reshape(-1, VOCAB), targets.reshape(-1), LOGIT_SOFTCAP)


# ---------------------------------------------------------------- int8 round trip

def quantize_rows(w: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor]:
    """Per-row symmetric int8: scale = max|row| / 127 (fp32), q = round(w / scale)
    in [-127, 127] over the last axis."""
    w32 = w.detach().float()
    rows = w32.reshape(-1, w32.shape[-1])
    scale = rows.abs().amax(-1, keepdim=True) / 127.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    q = torch.clamp(torch.round(rows / scale), -127, 127).to(torch.int8)
    return q.view(w.shape), scale.view(*w.shape[:-1], 1)


def dequantize_rows(q: torch.Tensor, scale: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    return (q.float() * scale).to(dtype)


def int8_round_trip(model: nn.Module) -> dict:
    """The model's state dict with every weight matrix (two or more axes)
    replaced by its per-row int8 round trip; vectors and buffers unchanged."""
    out = {}
    for name, t in model.state_dict().items():
        if t.is_floating_point() and t.ndim >= 2:
            q, s = quantize_rows(t)
            out[name] = dequantize_rows(q, s, t.dtype)
        else:
            out[name] = t
    return out


def parameter_count(model: nn.Module) -> int:
    return sum(p.numel() for p in model.parameters())
