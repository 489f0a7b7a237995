"""Causal attention of the hybrid LM (ts_causal_attention_fwd where nothing is
recorded, torch's fused attention otherwise) against float64.

Sequence lengths at the edges of the 64-key tiles, the 32 queries of a wave
and the 128 of a workgroup, grouped and plain heads, token-major and
contiguous memory.  The probabilities and the output are rounded to bf16 once
each (2^-9 relative): 2-norm bar 6e-3; each row on its own 2e-2.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v):
    rep = q.shape[1] // k.shape[1]
    q, k, v = q.double(), k.double().repeat_interleave(rep, 1), v.double().repeat_interleave(rep, 1)
    T = q.shape[2]
    s = (q @ k.transpose(-1, -2)) * 0.125
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool).triu(1), -float("inf"))
    return torch.softmax(s, -1) @ v


@pytest.mark.parametrize("T", [1, 31, 33, 64, 65, 127, 129, 300])
@pytest.mark.parametrize("heads,kv_heads", [(8, 4), (3, 3), (4, 1)])
@pytest.mark.parametrize("order", ["heads", "tokens"])
def test_attention_matches_float64(cuda, T, heads, kv_heads, order):
    from thetascan_amd import _lib, hybrid_lm as lm

    g = torch.Generator().manual_seed(T + heads)
    q, k, v = (torch.randn(2, T, h, 64, generator=g).bfloat16().transpose(1, 2) for h in (heads, kv_heads, kv_heads))
    q = q * 2.0  # sharper rows: a running maximum that moves between tiles
    ref = _reference(q, k, v)
    dev = [t.transpose(1, 2).contiguous().to(cuda).transpose(1, 2) for t in (q, k, v)]
    if order == "heads":
        dev = [t.contiguous() for t in dev]
    with torch.no_grad(), _lib.record_launches() as recs:
        y = lm.attention(*dev)
        torch.cuda.synchronize()
    assert "ts_causal_attention_fwd" in {r[0] for r in recs}
    assert y.shape == q.shape and (T == 1 or (y.transpose(1, 2).is_contiguous() == (order == "tokens")))
    err = y.double().cpu() - ref
    print(f"attention T={T} {heads}/{kv_heads} {order}: {float(err.norm() / ref.norm()):.2e}", flush=True)
    assert float(err.norm() / ref.norm()) < 6e-3
    assert float((err.norm(dim=-1) / ref.norm(dim=-1)).max()) < 2e-2


@pytest.mark.parametrize("order", ["heads", "tokens"])
def test_recorded_attention_takes_heads_in_either_order(cuda, order):
    """With gradients torch's fused attention runs; its gradients agree with
    float64 from token-major heads as from contiguous ones (bf16: 1e-2)."""
    from thetascan_amd import hybrid_lm as lm

    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.randn(2, 130, h, 64, generator=g).bfloat16().transpose(1, 2) for h in (8, 4, 4))
    dy = torch.randn(2, 130, 8, 64, generator=g).bfloat16().transpose(1, 2)
    leaves = [t.double().requires_grad_(True) for t in (q, k, v)]
    ref = _reference(*leaves)
    ref.backward(dy.double())
    dev = [t.to(cuda) if order == "tokens" else t.contiguous().to(cuda) for t in (q, k, v)]
    dev = [t.requires_grad_(True) for t in dev]
    y = lm.attention(*dev)
    y.backward(dy.to(cuda))
    torch.cuda.synchronize()
    for got, want in [(y.detach(), ref.detach())] + [(t.grad, l.grad) for t, l in zip(dev, leaves)]:
        assert float((got.double().cpu() - want).norm() / want.norm()) < 1e-2


def test_what_the_kernel_leaves_to_torch(cuda):
    from thetascan_amd._core.ops import attention

    q = torch.zeros(1, 2, 5, 64, device=cuda, dtype=torch.bfloat16)
    assert attention.supported(q, q, q)
    assert not attention.supported(q.float(), q.float(), q.float())
    assert not attention.supported(q[..., :32], q[..., :32], q[..., :32])
    assert not attention.supported(q, q[:, :, :4], q[:, :, :4])
    assert not attention.supported(q.clone().requires_grad_(True), q, q)
    off = torch.zeros(1 * 2 * 5 * 64 + 4, device=cuda, dtype=torch.bfloat16)[4:].view(1, 2, 5, 64)
    assert not attention.supported(off, q, q)
