"""The operands of a ts_bank_read launch live until it (no GPU: the launch is
a stand-in that looks at what its arguments point to)."""
from __future__ import annotations

import weakref

import pytest
import torch


@pytest.mark.parametrize("coef_dtype", [torch.float32, torch.bfloat16, torch.float64])
def test_converted_operands_live_until_the_launch(monkeypatch, coef_dtype):
    from thetascan_amd._core.ops import bankread

    n, B, H, T, d = 2, 1, 2, 3, 16
    nums = [torch.randn(B, H, T, d) for _ in range(n)]
    masses = [torch.rand(B, H, T, dtype=torch.float64) for _ in range(n)]
    gate, bias = torch.randn(B, H, T, d), torch.zeros(H * d, dtype=torch.bfloat16)
    coef = torch.ones(n, H).to(coef_dtype)
    kept, alive = [], []
    call = bankread._call

    def tracked(*args):
        desc, io, tensors = call(*args)
        for t in tensors:
            kept.extend(weakref.ref(x) for x in (t if isinstance(t, list) else [t]))
        return desc, io, tensors

    class Library:
        def ts_bank_read_fwd(self, *args):
            alive.extend(ref() is not None for ref in kept)
            return 0

    monkeypatch.setattr(bankread, "_call", tracked)
    monkeypatch.setattr(bankread._lib, "load", Library)
    monkeypatch.setattr(bankread._lib, "stream_handle", lambda device: None)
    bankread._forward(nums, masses, [nums[0]], coef, gate, bias, 1.0, 1e-6)
    assert len(alive) == 2 * n + 4 and all(alive)
