"""What reaches a read epilogue's launch (no GPU: the launch is a stand-in):
its operands live until it, and a gate it would misread does not reach it."""
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


def _under_autocast(monkeypatch):
    monkeypatch.setattr(torch, "is_autocast_enabled", lambda device: device == "cuda")
    monkeypatch.setattr(torch, "get_autocast_dtype", lambda device: torch.bfloat16)


@pytest.mark.parametrize("views", [1, 3])
def test_a_gate_of_another_dtype_stays_out_of_the_read(monkeypatch, views):
    """Under autocast to bf16 the gate of an fp32 input is a bf16 product,
    which an epilogue of fp32 reads would read past its end: the request does
    not fit such reads (as they may be, where fp32 biases are added to the
    projections), and the read itself refuses the gate before any launch."""
    from thetascan_amd._core.ops import bankread, composed, gn

    B, H, T, d = 1, 2, 3, 16
    monkeypatch.setattr(bankread, "eligible", lambda nums, masses, resids, heads: True)
    x, weight = torch.randn(B, T, H * d), torch.randn(H * d, H * d)
    nums = [torch.randn(B, H, T, d) for _ in range(views)]
    coef = torch.ones(views, H)
    request = composed.OutputRequest(x, weight, torch.zeros(H * d), H, d, coef)
    args = (nums, [None] * views, [nums[0]])
    assert request.fits(*args)
    with monkeypatch.context() as m:
        _under_autocast(m)
        assert not request.fits(*args)
        assert composed.OutputRequest(x, None, None, H, d, coef).fits(*args)
    for gate in (nums[0].to(torch.bfloat16), nums[0][:, :1]):
        with pytest.raises(ValueError, match="does not match the reads"):
            bankread.bank_read(nums, [None] * views, [nums[0]], coef, gate=gate)
        with pytest.raises(ValueError, match="does not match the reads"):
            gn.normalized_read(nums[0], None, nums[0], gate=gate)
