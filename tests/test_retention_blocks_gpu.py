"""ts_retention_grad over the key widths and value-block counts its kernels are
built for (a wave owns a key block and every S-th value block; counts round up
to 4, 5 or 8), against the pair sums in float64.

Tolerance: the weighted queries and keys enter their products as bf16 pairs
hi + lo (relative error at most 2^-17 each; a pair across tiles meets one of
each kind), the sums are fp32, so the error stays below 2^-15 of the sum of the
pairs' magnitudes.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk", [16, 32, 48, 64, 80, 96, 112, 128])
@pytest.mark.parametrize("dv,mass", [(8, False), (64, False), (64, True), (72, True), (112, True), (128, False)])
@pytest.mark.parametrize("T,seg", [(1, 0), (129, 0), (450, 2)])
def test_retention_blocks(cuda, dk, dv, mass, T, seg):
    from thetascan_amd._core.ops import scan_hip

    B, H = 1, 3
    g = torch.Generator().manual_seed(dk * 1000 + dv + T)
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda, torch.bfloat16)  # noqa: E731
    q, k, v, do = rnd(B, H, T, dk), rnd(B, H, T, dk), rnd(B, H, T, dv), rnd(B, H, T, dv)
    dm = torch.randn(B, H, T, generator=g).to(cuda) if mass else None
    la = torch.tensor([-2.0, -0.05, -0.001], device=cuda)
    got = scan_hip.retention_grad(q, k, v, do, dm, la, seg).double().cpu()
    q, k, v, do = (t.double().cpu() for t in (q, k, v, do))
    pairs = q @ k.mT * (do @ v.mT + (dm.double().cpu()[..., None] if mass else 0.0))
    lag = (torch.arange(T)[:, None] - torch.arange(T)[None, :]).double().clamp(min=0)
    pairs = pairs * lag * torch.exp(la.double().cpu()[:, None, None] * lag)
    err = (got - pairs.sum((-1, -2))).abs()
    assert (err <= 2.0 ** -15 * pairs.abs().sum((-1, -2)) + 1e-12).all()
