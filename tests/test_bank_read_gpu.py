"""ts_bank_read_fwd / ts_bank_read_bwd (a bank's reads, blend and output gate
in one pass) against float64 autograd of the same expression (GPU tests).

Bars: fp32 2e-5 (fp32 sums of up to 8 views, a hardware reciprocal and exp2
of about 1 ulp each); bf16 1e-2 of the largest value (one rounding of each
bf16 output, 2^-9 relative, and the coefficient and bias sums over rounded
inputs, which the float64 side sees too).
"""
from __future__ import annotations

import pytest
import torch

from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-5, torch.bfloat16: 1e-2}


def _reference(nums, masses, resids, coef, gate, bias, s, eps):
    y = 0.0
    for j, num in enumerate(nums):
        read = s * num if masses is None else s * num / (masses[j].unsqueeze(-1) + eps)
        y = y + coef[j].view(1, -1, 1, 1) * (resids[j if len(resids) > 1 else 0] + read)
    if gate is None:
        return y
    pre = gate + bias.view(1, gate.shape[1], 1, -1)
    return y * torch.nn.functional.silu(pre)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,per_view", [(1, False), (2, True), (3, False), (5, True), (8, False)])
@pytest.mark.parametrize("mass,gated", [(True, True), (True, False), (False, True)])
def test_bank_read_matches_float64(cuda, dtype, n, per_view, mass, gated):
    from thetascan_amd._core.ops import bankread

    for B, H, T, d in ((2, 3, 130, 64), (1, 2, 1, 16), (1, 1, 129, 40), (2, 1, 65, 128)):
        g = torch.Generator().manual_seed(100 * n + T + d)
        rnd = lambda *shape: torch.randn(*shape, generator=g, dtype=torch.float64).to(dtype)  # noqa: E731
        nums = [rnd(B, H, T, d) for _ in range(n)]
        resids = [rnd(B, H, T, d) for _ in range(n if per_view else 1)]
        masses = [torch.rand(B, H, T, generator=g, dtype=torch.float64).float() + 0.2 for _ in range(n)] if mass else None
        coef = torch.randn(n, H, generator=g, dtype=torch.float64).float()
        # the gate's pre-activation as the projection leaves it: token-major
        gate = rnd(B, T, H, d).transpose(1, 2) if gated else None
        bias = rnd(H * d) if gated else None
        dy = rnd(B, T, H, d).transpose(1, 2)
        leaves = nums + resids + (masses or []) + [coef] + ([gate, bias] if gated else [])
        want_in = [t.double().requires_grad_(True) for t in leaves]
        got_in = [t.to(cuda).detach().requires_grad_(True) for t in leaves]

        def split(ts):
            r = len(resids)
            m = list(ts[n + r:n + r + n]) if mass else None
            rest = ts[n + r + (n if mass else 0):]
            return list(ts[:n]), m, list(ts[n:n + r]), rest[0], (rest[1] if gated else None), (rest[2] if gated else None)

        a, b = split(want_in), split(got_in)
        want = _reference(*a, 0.7, 1e-6)
        got = bankread.bank_read(b[0], b[1] if mass else [None] * n, b[2], b[3], s=0.7, eps=1e-6, gate=b[4],
                                 gate_bias=b[5])
        assert got.transpose(1, 2).is_contiguous() and got.dtype == dtype
        assert rel_err(got, want) < TOL[dtype], (n, T, d)
        want.backward(dy.double())
        got.backward(dy.to(cuda))
        for i, (x, y) in enumerate(zip(got_in, want_in)):
            assert x.grad.shape == y.grad.shape and x.grad.dtype == x.dtype
            assert rel_err(x.grad, y.grad) < TOL[dtype], (n, T, d, i)


def test_views_the_kernel_does_not_take(cuda):
    """Mixed dtypes (a stale view's fp32 numerators), more than eight views
    and rows above 512 bytes stay with the separate reads and blend."""
    from thetascan_amd._core.ops import bankread

    x = torch.zeros(1, 2, 8, 64, device=cuda, dtype=torch.bfloat16)
    assert bankread.eligible([x, x], [None, None], [x], 2)
    assert not bankread.eligible([x, x.float()], [None, None], [x], 2)
    assert not bankread.eligible([x] * 9, [None] * 9, [x], 2)
    assert not bankread.eligible([x, x, x], [None] * 3, [x, x], 2)
    wide = torch.zeros(1, 2, 8, 264, device=cuda, dtype=torch.bfloat16)
    assert not bankread.eligible([wide], [None], [wide], 2)
