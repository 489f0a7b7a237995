"""ts_bank_params_fwd / _bwd (a fast bank's log retentions and blend
coefficients in one launch) against the tensor expressions (GPU tests).

The forward rounds through the parameter's and the streams' dtypes as the
expressions do: equal to one ulp of fp32 before those roundings (2e-7), so a
bf16 value may land on a neighbour (2^-8 relative).  Gradients: 1e-6 in fp32,
one bf16 rounding otherwise (4e-3); alpha covers both sides of softplus's
linear range.
"""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pdt,xdt", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16),
                                     (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("n,H", [(1, 1), (2, 8), (6, 130)])
@pytest.mark.parametrize("tanh", [False, True])
def test_bank_params_match_expressions(cuda, pdt, xdt, n, H, tanh):
    from thetascan_amd._core.ops import bankread, maps

    g = torch.Generator().manual_seed(n * H)
    alpha = (torch.randn(n, H, generator=g) * 4 + 2).to(pdt)
    alpha[0, 0] = -25.0
    eta = (torch.randn(n, H, generator=g) * 0.5).to(pdt)
    dla = torch.randn(n, H, generator=g)
    dcoef = torch.randn(n + 1, H, generator=g)

    a, e = (t.clone().to(cuda).requires_grad_(True) for t in (alpha, eta))
    las, coef = bankread.bank_params(a, e, tanh, xdt)
    a64, e64 = (t.double().requires_grad_(True) for t in (alpha, eta))
    want_la = -F.softplus(-a64)
    blends = torch.tanh(e64) if tanh else e64
    want_coef = torch.cat([1.0 - blends.sum(0, keepdim=True), blends])
    low = torch.bfloat16 in (pdt, xdt)
    assert all(x.dtype == torch.float32 and x.shape == (H,) for x in las)
    for j in range(n):
        assert torch.allclose(las[j].cpu().double(), want_la[j], rtol=2 ** -8 if low else 1e-6, atol=0)
        same = (-F.softplus(-alpha[j].to(cuda))).to(xdt).float()
        assert torch.allclose(las[j], same, rtol=2 ** -7 if low else 1e-6, atol=0)
    assert rel_err(coef, want_coef) < (2 ** -8 if tanh and pdt == torch.bfloat16 else 1e-6)
    assert maps.fast_coefficients(list(blends.view(n, 1, H, 1, 1))).shape == coef.shape
    torch.autograd.backward([*las, coef], [*dla.to(cuda), dcoef.to(cuda)])
    torch.autograd.backward([want_la, want_coef], [dla.double(), dcoef.double()])
    tol = 4e-3 * (2 if tanh else 1) if pdt == torch.bfloat16 else 1e-5
    assert rel_err(a.grad, a64.grad) < tol and rel_err(e.grad, e64.grad) < tol
    # a retention without a gradient (its view's outputs unused) counts as zero
    a.grad = None
    bankread.bank_params(a, e, tanh, xdt)[1].backward(dcoef.to(cuda))
    assert not a.grad.any()
