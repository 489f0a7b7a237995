"""ts_contract_sums (the GN backward's weight gradients in one launch) against
float64 sums of the same rounded tiles: widths on both sides of the 128-column
blocks, several terms and a scaled sum, and token counts from none to a ragged
last tile and several slices.

Tolerance: products of the tiles' values are exact in fp32 (bf16) or rounded
once (fp32); the N-term fp32 sums err by at most N 2^-24 of the terms'
magnitudes (far less: partial sums per slice), and a bf16 output rounds once.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("p,q", [(16, 16), (64, 128), (144, 64), (64, 192), (384, 32), (128, 256)])
@pytest.mark.parametrize("N", [0, 1, 63, 130, 2049])
def test_contract_sums(cuda, dtype, p, q, N):
    from thetascan_amd._core.ops import gn

    H = 3
    g = torch.Generator().manual_seed(p + q + N)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype)  # noqa: E731
    a, b, a2, b2 = rnd(4, H, N, p), rnd(4, H, N, q), rnd(H, N, q), rnd(H, N, p)
    w = rnd(H, p, q)
    ac, bc = a.to(cuda), b.to(cuda)
    got = gn._contract_sums([[(ac[0], bc[0])], [(a2.to(cuda), b2.to(cuda))], [(ac[1], bc[1]), (ac[2], bc[2])],
                             [(ac[3], bc[3])]],
                            [(1, None), (2, (w.to(cuda), 3, 2.0)), (0, None)], [dtype] * 3)
    c = [x.double().mT @ y.double() for x, y in zip(a, b)]
    m = [x.double().abs().mT @ y.double().abs() for x, y in zip(a, b)]
    want = [a2.double().mT @ b2.double(), c[1] + c[2] + 2 * w.double() * c[3], c[0]]
    mag = [a2.double().abs().mT @ b2.double().abs(), m[1] + m[2] + 2 * w.double().abs() * m[3], m[0]]
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23
    for y, r, s in zip(got, want, mag):
        assert y.dtype == dtype
        assert ((y.cpu().double() - r).abs() <= unit * r.abs() + max(N, 4) * 2.0 ** -24 * s).all()
