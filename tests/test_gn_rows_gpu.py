"""GN stages on streams whose token rows are strided, shared or few: the
kernels address a group's rows through offsets that end after the last token,
so rows of any stride and one row broadcast over the tokens have to give the
same bits as contiguous copies of them (the arithmetic is the same)."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(B, H, T, w, layout, dtype, dev, g):
    if layout == "broadcast":
        return torch.randn(B, H, 1, w, generator=g).to(dev, dtype).expand(B, H, T, w)
    if layout == "token_major":
        return torch.randn(B, T, H, w, generator=g).to(dev, dtype).transpose(1, 2)
    # rows of a wider matrix whose tail would change a sum if it were read
    return torch.randn(B, H, T, w + 64, generator=g).to(dev, dtype)[..., :w]


@pytest.mark.parametrize("nonlin", ["relu2", "tanh", "silu"])
@pytest.mark.parametrize("dtype,d,m", [(torch.bfloat16, 64, 128), (torch.float32, 32, 48), (torch.bfloat16, 32, 192)])
@pytest.mark.parametrize("layout", ["broadcast", "token_major", "padded"])
@pytest.mark.parametrize("T", [1, 65, 130])
def test_gn_rows_of_any_stride(cuda, dtype, d, m, layout, T, nonlin):
    from thetascan_amd._core.ops import gn

    B, H = 2, 3
    g = torch.Generator().manual_seed(7 * d + m + T)
    w1 = (torch.randn(H, m, d, generator=g) / d ** 0.5).to(cuda, dtype)
    w2 = (torch.randn(H, d, m, generator=g) * 0.3).to(cuda, dtype)
    x, v, num = (_rows(B, H, T, w, layout, dtype, cuda, g) for w in (d, d, m))
    mass = torch.rand(B, H, T, generator=g).to(cuda) + 0.5
    dys = [_rows(B, H, T, w, layout, dtype, cuda, g) for w in (m, d, m, m, d)]

    def run(x, v, num, dys):
        x, v, num = (t.detach().requires_grad_(True) for t in (x, v, num))
        ws = [t.clone().requires_grad_(True) for t in (w1, w2)]
        out = list(gn.write(x, v, *ws, nonlin=nonlin))
        out += list(gn.read_stage(x, *ws, None, num, mass, corr=gn.READ_NORMALIZED, want_resid=True, nonlin=nonlin))
        grads = torch.autograd.grad(out, [x, v, num, *ws], dys)
        return [*out, *grads]

    got = run(x, v, num, dys)
    want = run(x.contiguous(), v.contiguous(), num.contiguous(), [t.contiguous() for t in dys])
    for a, b in zip(got, want):
        assert torch.isfinite(a).all()
        assert torch.equal(a, b)


def _backwards(real):
    """Descriptors of the same rows from the last token to the first."""
    from thetascan_amd import _lib

    def strided(t):
        s = real(t)
        if t is None or t.ndim != 4:
            return s
        st = t.stride(2)
        return _lib.Strided(t.data_ptr() + (t.shape[2] - 1) * st * t.element_size(), t.stride(0), t.stride(1), -st)

    return strided


@pytest.mark.parametrize("dtype,d,m", [(torch.bfloat16, 64, 128), (torch.float32, 32, 48), (torch.bfloat16, 32, 192)])
@pytest.mark.parametrize("T", [2, 64, 130])
def test_gn_rows_of_negative_stride(cuda, monkeypatch, dtype, d, m, T):
    """The stages work token by token: with every stream described from its
    last row to its first they give the same bits in the same rows (the weight
    gradients sum the tokens in the other order)."""
    from thetascan_amd._core.ops import gn
    from tests.conftest import rel_err

    B, H = 2, 3
    g = torch.Generator().manual_seed(d + m + T)
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda, dtype)  # noqa: E731
    weights = [rnd(H, m, d) / d ** 0.5, rnd(H, d, m) * 0.3]
    streams = [rnd(B, H, T, w) for w in (d, d, m)]
    dys = [rnd(B, H, T, w) for w in (m, d, m, m, d)]

    def run():
        x, v, num = (t.clone().requires_grad_(True) for t in streams)
        ws = [t.clone().requires_grad_(True) for t in weights]
        out = list(gn.write(x, v, *ws))
        out += list(gn.read_stage(x, *ws, None, num, None, corr=gn.READ_PLAIN, want_resid=True))
        return [*out, *torch.autograd.grad(out, [x, v, num, *ws], dys)]

    want = run()
    monkeypatch.setattr(gn._lib, "strided", _backwards(gn._lib.strided))
    got = run()
    for i, (a, b) in enumerate(zip(got, want)):
        if i < len(got) - 2:
            assert torch.equal(a, b), i
        else:
            assert rel_err(a, b) < (2e-2 if dtype == torch.bfloat16 else 1e-5), i


@pytest.mark.parametrize("dtype,d,m", [(torch.bfloat16, 64, 128), (torch.bfloat16, 32, 192)])
@pytest.mark.parametrize("layout", ["token_major", "one for all tokens"])
def test_gn_read_with_a_strided_mass(cuda, dtype, d, m, layout):
    """The gradient of a mass of any strides is the contiguous copy's."""
    from thetascan_amd._core.ops import gn

    B, H, T = 2, 3, 70
    g = torch.Generator().manual_seed(m)
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda, dtype)  # noqa: E731
    q, num, w1 = rnd(B, H, T, d), rnd(B, H, T, m), rnd(H, m, d) / d ** 0.5
    if layout == "token_major":
        mass = (torch.rand(B, T, H, generator=g) + 0.5).to(cuda).transpose(1, 2)
    else:
        mass = (torch.rand(B, H, 1, generator=g) + 0.5).to(cuda).expand(B, H, T)
    dy = rnd(B, H, T, m)

    def run(mass):
        mass = mass.detach().requires_grad_(True)
        h, _ = gn.read_stage(q, w1, None, None, num, mass, corr=gn.READ_NORMALIZED)
        return torch.autograd.grad(h, mass, dy)[0]

    assert torch.equal(run(mass), run(mass.contiguous()))
