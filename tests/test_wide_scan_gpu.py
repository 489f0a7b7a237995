"""bf16 scans of more than 128 keys or values in one call (GPU tests).

Every retention, ext column and output mode the backward passes use, at the
key widths with a kernel (192, 256, 384) and between them (padded), value
widths of one to six 64-column slices with a ragged last one, sequences that
end inside a tile and in one segment or several, against the float64 recurrence.
Bar: rel 2e-2 (bf16 inputs and outputs; the fp32 outputs carry the bf16
rounding of the score tiles and the published state, about 1e-2 of the largest).
"""
from __future__ import annotations

import pytest
import torch

from oracle import scans as oracle
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 2e-2
WIDTHS = [(136, 64), (192, 192), (256, 72), (384, 64), (64, 384), (64, 136), (32, 512), (384, 200)]


def _case(Dk, Dv, kind, T, seed):
    g = torch.Generator().manual_seed(seed)
    B, H = 2, 2
    # feature-like keys and queries: positive and of unit mass, so sums do not cancel
    q, k = ((torch.rand(B, H, T, Dk, generator=g, dtype=torch.float64) * 2 / Dk).to(torch.bfloat16) for _ in range(2))
    v = torch.randn(B, H, T, Dv, generator=g, dtype=torch.float64).to(torch.bfloat16)
    ret = None
    if kind == "static":
        ret = torch.log(torch.tensor([0.9, 0.99], dtype=torch.float64))
    elif kind == "stream":
        ret = -torch.rand(B, H, T, 1, generator=g, dtype=torch.float64) * 0.1
    return q, k, v, ret


def _expected(q, k, v, ret, reverse):
    q, k, v = q.double(), k.double(), v.double()
    dec = None if ret is None else (oracle.as_stream(ret, q) if ret.ndim == 1 else ret)
    if not reverse:
        return oracle.linattn_chunk(q, k, v, dec)
    f = lambda t: t.flip(2)  # noqa: E731
    # a reversed step from s+1 to s applies the decay of s+1
    if dec is not None:
        dec = torch.cat([torch.zeros_like(dec[:, :, :1]), f(dec)[:, :, :-1]], 2)
    return f(oracle.linattn_chunk(f(q), f(k), f(v), dec))


@pytest.mark.parametrize("widths", WIDTHS)
@pytest.mark.parametrize("kind", ["none", "static", "stream"])
@pytest.mark.parametrize("ext", ["none", "key", "value"])
def test_wide_scan_matches_recurrence(cuda, widths, kind, ext):
    from thetascan_amd import _lib
    from thetascan_amd._core.ops import scan_hip

    Dk, Dv = widths
    for T, reverse, f32 in ((333, False, False), (64, True, False), (450, True, True), (1, False, True)):
        q, k, v, ret = _case(Dk, Dv, kind, T, Dk + Dv + T)
        kw = {"retention": {"none": _lib.RET_NONE, "static": _lib.RET_STATIC, "stream": _lib.RET_STREAM}[kind]}
        if kind == "static":
            kw["log_alpha"] = ret.to(cuda, torch.float32)
        if kind == "stream":
            kw["decay"] = ret.to(cuda, torch.float32)
        g = torch.Generator().manual_seed(5)
        col = torch.rand(*q.shape[:3], generator=g, dtype=torch.float64)
        qx, kx, vx = q.double(), k.double(), v.double()
        if ext == "key":
            kw.update(q_ext=col.to(cuda, torch.float32), k_ext="ones")
            qx, kx = torch.cat([qx, col[..., None].float().double()], -1), torch.cat([kx, torch.ones_like(kx[..., :1])], -1)
        if ext == "value":
            kw.update(v_ext="ones", want_ext_out=True)
            vx = torch.cat([vx, torch.ones_like(vx[..., :1])], -1)
        want = _expected(qx, kx, vx, ret, reverse)
        dev = [t.to(cuda) for t in (q, k, v)]
        if f32 and ext != "value":
            out = torch.full((*q.shape[:3], Dv), 0.25, dtype=torch.float32, device=cuda)
            scan_hip.scan_launch(*dev, reverse=reverse, out=out, out_mode=_lib.OUT_ACCUM_F32, out_scale=2.0,
                                 seg_chunks=2, **kw)
            got, mass = (out - 0.25) / 2.0, None
        else:
            mode = _lib.OUT_STORE_F32 if f32 else _lib.OUT_STORE
            got, mass, _ = scan_hip.scan_launch(*dev, reverse=reverse, out_mode=mode, **kw)
        assert got.shape == v.shape
        assert rel_err(got, want[..., :Dv]) < TOL, (T, reverse, f32)
        if ext == "value":
            assert rel_err(mass, want[..., Dv]) < TOL, (T, reverse, f32)


def test_states_of_wide_scans_stay_refused(cuda):
    from thetascan_amd._core.ops import scan_hip

    q, k, v, _ = _case(192, 64, "none", 64, 1)
    dev = [t.to(cuda) for t in (q, k, v)]
    with pytest.raises(NotImplementedError):
        scan_hip.scan_launch(*dev, want_final=True)
    with pytest.raises(NotImplementedError):
        scan_hip.scan_launch(*dev, init_state=torch.zeros(2, 2, 192, 64, device=cuda))


@pytest.mark.parametrize("Dk", [192, 384])
def test_an_overflowed_score_is_infinite(cuda, monkeypatch, Dk):
    """A score past the largest float gives an infinite output of its sign, as
    the block-wise scan gives, not NaN (its hi + lo pair is inf + 0)."""
    from thetascan_amd._core.ops import scan_hip

    g = torch.Generator().manual_seed(9)
    q, k, v = (torch.rand(1, 1, 150, w, generator=g) + 0.5 for w in (Dk, Dk, 64))
    q[:, :, 20] *= 1e20
    k[:, :, 10] *= 1e20
    v[..., ::2] *= -1
    q, k, v = (t.to(cuda, torch.bfloat16) for t in (q, k, v))
    got, _, _ = scan_hip.scan_launch(q, k, v)
    monkeypatch.setattr(scan_hip, "WIDE_KEYS", 128)
    want, _, _ = scan_hip.scan_launch(q, k, v)
    assert torch.isinf(want[0, 0, 20]).all() and not torch.isnan(want).any()
    off = torch.isinf(want)
    assert not torch.isnan(got).any() and torch.equal(torch.isinf(got), off)
    assert torch.equal(got[off], want[off]) and rel_err(got[~off], want[~off]) < TOL
