"""ts_views_bwd (the gradients of several retentions' scans in one causal and
one anti-causal pass) against float64 autograd through the tiled recurrence
(GPU tests).

Bar: rel 2e-2 of the largest value (bf16 operands; the score sums enter as
hi + lo, the weighted values and the published states as bf16).  Widths at
the edges of the 64-column slices, sequences that end inside a tile, one
segment and several, with and without the key mass, two and three views.
"""
from __future__ import annotations

import pytest
import torch

from oracle import scans as oracle
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu

RATES = (None, (0.9, 0.97), (0.99, 0.5))


@pytest.mark.parametrize("n", [2, 3])
@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("m,dv", [(64, 64), (8, 8), (72, 64), (128, 40), (384, 64)])
def test_views_backward_matches_float64(cuda, n, mass, m, dv):
    from thetascan_amd._core.ops import scan_hip

    for T, seg in ((1, 0), (64, 0), (333, 0), (333, 2), (450, 1)):
        g = torch.Generator().manual_seed(m + dv + T)
        B, H = 2, 2
        q, k = ((torch.rand(B, H, T, m, generator=g, dtype=torch.float64) * 2 / m).to(torch.bfloat16) for _ in range(2))
        # values as the stacked projection holds them: token-major rows
        v = torch.randn(B, T, H, dv, generator=g, dtype=torch.float64).to(torch.bfloat16).transpose(1, 2)
        dos = [torch.randn(B, H, T, dv, generator=g, dtype=torch.float64).to(torch.bfloat16) for _ in range(n)]
        dms = [torch.randn(B, H, T, generator=g, dtype=torch.float64).float() for _ in range(n)] if mass else None
        las = [None if r is None else torch.log(torch.tensor(r, dtype=torch.float64)) for r in RATES[:n]]
        leaves = [t.double().requires_grad_(True) for t in (q, k, v)]
        vx = torch.cat([leaves[2], torch.ones_like(leaves[2][..., :1])], -1) if mass else leaves[2]
        loss = 0.0
        for j, la in enumerate(las):
            out = oracle.linattn_chunk(leaves[0], leaves[1], vx, None if la is None else oracle.as_stream(la, leaves[0]))
            loss = loss + (out[..., :dv] * dos[j].double()).sum()
            if mass:
                loss = loss + (out[..., dv] * dms[j].double()).sum()
        loss.backward()
        dev = lambda ts: None if ts is None else [None if t is None else t.to(cuda) for t in ts]  # noqa: E731
        got = scan_hip.views_bwd_launch(q.to(cuda), k.to(cuda), v.to(cuda), dev(las), dev(dos), dev(dms), need_q=True,
                                        need_kv=True, seg_chunks=seg)
        for name, a, e in zip(("dq", "dk", "dv"), got, leaves):
            assert a.shape == e.shape and a.dtype == torch.bfloat16
            assert rel_err(a, e.grad) < 2e-2, (name, T, seg)
        only_q = scan_hip.views_bwd_launch(q.to(cuda), k.to(cuda), v.to(cuda), dev(las), dev(dos), dev(dms),
                                           need_q=True, need_kv=False, seg_chunks=seg)
        assert only_q[1] is None and only_q[2] is None and torch.equal(only_q[0], got[0])


def test_bank_of_static_views_takes_the_passes(cuda):
    """The gradients of a bank's views through autograd run in ts_views_bwd,
    and equal the per-view scans' to bf16 rounding."""
    from thetascan_amd import _lib
    from thetascan_amd._core.ops import scan_hip

    g = torch.Generator().manual_seed(3)
    B, H, T, m, dv = 2, 2, 200, 64, 64
    base = [torch.rand(B, H, T, m, generator=g).to(cuda, torch.bfloat16) / 32 for _ in range(2)]
    base.append(torch.randn(B, H, T, dv, generator=g).to(cuda, torch.bfloat16))
    la = torch.log(torch.tensor([0.9, 0.97], device=cuda))
    dys = [torch.randn(B, H, T, dv, generator=g).to(cuda, torch.bfloat16) for _ in range(2)]

    def run():
        ts = [t.clone().requires_grad_(True) for t in base]
        r = la.clone().requires_grad_(True)
        with _lib.record_launches() as recs:
            outs = scan_hip.linattn_views(*ts, (None, r), 64)
            torch.autograd.backward(outs, dys)
            torch.cuda.synchronize()
        return [t.grad for t in ts] + [r.grad], {rec[0] for rec in recs}

    got, names = run()
    assert "ts_views_bwd" in names and "ts_scan_pair_fwd" not in names
    real = scan_hip.views_bwd_eligible
    try:
        scan_hip.views_bwd_eligible = lambda *a: False
        want, names = run()
    finally:
        scan_hip.views_bwd_eligible = real
    assert "ts_views_bwd" not in names
    for a, e in zip(got, want):
        assert rel_err(a, e) < 1e-2


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", ["q", "k", "v", "dout", "dmass"])
@pytest.mark.parametrize("m", [64, 136])
def test_values_that_are_not_finite_stay_where_the_scans_leave_them(cuda, where, value, m):
    """One such value makes the same gradients not finite as in one scan per
    view and gradient: those that depend on it, none on the other side of the
    causal mask."""
    from thetascan_amd._core.ops import scan_hip

    g = torch.Generator().manual_seed(5)
    B, H, T, dv = 1, 2, 200, 64
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda)  # noqa: E731
    ts = {"q": rnd(B, H, T, m).bfloat16(), "k": rnd(B, H, T, m).bfloat16(), "v": rnd(B, H, T, dv).bfloat16()}
    las = [None, torch.log(torch.tensor([0.9, 0.97], device=cuda)), torch.log(torch.tensor([0.99, 0.5], device=cuda))]
    dos, dms = [rnd(B, H, T, dv).bfloat16() for _ in las], [rnd(B, H, T) for _ in las]
    hit = {"dout": dos[1], "dmass": dms[1]}.get(where, ts.get(where))
    hit[(0, 1, 90, 3)[: hit.ndim]] = value
    need_r = [False] * 3

    def grads():
        return scan_hip._views_backward(ts["q"], ts["k"], ts["v"], las, dos, dms, True, True, True, need_r)[:3]

    got = grads()
    real = scan_hip.views_bwd_eligible
    try:
        scan_hip.views_bwd_eligible = lambda *a: False
        want = grads()
    finally:
        scan_hip.views_bwd_eligible = real
    for name, a, e in zip(("dq", "dk", "dv"), got, want):
        off = ~torch.isfinite(e.float())
        assert off.any() or (where, name) in {("q", "dq"), ("k", "dk"), ("v", "dv"), ("dmass", "dv")}, name
        assert torch.equal(~torch.isfinite(a.float()), off), name


def test_an_overflowed_score_is_infinite(cuda):
    """An upstream score dO . v past the largest float gives infinite gradients
    of its sign, as one scan per view gives, not NaN."""
    from thetascan_amd._core.ops import scan_hip

    g = torch.Generator().manual_seed(9)
    q, k, v, do = ((torch.rand(1, 1, 150, 64, generator=g) + 0.5) for _ in range(4))
    k[..., ::2] *= -1
    do[:, :, 20] *= 1e20
    v[:, :, 10] *= 1e20
    q, k, v, do = (t.to(cuda, torch.bfloat16) for t in (q, k, v, do))
    las = [None, torch.log(torch.tensor([0.9], device=cuda))]
    args = (q, k, v, las, [do, do], [None, None], True, True, True, [False, False])
    got = scan_hip._views_backward(*args)[:3]
    real = scan_hip.views_bwd_eligible
    try:
        scan_hip.views_bwd_eligible = lambda *a: False
        want = scan_hip._views_backward(*args)[:3]
    finally:
        scan_hip.views_bwd_eligible = real
    assert torch.isinf(want[0][0, 0, 20]).all() and torch.isinf(want[1][0, 0, 10]).all()
    for name, a, e in zip(("dq", "dk", "dv"), got, want):
        off = torch.isinf(e)
        assert not torch.isnan(e).any() and not torch.isnan(a).any(), name
        assert torch.equal(torch.isinf(a), off) and torch.equal(a[off].float(), e[off].float()), name


@pytest.mark.parametrize("layout", ["token_major", "padded", "one row for all tokens", "one value for all"])
def test_upstream_gradients_of_any_layout(cuda, layout):
    """Upstream gradients as autograd hands them on: rows of a projection or of
    a wider matrix, and broadcast ones (a sum's), give the contiguous copies'
    bits."""
    from thetascan_amd._core.ops import scan_hip

    g = torch.Generator().manual_seed(4)
    B, H, T, m, dv = 2, 2, 150, 72, 40
    rnd = lambda *s: torch.randn(*s, generator=g).to(cuda)  # noqa: E731

    def upstream():
        if layout == "token_major":
            return rnd(B, T, H, dv).bfloat16().transpose(1, 2), rnd(B, T, H).transpose(1, 2)
        if layout == "padded":
            return rnd(B, H, T, dv + 4).bfloat16()[..., 4:], rnd(B, H, T + 3)[..., 3:]
        if layout == "one row for all tokens":
            return rnd(B, H, 1, dv).bfloat16().expand(B, H, T, dv), rnd(B, H, 1).expand(B, H, T)
        return rnd(1).bfloat16().expand(B, H, T, dv), rnd(1).expand(B, H, T)

    q, k, v = rnd(B, H, T, m).bfloat16(), rnd(B, H, T, m).bfloat16(), rnd(B, H, T, dv).bfloat16()
    las = [None, torch.log(torch.tensor([0.9, 0.97], device=cuda)), torch.log(torch.tensor([0.99, 0.5], device=cuda))]
    dos, dms = zip(*(upstream() for _ in las))
    run = lambda dos, dms: scan_hip.views_bwd_launch(q, k, v, las, dos, dms, need_q=True, need_kv=True)  # noqa: E731
    for a, b in zip(run(dos, dms), run([t.contiguous() for t in dos], [t.contiguous() for t in dms])):
        assert torch.isfinite(a).all() and torch.equal(a, b)
