"""Feature widths of 192 and 384 on the wide feature kernels (GPU tests).

The published expanded kernel preset has m = 384 (192 trainable projection
rows, sign-expanded twice); a memory multiplier of 3 at head width 64, or of
6 at head width 32, gives m = 192.  These widths run the wide kernels in
bf16 (a token's whole feature row in registers).  Each mixer below runs
them on the multi-view path and is checked against the float64 oracle, across
both feature maps, input and feature RoPE, the learned ReLU^2 threshold,
shared key/query, banks, the ema stream and the plain sum, with a ragged last
tile.  ReLU^2 mixers take the bf16 bar, rel 2e-2, on outputs, dx and every
parameter gradient (measured at most 1.6e-2).  The softmax partition at
sharpness 8 multiplies the bf16 rounding of its pre-activations by 8: on the
same configurations the 64- and 128-wide feature kernels reach 2.4-2.5 % in dx
and the composed bf16 path 5-7 %, so the softmax mixers take 3e-2 (outputs,
dx) and 4e-2 (parameters); measured at most 2.9e-2 (m = 192) and 3.3e-2
(m = 384).
"""
from __future__ import annotations

import pytest
import torch

import thetascan_amd as ts
from oracle import mixer as oracle_mixer
from tests.conftest import rel_err
from tests.test_mixer_gpu import _headline_config, _seeded, build_module

pytestmark = pytest.mark.gpu


def _preset(d_model=128, heads=2):
    """kernel_expanded_reference_v0_1 at a small model width (head width 64, m = 384)."""
    pub = ts.ThetaScanConfig.kernel_expanded_reference_v0_1(d_model=d_model, n_heads=heads).to_dict()
    pub["runtime"].update(backend="hip", scan_chunk=64)
    return pub


def _case(name):
    if name == "preset_m384":
        return _preset()
    if name == "softmax_m192_feature_rope_ema":
        pub = _headline_config("feature", "none", "softmax_partition", d_model=128, heads=2, mult=3)
        pub["temporal"]["mode"] = "ema"
        return pub
    if name == "relu2_m192_d32_input_rope_sum":
        return _headline_config("input", "key_mass", "relu2_ridge", d_model=128, heads=4, mult=6)
    if name == "softmax_m384_stale_bank":
        pub = _headline_config("input", "key_mass", "softmax_partition", d_model=128, heads=2, mult=6)
        pub["temporal"].update(mode="bank", bank_mode="stale", recency_branches=2, retention_inits=[0.9, 0.99])
        return pub
    raise KeyError(name)


@pytest.mark.parametrize("name", ["preset_m384", "softmax_m192_feature_rope_ema", "relu2_m192_d32_input_rope_sum",
                                  "softmax_m384_stale_bank"])
def test_wide_feature_mixer_matches_float64_oracle(cuda, name):
    pub = _case(name)
    module = build_module(pub, cuda, torch.float32)
    _seeded(module, 5)
    with torch.no_grad():
        for pname, p in module._core.named_parameters():
            if pname in ("fade_eta", "kernel_relu2_threshold"):
                p.copy_(torch.randn(p.shape, generator=torch.Generator().manual_seed(6)) * 0.3)
    core = oracle_mixer.core_config(pub)
    assert core["mem_hidden"] in (192, 384)
    params64 = {k: v.detach().double().cpu().clone().requires_grad_(True) for k, v in module._core.named_parameters()}
    g = torch.Generator().manual_seed(7)
    B, T, D = 2, 150, pub["d_model"]
    x = torch.randn(B, T, D, generator=g, dtype=torch.float64)
    dy = torch.randn(B, T, D, generator=g, dtype=torch.float64) * 0.1
    x64 = x.clone().requires_grad_(True)
    y64 = oracle_mixer.forward(core, params64, x64)
    (y64 * dy).sum().backward()

    module = module.to(torch.bfloat16)
    xb = x.to(cuda, torch.bfloat16).requires_grad_(True)
    yb = module(xb)
    print(f"wide {name}: m={core['mem_hidden']} path={module._core.last_path}", flush=True)
    assert module._core.last_path == "fused"
    (yb.float() * dy.to(cuda, torch.float32)).sum().backward()
    tol, ptol = (3e-2, 4e-2) if "softmax" in name else (2e-2, 2e-2)
    assert rel_err(yb, y64) < tol
    assert rel_err(xb.grad, x64.grad) < tol
    for pname, p in module._core.named_parameters():
        if params64[pname].grad is not None and params64[pname].grad.abs().max() > 0:
            assert rel_err(p.grad, params64[pname].grad) < ptol, pname


def test_wide_widths_stay_on_the_composed_path_in_fp32(cuda):
    """The wide kernels are bf16 only: an fp32 mixer at m = 384 takes the
    composed path and still matches the oracle at the fp32 bar."""
    pub = _preset()
    module = build_module(pub, cuda, torch.float32)
    _seeded(module, 5)
    core = oracle_mixer.core_config(pub)
    params64 = {k: v.detach().double().cpu().clone().requires_grad_(True) for k, v in module._core.named_parameters()}
    g = torch.Generator().manual_seed(8)
    x = torch.randn(1, 70, pub["d_model"], generator=g, dtype=torch.float64)
    y64 = oracle_mixer.forward(core, params64, x)
    y = module(x.to(cuda, torch.float32))
    assert module._core.last_path == "composed"
    assert rel_err(y, y64) < 1e-3


@pytest.mark.parametrize("T", [1, 63, 65, 257])
@pytest.mark.parametrize("kind,m,d,feat_rot", [("relu2", 384, 64, 0), ("relu2", 192, 32, 64), ("softmax", 384, 64, 128),
                                               ("softmax", 192, 64, 0)])
def test_wide_features_at_tile_edges(cuda, T, kind, m, d, feat_rot):
    """Features, the query's residual read and every gradient at the edges of
    the 64-token groups, rows of a strided view, keys (no residual) and
    queries, against float64 autograd of the definition on the same bf16
    inputs.  The bf16 rounding of xn (2^-9 per entry) and of the outputs puts
    a ReLU^2 feature off by about 2 * 2^-8, a softmax one of sharpness 8 by 8
    times its pre-activation's error: 2-norm bars of 2e-2 and 4e-2; the
    gradients add dphi's and da's roundings (3e-2 and 6e-2)."""
    from thetascan_amd._core.ops.features import kernel_features
    from thetascan_amd._core.ops.fused import FeatureSpec
    from thetascan_amd import _lib

    B, H, eps = 2, 3, 1e-6
    g = torch.Generator().manual_seed(T + m + d)
    x = torch.randn(B, T, H, d, generator=g).bfloat16()
    w1 = (torch.randn(H, m, d, generator=g)).bfloat16()
    w2 = (torch.randn(H, d, m, generator=g) * 0.3).bfloat16()
    tau = torch.randn(H, generator=g) * 0.1
    dphi = torch.randn(B, H, T, m, generator=g).bfloat16()
    dres = torch.randn(B, H, T, d, generator=g).bfloat16()
    in_rot = d // 2

    def turn(v, rot):
        inv = 1.0 / (10_000.0 ** (torch.arange(0, rot, 2, dtype=torch.float64) / rot))
        f = torch.outer(torch.arange(T, dtype=torch.float64), inv)
        a, b = v[..., :rot:2], v[..., 1:rot:2]
        r = torch.stack((a * f.cos() - b * f.sin(), a * f.sin() + b * f.cos()), -1).flatten(-2)
        return torch.cat((r, v[..., rot:]), -1)

    for resid in (False, True):
        leaves = [t.double().clone().requires_grad_(True) for t in (x, w1, w2, tau)]
        lx, l1, l2, lt = leaves
        xr = turn(lx.transpose(1, 2), in_rot)
        xn = xr / xr.norm(dim=-1, keepdim=True).clamp_min(eps)
        a = xn @ l1.transpose(-1, -2)
        pre = a * torch.rsqrt(a.square().mean(-1, keepdim=True) + eps) - lt.view(1, H, 1, 1)
        if kind == "relu2":
            f = torch.relu(pre).square()
            h = f / f.sum(-1, keepdim=True)
        else:
            h = torch.softmax(8.0 * pre, -1)
        phi = turn(h, feat_rot) if feat_rot else h
        r64 = xn + h @ l2.transpose(-1, -2)
        loss = (phi * dphi.double()).sum() + ((r64 * dres.double()).sum() if resid else 0.0)
        loss.backward()

        dev = [t.to(cuda).requires_grad_(True) for t in (x, w1, w2, tau)]
        spec = FeatureSpec(_lib.FEAT_RELU2 if kind == "relu2" else _lib.FEAT_SOFTMAX, m, 8.0, in_rot, feat_rot,
                           10_000.0, 1.0, eps)
        got, base = kernel_features(dev[0].transpose(1, 2), dev[1], dev[2] if resid else None, dev[3], spec, resid)
        out = (got.float() * dphi.to(cuda).float()).sum()
        if resid:
            out = out + (base.float() * dres.to(cuda).float()).sum()
        out.backward()
        torch.cuda.synchronize()

        def err(t, ref):
            return float((t.double().cpu() - ref).norm() / ref.norm())

        bar, gbar = (2e-2, 3e-2) if kind == "relu2" else (4e-2, 6e-2)
        errs = {"phi": err(got.detach(), phi.detach())}
        if resid:
            errs["resid"] = err(base.detach(), r64.detach())
        grads = {n: err(t.grad, l.grad) for n, t, l in zip(("dx", "dw1", "dw2", "dtau"), dev, leaves)
                 if l.grad is not None and (n != "dtau" or kind == "relu2")}  # (a shift leaves a softmax as it is)
        print(f"wide {kind} m={m} d={d} T={T} resid={resid}: {errs} {grads}", flush=True)
        assert all(e < bar for e in errs.values()), errs
        assert all(e < gbar for e in grads.values()), grads
