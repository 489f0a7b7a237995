"""Mixers under autocast (GPU tests): an fp32 mixer whose shared key/query
projection adds an fp32 bias has fp32 reads beside a bf16 output gate, which no
read epilogue may take as fp32 rows.  The output matches the call without
autocast at bf16's bar."""
from __future__ import annotations

import pytest
import torch

from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recording", [True, False])
@pytest.mark.parametrize("family", ["kernel", "gn"])
@pytest.mark.parametrize("mode,branches", [("sum", 1), ("ema", 1), ("bank", 1), ("bank", 2)])
def test_fp32_mixer_with_shared_projections(cuda, family, mode, branches, recording):
    import thetascan_amd as ts

    temporal = ts.TemporalConfig(mode=mode, recency_branches=branches,
                                 retention_inits=(0.9, 0.99)[:branches] if mode == "bank" else None)
    cfg = ts.ThetaScanConfig(d_model=128, n_heads=2, memory_multiplier=1, share_key_query=True, family=family,
                             temporal=temporal, kernel=ts.KernelConfig(feature_map="relu2_ridge"))
    torch.manual_seed(0)
    module = ts.ThetaScan(cfg)
    g = torch.Generator().manual_seed(1)
    with torch.no_grad():
        for _, p in sorted(module.named_parameters()):
            p.add_(torch.randn(p.shape, generator=g) * 0.05)
    module = module.to(cuda)
    x = torch.randn(2, 70, 128, generator=g).to(cuda)
    with torch.set_grad_enabled(recording):
        want = module(x)
        with torch.autocast("cuda", torch.bfloat16):
            y = module(x)
    assert rel_err(y, want) < 3e-2
