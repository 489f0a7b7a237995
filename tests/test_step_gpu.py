"""ts_memory_step and ts_skinny_linear: a decode step of the one-call kernel
memory (GPU tests).

A mixer fed a prompt and then pieces of at most eight tokens (the step kernel)
must continue the sequence that one whole call computes in float64: every
padded head width and feature count that a memory can have, both maps, both reads, with and without
the output gate and the learned threshold, RoPE at either placement.  Bars:
fp32 2e-5 (fp32 sums in another order), bf16 2e-2 (the activations' rounding).
The skinny product: fp32 accumulation of bf16 products, one rounding (8e-3 of
the largest value).
"""
from __future__ import annotations

import pytest
import torch

from oracle import mixer as oracle_mixer
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


def _config(head_dim, mult, feature_map, norm, rope, gate, threshold=False):
    import thetascan_amd as ts

    return ts.ThetaScanConfig(
        d_model=2 * head_dim, n_heads=2, memory_multiplier=mult, family="kernel", output_gate=gate,
        kernel=ts.KernelConfig(feature_map=feature_map, read_normalization=norm,
                               relu2_threshold_mode="learned_per_head" if threshold else "none"),
        rope=ts.RoPEConfig() if rope is None else ts.RoPEConfig(mode="partial", fraction=0.5, placement=rope))


CASES = [
    (64, 1, "relu2_ridge", "none", "feature", True, False),
    (64, 2, "relu2_ridge", "key_mass", "input", True, True),
    (16, 1, "softmax_partition", "key_mass", None, False, False),
    (32, 2, "softmax_partition", "none", "feature", True, False),
    (128, 1, "relu2_ridge", "key_mass", "input", False, True),
]


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2e-2)])
@pytest.mark.parametrize("case", CASES)
def test_step_continues_the_sequence(cuda, case, dtype, tol):
    import thetascan_amd as ts
    from thetascan_amd import _lib

    cfg = _config(*case)
    torch.manual_seed(1)
    module = ts.ThetaScan(cfg)
    g = torch.Generator().manual_seed(2)
    with torch.no_grad():
        for _, p in sorted(module.named_parameters()):
            p.add_(torch.randn(p.shape, generator=g) * 0.05)
    module = module.to(dtype)
    B, T = 3, 90
    x = torch.randn(B, T, cfg.d_model, generator=g).to(dtype)
    params = {k: v.detach().double() for k, v in module._core.named_parameters()}
    want = oracle_mixer.forward(oracle_mixer.core_config(cfg.to_dict()), params, x.double(), backend="chunk")
    module = module.to(cuda)
    xd, got = x.to(cuda), []
    with torch.no_grad(), _lib.record_launches() as recs:
        y, state = module(xd[:, :67], state=module.initial_state())
        got.append(y)
        t = 67
        for n in (1, 8, 3, 1, 8, 2):
            before = [c.clone() for c in state._tensors()]
            y, new = module(xd[:, t:t + n], state=state)
            assert all(torch.equal(a, b) for a, b in zip(state._tensors(), before))  # the given state is unchanged
            state, t = new, t + n
            got.append(y)
        # a first call of few tokens starts from a zero state
        first, _ = module(xd[:, :5], state=module.initial_state())
    assert t == T and state.position == T
    assert sum(r[0] == "ts_memory_step" for r in recs) == 7
    assert rel_err(torch.cat(got, 1), want) < tol
    assert rel_err(first, want[:, :5]) < tol


@pytest.mark.parametrize("n,k,na,nb", [(1, 512, 1536, 512), (8, 512, 512, 0), (17, 32, 16, 16), (64, 160, 48, 0),
                                       (5, 1024, 64, 32)])
def test_skinny_linear(cuda, n, k, na, nb):
    from thetascan_amd._core.ops import step

    g = torch.Generator().manual_seed(n + k)
    x, wa, wb = (torch.randn(r, k, generator=g).to(torch.bfloat16) for r in (n, na, max(nb, 1)))
    want = x.double() @ torch.cat([wa, wb[:nb]]).double().t()
    got = step._linear(x.to(cuda), wa.to(cuda), wb.to(cuda) if nb else None)
    assert got.shape == (n, na + nb)
    assert rel_err(got, want) < 8e-3
    # rows beyond the kernel's limit take the library product
    many = step._linear(x.to(cuda).repeat(66, 1), wa.to(cuda), None)
    assert rel_err(many[:n], want[:, :na]) < 8e-3


def _same_values_unaligned(p):
    buf = p.new_empty(p.numel() + 1)[1:].view_as(p)
    buf.copy_(p)
    return buf


def test_other_continuations_keep_their_path(cuda):
    """Nine tokens, and parameters that the kernel cannot read (another dtype,
    memory order or alignment), take the multi-view path and give its values."""
    from thetascan_amd import _lib

    module, state, x = _prompted(cuda, torch.float32)
    nine = torch.cat([x, x[:, :1]], 1)
    with torch.no_grad():
        pieces, s = [], state
        for t in range(9):
            y, s = module(nine[:, t:t + 1], state=s)
            pieces.append(y)
        with _lib.record_launches() as recs:
            y, _ = module(nine, state=state)
        assert "ts_memory_step" not in {r[0] for r in recs}
        assert rel_err(y, torch.cat(pieces, 1)) < 2e-5
        core = module._core
        bias = core.ogate.g.lin.bias
        changes = [(bias, bias.data.to(torch.bfloat16).to(torch.float64)),
                   (core.proj_qkv.weight, core.proj_qkv.weight.data.t().contiguous().t()),
                   (core.proj_out.weight, _same_values_unaligned(core.proj_out.weight.data))]
        for param, other in changes:
            held, param.data = param.data, other
            if other.dtype == torch.float64:
                held = other.float()  # the same numbers in the kernel's dtype
            with _lib.record_launches() as recs:
                y, new = module(x[:, :2], state=state)
            assert "ts_memory_step" not in {r[0] for r in recs}
            param.data = held
            with _lib.record_launches() as recs:
                want, ref = module(x[:, :2], state=state)
            assert "ts_memory_step" in {r[0] for r in recs}
            assert rel_err(y, want) < 2e-5
            for a, b in zip(new._tensors(), ref._tensors()):
                assert rel_err(a, b) < 2e-5


def test_fewer_features_than_channels_are_refused(cuda):
    """No memory has them: the kernels are built without that combination (a
    host check, before any launch)."""
    import ctypes

    from thetascan_amd import _lib

    t = torch.zeros(4096, device=cuda)
    s = _lib.strided(t.view(1, 1, 32, 128))
    desc = _lib.MemoryStepDesc(1, 1, 1, 128, 64, _lib.dtype_code(t.dtype), _lib.dtype_code(t.dtype), _lib.FEAT_RELU2,
                               0, 0, 0, 0, 1.0, 1.0, 1e-6, 0)
    p = t.data_ptr()
    io = _lib.MemoryStepIO(s, s, s, _lib.strided(None), s, p, p, None, None, None, None, None, None, None)
    status = _lib.load().ts_memory_step(ctypes.byref(desc), ctypes.byref(io), _lib.stream_handle(cuda))
    with pytest.raises(NotImplementedError, match="below the head width"):
        _lib.check(status, "ts_memory_step")


def _prompted(cuda, dtype, case=CASES[0], seed=3, batch=3):
    """A mixer of ``case`` on the GPU, its state after a prompt of 20 tokens and the next 8 tokens."""
    import thetascan_amd as ts

    torch.manual_seed(seed)
    module = ts.ThetaScan(_config(*case))
    g = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for _, p in sorted(module.named_parameters()):
            p.add_(torch.randn(p.shape, generator=g) * 0.05)  # (the output projection starts at zero)
    module = module.to(cuda, dtype)
    x = torch.randn(batch, 28, module.config.d_model, generator=g).to(cuda, dtype)
    with torch.no_grad():
        _, state = module(x[:, :20], state=module.initial_state())
    return module, state, x[:, 20:].contiguous()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("change", [-32, 32])
def test_another_input_width_is_refused(cuda, dtype, change):
    """An input of another width than the projection's rows raises, as its
    product always did, before any launch of the step."""
    from thetascan_amd import _lib
    from thetascan_amd._core.ops import step

    module, state, x = _prompted(cuda, dtype)
    D = x.shape[-1]
    other = torch.randn(3, 1, D + change, device=cuda).to(dtype)
    before = [c.clone() for c in state._tensors()]
    with torch.no_grad(), _lib.record_launches() as recs:
        with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
            module(other, state=state)
        with pytest.raises(RuntimeError, match="shapes cannot be multiplied"):
            step._linear(other.view(3, -1), module._core.proj_qkv.weight, None)
    assert not recs
    assert all(torch.equal(a, b) for a, b in zip(state._tensors(), before))


def _layouts(x):
    """The values of x [B,T,D] in other memory orders, by name."""
    B, T, D = x.shape
    wide = x.new_zeros(B, T, 2 * D)
    wide[..., ::2] = x
    padded = x.new_zeros(B, T, D + 4)
    padded[..., :D] = x
    longer = x.new_zeros(B, T + 7, D)
    longer[:, 7:] = x
    channels = x.new_zeros(B, D, 16)
    channels[..., 8:8 + T] = x.transpose(1, 2)
    return {
        "every second channel": wide[..., ::2],
        "rows of a wider buffer": padded[..., :D],
        "the last tokens of a longer sequence": longer[:, 7:],
        "channel-major": channels[..., 8:8 + T].transpose(1, 2),
        "batch innermost": x.permute(1, 2, 0).contiguous().permute(2, 0, 1),
        "one sequence for all": x[:1].expand(B, T, D),
    }


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 3])
def test_inputs_of_any_layout(cuda, dtype, tokens):
    """An input of any strides gives what its contiguous copy gives, in the
    output and in the carried state.  Bars: fp32 1e-5 (a product's sums in
    another order), bf16 1e-2 (its one rounding carried to the output)."""
    module, state, x = _prompted(cuda, dtype)
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    for name, view in _layouts(x[:, :tokens]).items():
        same = view.clone(memory_format=torch.contiguous_format)
        with torch.no_grad():
            y, new = module(view, state=state)
            want, ref = module(same, state=state)
        assert rel_err(y, want) < tol, name
        for a, b in zip(new._tensors(), ref._tensors()):
            assert rel_err(a, b) < tol, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tokens", [1, 8])
def test_autocast(cuda, dtype, tokens):
    """Under autocast to bf16 an fp32 mixer's projections are bf16: its steps
    take the multi-view path, which follows them, and match the fp32 step at
    bf16's bar; a bf16 mixer keeps its step."""
    from thetascan_amd import _lib

    module, state, x = _prompted(cuda, dtype)
    with torch.no_grad():
        want, ref = module(x[:, :tokens], state=state)
        with torch.autocast("cuda", torch.bfloat16), _lib.record_launches() as recs:
            y, new = module(x[:, :tokens], state=state)
    assert ("ts_memory_step" in {r[0] for r in recs}) == (dtype == torch.bfloat16)
    assert y.dtype == torch.bfloat16
    assert rel_err(y, want) < 2e-2
    for a, b in zip(new._tensors(), ref._tensors()):
        assert rel_err(a, b) < 2e-2


def test_parameters_on_another_device_are_refused(cuda):
    """A mixer left on the host raises on a GPU input, as its product always did."""
    import thetascan_amd as ts

    module = ts.ThetaScan(_config(*CASES[0]))
    x = torch.randn(2, 1, module.config.d_model, device=cuda)
    with torch.no_grad(), pytest.raises(RuntimeError, match="same device"):
        module(x, state=module.initial_state())


def test_states_as_the_scan_takes_them(cuda):
    """A carried state is taken in the forms the scan takes: folded batch and
    head axes, another memory order; a captured step, which writes its state in
    place, refuses one it could not write."""
    import dataclasses

    import thetascan_amd as ts

    module, state, x = _prompted(cuda, torch.float32)
    (block,), = state.carries
    with torch.no_grad():
        want, ref = module(x[:, :1], state=state)
        turned = block.transpose(2, 3).contiguous().transpose(2, 3)
        for other in (block.flatten(0, 1), turned):
            y, new = module(x[:, :1], state=dataclasses.replace(state, carries=([other],)))
            assert torch.equal(y, want)
            assert torch.equal(new.carries[0][0], ref.carries[0][0])
        with pytest.raises(ValueError, match="contiguous"):
            ts.DecodeGraph(module, dataclasses.replace(state, carries=([turned],)))


@pytest.mark.parametrize("tokens", [1, 9])
def test_expanded_weights_are_formed_once(cuda, monkeypatch, tokens):
    """A call forms its expanded weights once, whichever path takes it."""
    import dataclasses

    import thetascan_amd as ts

    cfg = dataclasses.replace(_config(64, 2, "relu2_ridge", "none", "feature", True), feature_expansion=2)
    module = ts.ThetaScan(cfg).to(cuda)
    core, formed = module._core, []
    weights = core._weights
    monkeypatch.setattr(core, "_weights", lambda: formed.append(1) or weights())
    x = torch.randn(2, tokens, cfg.d_model, device=cuda)
    with torch.no_grad():
        module(x, state=module.initial_state())
    assert len(formed) == 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", [CASES[2], (32, 1, "softmax_partition", "none", "input", True, False)])
def test_an_infinite_value_spreads_as_in_the_multi_view_path(cuda, monkeypatch, case, dtype):
    """Feature counts below the kernel's padded width: an infinite value makes
    the reads that see it infinite, not NaN (the padding's zeros stay out)."""
    from thetascan_amd._core.ops import step

    module, state, x = _prompted(cuda, dtype, case)
    cfg = module.config
    with torch.no_grad():
        # channel 5 of head 1's values overflows for the tokens whose first channel is large
        w = module._core.proj_qkv.weight
        w[2 * cfg.d_model + cfg.d_model // 2 + 5, 0] = 3e38
        x = x.clone()
        x[..., 0] = 0.0
        x[1, 1, 0] = 16.0
        y, new = module(x[:, :3], state=state)
        monkeypatch.setattr(step, "eligible", lambda *a: False)
        want, ref = module(x[:, :3], state=state)
    assert torch.isinf(want[1, 1:]).any() and not torch.isnan(want).any()
    assert torch.equal(torch.isinf(y), torch.isinf(want)) and not torch.isnan(y).any()
    for a, b in zip(new._tensors(), ref._tensors()):
        assert torch.equal(torch.isinf(a), torch.isinf(b)) and torch.equal(torch.isnan(a), torch.isnan(b))
