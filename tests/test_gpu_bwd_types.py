"""GPU tests of the backward's result types and of the model's backward.

``pm_delta_bwd_bf16``: bf16 gradients are the fp32 entry points' rounded once. The model's
``linear_attention`` backward (``pm_linear_attention_bwd``): the fp64 VJP of the recurrence on
normalised rows (oracle/delta_oracle.delta_vjp) taken through x / max(||x||, 1e-6) in NumPy."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import delta_oracle as ref
from prometheus_amd import _native, kernels, model, synth
from tests.parity import assert_bf16_parity, assert_f32_parity

pytestmark = pytest.mark.gpu


def _bf(bits):
    return torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda()


def _f(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda()


@pytest.mark.parametrize("rule", ["delta", "gated", "kda"])
@pytest.mark.parametrize("shape", [(1, 64, 3, 128), (2, 150, 2, 64), (1, 17, 9, 128)])
def test_bf16_gradients_are_the_fp32_ones_rounded(rule, shape):
    """Autograd with bf16 leaves (the bf16 entry point) against the explicit pair's fp32
    gradients, bit for bit; the other gradients stay fp32 and equal."""
    x = synth.fwd_inputs(shape, seed=sum(shape), dtype="bf16", s0_std=0.02)
    rng = np.random.default_rng(3)
    leaves = [_bf(x.q_bits), _bf(x.k_bits), _bf(x.v_bits), _f(x.beta)]
    if rule != "delta":
        leaves.append(_f(-0.2 * np.abs(rng.standard_normal(shape if rule == "kda" else shape[:3]))))
    leaves = [t.requires_grad_(True) for t in (*leaves, _f(x.s0))]
    go, gs = _f(rng.standard_normal(shape)), _f(0.05 * rng.standard_normal(x.s0.shape))
    name = {"delta": "chunked_delta_rule", "gated": "chunked_gated_delta_rule", "kda": "chunked_kda_rule"}[rule]
    got = torch.autograd.grad(getattr(kernels, name)(*leaves), leaves, (go, gs))
    _, res = getattr(kernels, name + "_fwd")(*(t.detach() for t in leaves), kernels.LinearAttnConfig())
    exp = getattr(kernels, name + "_bwd")(res, (go, gs))
    for i, (a, e, leaf) in enumerate(zip(got, exp, leaves)):
        assert a.dtype == leaf.dtype and e.dtype == torch.float32
        assert torch.equal(a, e.to(a.dtype)), (rule, i)


def test_bf16_gradients_off_the_chunked_paths():
    """Other head dimensions and the per-token path: the entry point refuses, autograd casts."""
    x = synth.fwd_inputs((1, 20, 2, 48), seed=5, dtype="bf16", s0_std=0.02)
    leaves = [t.requires_grad_(True) for t in (_bf(x.q_bits), _bf(x.k_bits), _bf(x.v_bits), _f(x.beta), _f(x.s0))]
    out = kernels.chunked_delta_rule(*leaves)
    go, gs = torch.randn_like(out[0]), torch.randn_like(out[1])
    got = torch.autograd.grad(out, leaves, (go, gs))
    _, res = kernels.chunked_delta_rule_fwd(*(t.detach() for t in leaves), kernels.LinearAttnConfig())
    for a, e in zip(got, kernels.chunked_delta_rule_bwd(res, (go, gs))):
        assert torch.equal(a, e.to(a.dtype))
    p = torch.zeros(1 << 16, device="cuda").data_ptr()
    with _native.use_knobs(1, 0):
        assert _native.lib().pm_delta_bwd_bf16(p, p, p, p, None, p, p, p, p, p, p, p, None, p, 1, 4, 1, 64, 0, p,
                                               1 << 18, None) == _native.E_UNSUPPORTED


def _model_grads(q, k, v, go, gs, s0):
    """fp64: the recurrence's VJP on the normalised rows, then the normalisation's."""
    def norm(x):
        n = np.linalg.norm(x, axis=-1, keepdims=True)
        return x / np.maximum(n, 1e-6), n

    q, k = q.astype(np.float64), k.astype(np.float64)
    (qh, qn), (kh, kn) = norm(q), norm(k)
    gq, gk, gv, _, gs0 = ref.delta_vjp(qh, kh, v, np.ones(q.shape[:3]), go, gs, s0)

    def back(g, xh, n):
        live = n >= 1e-6
        return np.where(live, (g - xh * (xh * g).sum(-1, keepdims=True)) / np.maximum(n, 1e-6), g / 1e-6)

    return back(gq, qh, qn), back(gk, kh, kn), gv, gs0


@pytest.mark.parametrize("dtype,dim", [("fp32", 16), ("fp32", 48), ("fp32", 64), ("fp32", 128), ("fp32", 256),
                                       ("bf16", 64), ("bf16", 128), ("bf16", 40)])
@pytest.mark.parametrize("tokens", [1, 75])
def test_linear_attention_backward(dtype, dim, tokens):
    """Every row layout (8 to 32 lanes a row, and the element-wise kernel), with a state."""
    shape = (2, tokens, 3, dim)
    x = synth.fwd_inputs(shape, seed=dim + tokens, dtype=dtype, s0_std=0.05, normalize=False)
    rng = np.random.default_rng(dim)
    go, gs = rng.standard_normal(shape), 0.05 * rng.standard_normal(x.s0.shape)
    go, gs = go.astype(np.float32), gs.astype(np.float32)
    qkv = [_bf(b) for b in (x.q_bits, x.k_bits, x.v_bits)] if dtype == "bf16" else [_f(a) for a in (x.q, x.k, x.v)]
    leaves = [t.requires_grad_(True) for t in (*qkv, _f(x.s0))]
    got = torch.autograd.grad(model.linear_attention(*leaves), leaves, (_f(go), _f(gs)))
    exp = _model_grads(x.q, x.k, x.v, go, gs, x.s0)
    for name, a, e, leaf in zip(("gq", "gk", "gv", "gs0"), got, exp, leaves):
        assert a.dtype == leaf.dtype
        if dtype == "fp32":
            assert_f32_parity(a.cpu().numpy(), e, name, scaled=True)
        else:
            assert_bf16_parity(a.float().cpu().numpy(), e, name)


def test_linear_attention_backward_of_zero_and_tiny_rows():
    """Rows below the norm's bound: dL/dx = dL/d(x / 1e-6) / 1e-6, no norm term; no output
    gradient on some tokens; the other rows as usual."""
    shape = (1, 40, 2, 64)
    x = synth.fwd_inputs(shape, seed=9, dtype="fp32", normalize=False)
    q, k = x.q.copy(), x.k.copy()
    k[0, 7], q[0, 9], k[0, 11] = 0.0, 0.0, k[0, 11] * 1e-9
    go = np.random.default_rng(1).standard_normal(shape).astype(np.float32)
    go[0, 20:25] = 0.0
    leaves = [_f(a).requires_grad_(True) for a in (q, k, x.v)]
    o, _ = model.linear_attention(*leaves)
    got = torch.autograd.grad(o, leaves, _f(go))
    exp = _model_grads(q, k, x.v, go, None, None)
    rows = np.ones(40, bool)
    rows[[7, 9, 11]] = False  # their gradients are a million times the others': apart
    for name, a, e in zip(("gq", "gk", "gv"), got, exp):
        a = a.cpu().numpy()
        assert_f32_parity(a[:, rows], e[:, rows], name, scaled=True)
        assert_f32_parity(a[:, ~rows], e[:, ~rows], name + " small rows", scaled=True)


@pytest.mark.parametrize("dim", [16, 64, 128])
def test_linear_attention_backward_of_a_nan_row(dim):
    """A query row with one NaN: its whole gradient row is NaN, as the elementwise normalisation's
    reverse gives it, and only the rows of that head can be affected."""
    shape = (1, 20, 2, dim)
    x = synth.fwd_inputs(shape, seed=dim, dtype="fp32", normalize=False)
    q = x.q.copy()
    q[0, 19, 1, 3] = np.nan
    leaves = [_f(a).requires_grad_(True) for a in (q, x.k, x.v)]
    o, _ = model.linear_attention(*leaves)
    gq, gk, gv = torch.autograd.grad(o, leaves, torch.ones_like(o))
    assert gq[0, 19, 1].isnan().all()
    assert all(t[:, :, 0].isfinite().all() for t in (gq, gk, gv))


def test_linear_attention_backward_under_saved_tensor_hooks():
    """Saved tensors that come back in another memory layout give the same gradients."""
    shape = (2, 37, 3, 64)
    x = synth.fwd_inputs(shape, seed=4, dtype="fp32", normalize=False)
    leaves = [_f(a).requires_grad_(True) for a in (x.q, x.k, x.v)]
    go = torch.randn(shape, device="cuda")
    exp = torch.autograd.grad(model.linear_attention(*leaves)[0], leaves, go)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.transpose(1, 2).contiguous(), lambda t: t.transpose(1, 2)):
        o = model.linear_attention(*leaves)[0]
    for a, e in zip(torch.autograd.grad(o, leaves, go), exp):
        assert torch.equal(a, e)


@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("dim", [5, 16, 48, 64, 96, 128, 160, 256])
def test_linear_attention_backward_normalises_as_tensor_operations_do(dtype, dim):
    """Bit for bit the reverse kernels on rows normalised by elementwise tensor operations and
    those operations' own reverse, rows at and below the norm's bound among them: a sum of
    squares in another order moves the rounding of the normalised rows to bf16, and with it the
    gradients by 1e-3."""
    shape = (2, 67, 3, dim)
    x = synth.fwd_inputs(shape, seed=dim, dtype=dtype, s0_std=0.05, normalize=False)
    qkv = [_bf(b) for b in (x.q_bits, x.k_bits, x.v_bits)] if dtype == "bf16" else [_f(a) for a in (x.q, x.k, x.v)]
    qkv[0][0, 3], qkv[1][1, 5], qkv[0][1, 9] = 0.0, qkv[1][1, 5] * 1e-9, 0.0
    qkv[0][1, 9, :, 0] = 1e-6
    s0 = _f(x.s0)
    go, gs = torch.randn(shape, device="cuda"), 0.05 * torch.randn(s0.shape, device="cuda")
    leaves = [t.requires_grad_(True) for t in (*qkv, s0)]
    got = torch.autograd.grad(model.linear_attention(*leaves), leaves, (go, gs))

    def norm(t):
        return t / torch.clamp_min(torch.linalg.vector_norm(t, dim=-1, keepdim=True), 1e-6)

    raw = [t.detach().float().requires_grad_(True) for t in qkv[:2]]
    rows = [norm(t) for t in raw]
    res = kernels._DeltaResidual(q=rows[0].detach().to(qkv[0].dtype), k=rows[1].detach().to(qkv[0].dtype),
                                 v=qkv[2].detach(), beta=torch.ones(shape[:3], device="cuda"), state0=s0.detach(), chunk=64)
    gqn, gkn, gv, _, gs0 = kernels.chunked_delta_rule_bwd(res, (go, gs))
    exp = (*torch.autograd.grad(rows, raw, (gqn, gkn)), gv, gs0)
    for name, a, e in zip(("gq", "gk", "gv", "gs0"), got, exp):
        assert torch.equal(a, e.to(a.dtype)), (name, (a != e.to(a.dtype)).sum().item())
