"""GPU tests of the chunked fp32 kernels of the rules with a decay (gated and KDA, D in {64,
128}: the backward from 16 tokens, the forward of fp32 q/k/v from 160) against the fp64
oracles at the fp32 bounds, at the edges of their 16-token chunks and of the spans of chunks,
and against the per-token kernels that every other call runs.

The backward's plan follows the pairs n (batch x heads) and the chunks of 16 tokens c: a
workgroup of its sweep takes 16 columns up to n D/16 = 256 and 32 above, a span is 8 chunks
where n ceil(c / 8) >= 256, else 4 where n ceil(c / 4) >= 256, else 2."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import gated_oracle as gref
from prometheus_amd import _native, kernels, synth
from tests.parity import assert_f32_parity

pytestmark = pytest.mark.gpu

NAMES = ("gq", "gk", "gv", "gbeta", "gg", "gstate")


def _dev(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda()


def _case(shape, seed, chan, dtype="fp32", scale=0.3, state=True):
    x = synth.fwd_inputs(shape, seed=seed, dtype=dtype, s0_std=0.05 if state else None)
    rng = np.random.default_rng(seed + 1)
    b, t, h, d = shape
    g = (-scale * np.abs(rng.standard_normal(shape if chan else shape[:3]))).astype(np.float32)
    go = rng.standard_normal(shape).astype(np.float32)
    gs = (rng.standard_normal((b, h, d, d)) * 0.05).astype(np.float32)
    return x, g, go, gs


def _bwd(x, g, go, gs, chan):
    def qkv(name):
        bits = getattr(x, name + "_bits")
        if bits is None:
            return _dev(getattr(x, name))
        return torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda()

    b, _, h, d = x.q.shape
    s0 = _dev(x.s0) if x.s0 is not None else torch.zeros((b, h, d, d), device="cuda")
    gd = g if isinstance(g, torch.Tensor) else _dev(g)
    res = kernels._GatedDeltaResidual(q=qkv("q"), k=qkv("k"), v=qkv("v"), beta=_dev(x.beta), g=gd, state0=s0, chunk=64)
    f = kernels.chunked_kda_rule_bwd if chan else kernels.chunked_gated_delta_rule_bwd
    return [t.cpu().numpy() for t in f(res, (_dev(go), _dev(gs)))]


def _check(x, g, go, gs, chan, what):
    got = _bwd(x, g, go, gs, chan)
    exp = (gref.kda_vjp if chan else gref.gated_vjp)(x.q, x.k, x.v, x.beta, g, go, gs, x.s0)
    for name, a, e in zip(NAMES, got, exp):
        assert_f32_parity(a, e, f"{what} {name}", scaled=True)


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("t,d", [(16, 128), (17, 64), (31, 64), (64, 128), (127, 64), (128, 128), (129, 64), (273, 128)])
def test_edges_of_chunks_and_spans(t, d, chan):
    """Whole and partial chunks, one chunk up to several spans (of two chunks here; longer ones
    below), with and without a state."""
    x, g, go, gs = _case((1, t, 3, d), t + d + chan, chan, state=t % 2 == 0)
    _check(x, g, go, gs, chan, f"T{t} D{d}")


@pytest.mark.parametrize("chan", [0, 1])
@pytest.mark.parametrize("d", [64, 128])
def test_every_length_from_a_chunk_on_is_served(d, chan):
    """The bf16 entry point, which the chunked kernels alone serve, takes the workspace that the
    size function gives for every length from 16 tokens on, and refuses shorter ones."""
    lib = _native.lib()
    size = lib.pm_kda_delta_bwd_workspace_bytes if chan else lib.pm_gated_delta_bwd_workspace_bytes
    p = torch.zeros(1 << 20, device="cuda").data_ptr()
    for t in (*range(15, 49), 64, 129):
        n = size(1, t, 3, d, _native.DTYPE_BF16)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        rc = lib.pm_delta_bwd_bf16(p, p, p, p, p, None, None, None, p, p, p, p, p, p, 1, t, 3, d, chan,
                                   ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
        assert rc == (0 if t >= 16 else _native.E_UNSUPPORTED), t
    torch.cuda.synchronize()


@pytest.mark.parametrize("chan", [False, True])
def test_bf16_inputs_in_fp32_arithmetic(chan):
    x, g, go, gs = _case((2, 145, 2, 128), 7, chan, dtype="bf16")
    _check(x, g, go, gs, chan, "bf16")


def test_decays_of_every_strength_side_by_side():
    """Channels that forget everything (alpha 0 and 1e-9), that keep everything (g = 0), that
    grow a little, and one strong decay in the middle of a chunk before weak ones: no factor
    is formed from a difference or quotient that the strong one would spoil."""
    x, g, go, gs = _case((1, 90, 2, 64), 17, True, scale=0.05)
    g[..., 0], g[..., 1], g[..., 2], g[..., 3] = -np.inf, -20.0, 0.0, 0.02
    g[:, 37, :, 8:24] = -60.0
    _check(x, g, go, gs, True, "mixed decays")


@pytest.mark.parametrize("chan", [False, True])
def test_against_the_per_token_kernels(chan):
    """Missing cotangents, several pairs per XCD slot, bitwise repeatable; a gate tensor that
    is not 16-byte aligned keeps its (per-token or chunked) route and its result."""
    shape = (3, 200, 5, 64)
    x, g, go, gs = _case(shape, 29, chan)
    for cot in ((go, gs), (None, gs), (go, None)):
        got = _bwd(x, g, *cot, chan)
        again = _bwd(x, g, *cot, chan)
        off = torch.empty(g.size + 1, device="cuda")[1:].copy_(_dev(g).flatten()).view(g.shape)
        shifted = _bwd(x, off, *cot, chan)
        with _native.use_knobs(1, 0):
            ref = _bwd(x, g, *cot, chan)
        for name, a, b, c, e in zip(NAMES, got, again, shifted, ref):
            np.testing.assert_array_equal(a, b, err_msg=name)
            assert_f32_parity(a, e, name, scaled=True)
            assert_f32_parity(c, e, f"shifted gate {name}", scaled=True)


def _fwd(x, g, chan, **kw):
    f = kernels.chunked_kda_rule if chan else kernels.chunked_gated_delta_rule
    gd = g if isinstance(g, torch.Tensor) else _dev(g)
    return [t.float().cpu().numpy() for t in f(_dev(x.q), _dev(x.k), _dev(x.v), _dev(x.beta), gd, _dev(x.s0), **kw)]


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("t,d,h", [(160, 128, 3), (161, 64, 9), (175, 128, 1), (333, 64, 4), (200, 128, 66)])
def test_forward_edges(t, d, h, chan):
    """Whole and partial chunks, both tile widths (66 pairs of D 128 take 32 columns), with and
    without a state; bf16 O is the fp32 one rounded."""
    x, g, _, _ = _case((1, t, h, d), t + d + chan, chan, state=t % 2 == 0)
    got = _fwd(x, g, chan)
    exp = (gref.kda_delta_rule if chan else gref.gated_delta_rule)(x.q, x.k, x.v, x.beta, g, x.s0)
    for name, a, e in zip(("o", "state"), got, exp):
        assert_f32_parity(a, e, f"T{t} D{d} {name}")
    with _native.use_knobs(0, 16):
        narrow = _fwd(x, g, chan)
    half = _fwd(x, g, chan, out_dtype=torch.bfloat16)
    np.testing.assert_array_equal(narrow[0], got[0])
    np.testing.assert_array_equal(half[0], torch.from_numpy(got[0]).bfloat16().float().numpy())
    np.testing.assert_array_equal(half[1], got[1])


def test_forward_decays_of_every_strength_and_routes():
    """Channels at alpha 0, 1e-9, 1 and above 1 with a strong decay inside a chunk; a gate that is
    not 16-byte aligned and other paths keep the per-token kernel; T = 0 passes the state."""
    x, g, _, _ = _case((1, 170, 2, 64), 17, True, scale=0.05)
    g[..., 0], g[..., 1], g[..., 2], g[..., 3] = -np.inf, -20.0, 0.0, 0.02
    g[:, 37, :, 8:24] = -60.0
    exp = gref.kda_delta_rule(x.q, x.k, x.v, x.beta, g, x.s0)
    off = torch.empty(g.size + 1, device="cuda")[1:].copy_(_dev(g).flatten()).view(g.shape)
    got, shifted = _fwd(x, g, True), _fwd(x, off, True)
    with _native.use_knobs(1, 0):
        per_token = _fwd(x, g, True)
    for name, a, b, c, e in zip(("o", "state"), got, shifted, per_token, exp):
        assert_f32_parity(a, e, name)
        np.testing.assert_array_equal(b, c)
    lib = _native.lib()
    f32, bf16 = _native.DTYPE_F32, _native.DTYPE_BF16
    assert lib.pm_decay_fwd_workspace_bytes(1, 170, 2, 64, f32) == 2 * 11 * (3 * 16 * 64 + 512 + 64) * 4
    for args in ((1, 159, 2, 64, f32), (1, 170, 2, 48, f32), (1, 170, 2, 64, bf16), (1, 170, 256, 64, f32)):
        assert lib.pm_decay_fwd_workspace_bytes(*args) == 0


def _alike(shape, seed, chan, rho, beta, dtype="fp32"):
    """Unit keys of mutual cosine rho^2 (rho 1: one repeated key a head), constant beta."""
    x, g, go, gs = _case(shape, seed, chan, dtype, scale=0.1)
    rng = np.random.default_rng(seed)

    def unit(z):
        return z / np.linalg.norm(z, axis=-1, keepdims=True)

    common = unit(rng.standard_normal((shape[0], 1, *shape[2:])))
    k = unit(rho * common + np.sqrt(1 - rho * rho) * unit(rng.standard_normal(shape)))
    x.k, x.k_bits = synth._cast(k.astype(np.float32), dtype)
    x.beta = np.full(shape[:3], beta, np.float32)
    return x, g, go, gs


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("rho,beta", [(0.8, 0.9), (0.95, 1.0), (1.0, 0.9), (1.0, 1.0), (1.0, 1.9), (0.95, 1.95)])
@pytest.mark.parametrize("shape,dtype", [((1, 256, 2, 64), "fp32"), ((1, 170, 2, 128), "fp32"), ((1, 100, 2, 128), "bf16")])
def test_alike_keys(shape, dtype, rho, beta, chan):
    """Repeated and near-repeated keys, up to betas where the powers of diag(beta) A' are large
    and the inverse of I + diag(beta) A' is not: forward (fp32) and all gradients."""
    x, g, go, gs = _alike(shape, 3, chan, rho, beta, dtype)
    if dtype == "fp32":
        exp = (gref.kda_delta_rule if chan else gref.gated_delta_rule)(x.q, x.k, x.v, x.beta, g, x.s0)
        for name, a, e in zip(("o", "state"), _fwd(x, g, chan), exp):
            assert_f32_parity(a, e, name)
    what = f"rho {rho} beta {beta}"
    if chan:
        _check(x, g, go, gs, chan, what)
        return
    got = _bwd(x, g, go, gs, chan)
    exp = gref.gated_vjp(x.q, x.k, x.v, x.beta, g, go, gs, x.s0)
    for name, a, e in zip(NAMES, got, exp):
        if name != "gg":
            assert_f32_parity(a, e, f"{what} {name}", scaled=True)
    # a head's gg sums its channels', which cancel where one key is repeated at beta 1 (the
    # per-token kernels' error there is 3e-6 of the sum): each channel's to 1e-5
    channels = gref.kda_vjp(x.q, x.k, x.v, x.beta, np.repeat(g[..., None], shape[3], -1), go, gs, x.s0)[4]
    assert np.linalg.norm(got[4] - exp[4]) <= 1e-5 * np.linalg.norm(channels), what


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("gate", [-1.0, -3.0, -5.0, -8.0, -12.0, -20.0])
@pytest.mark.parametrize("d", [64, 128])
def test_gate_gradient_of_strong_decays(d, gate, chan):
    """dL/dg alone, where every gate is equally strong and where single tokens are, among weak
    ones: it is about alpha times the sums that it must not be a difference of."""
    vjp = gref.kda_vjp if chan else gref.gated_vjp
    x, g, go, gs = _case((1, 150, 2, d), 11, chan)
    g = np.full_like(g, gate)
    exp = vjp(x.q, x.k, x.v, x.beta, g, go, gs, x.s0)[4]
    assert_f32_parity(_bwd(x, g, go, gs, chan)[4], exp, "all gates")
    g = (-0.1 * np.abs(np.random.default_rng(1).standard_normal(g.shape))).astype(np.float32)
    rows = [5, 20, 37, 64, 127, 149]
    g[:, rows] = gate
    got, exp = _bwd(x, g, go, gs, chan), vjp(x.q, x.k, x.v, x.beta, g, go, gs, x.s0)
    for name, a, e in zip(NAMES, got, exp):
        assert_f32_parity(a, e, name, scaled=True)
    assert_f32_parity(got[4][:, rows], exp[4][:, rows], "the strong tokens' gates")


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("shape", [(2, 520, 16, 64), (4, 505, 16, 64)])
def test_gate_gradient_of_strong_decays_in_long_spans(shape, chan):
    """Spans of four chunks (the first shape) and eight, whose strong chunks find their start state
    in the span's, in its middle's and in those kept per chunk: strong gates in every chunk of
    one head, in every other chunk of the next, in single tokens of the rest; against the
    per-token kernels, the strong tokens' gates apart."""
    x, g, go, gs = _case(shape, 3, chan, scale=0.1)
    strong = np.zeros(shape[:3], bool)
    strong[:, :, 0] = True
    strong[:, :, 1] = (np.arange(shape[1]) // 16 % 2 == 1)[None]
    strong[:, ::29, 2:] = True
    g[strong] = -6.0
    got = _bwd(x, g, go, gs, chan)
    with _native.use_knobs(1, 0):
        exp = _bwd(x, g, go, gs, chan)
    for name, a, e in zip(NAMES, got, exp):
        assert_f32_parity(a, e, name, scaled=True)
    for h in range(4):
        sel = strong[:, :, h]
        assert_f32_parity(got[4][:, :, h][sel], exp[4][:, :, h][sel], f"head {h}")


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("d,token", [(64, 105), (128, 96), (128, 111)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "g", "go", "s0", "gs"])
def test_infinities_and_nans_reach_what_they_reach_token_by_token(what, value, d, token, chan):
    """One infinity or NaN in an input: the outputs and gradients that the per-token kernels leave
    finite stay so (v: the tokens before it, and the other columns; q and dO: those after it),
    with their values, and no other becomes finite."""
    x, g, go, gs = _case((1, 200, 2, d), 5, chan, scale=0.1)
    x.q, x.k, x.v = x.q.copy(), x.k.copy(), x.v.copy()
    a = {"q": x.q, "k": x.k, "v": x.v, "beta": x.beta, "g": g, "go": go, "s0": x.s0, "gs": gs}[what]
    a[(0, 1, 7, token % d) if what in ("s0", "gs") else (0, token, 1, 7)[: a.ndim]] = value
    res = []
    for path in (0, 1):
        with _native.use_knobs(path, 0):
            res.append(_fwd(x, g, chan) + _bwd(x, g, go, gs, chan))
    for name, a, e in zip(("o", "state", *NAMES), *res):
        np.testing.assert_array_equal(np.isfinite(a), np.isfinite(e), err_msg=name)
        ok = np.isfinite(e)
        assert_f32_parity(a[ok], e[ok], name, scaled=True)


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
@pytest.mark.parametrize("d,h,t", [
    # 34 pairs of D = 128 and 66 of 64: 32 columns; spans of eight chunks, the last one of
    # 1, 4, 5 and 8, the last chunk whole or partial
    (128, 34, 912), (128, 34, 955), (128, 34, 971), (128, 34, 1024),
    (64, 66, 400), (64, 66, 443), (64, 66, 459), (64, 66, 512),
    # ... spans of four, the last one of 1, 2, 3 and 4
    (128, 34, 464), (128, 34, 475), (64, 66, 235), (64, 66, 256),
    # 16 columns, spans of eight
    (64, 64, 505), (128, 32, 1010)])
def test_plans_of_large_calls(d, h, t, dtype, chan):
    """Each form of the sweep and each span length, against the per-token kernels."""
    x, g, go, gs = _case((1, t, h, d), t + chan, chan, dtype, scale=0.1)
    got = _bwd(x, g, go, gs, chan)
    with _native.use_knobs(1, 0):
        exp = _bwd(x, g, go, gs, chan)
    for name, a, e in zip(NAMES, got, exp):
        assert_f32_parity(a, e, name, scaled=True)


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("d,h,t", [(64, 128, 165), (64, 255, 176), (64, 127, 161), (128, 40, 200)])
def test_forward_plans_of_large_calls(d, h, t, chan):
    """The forward's automatic 32 columns (128 pairs of D = 64 on, 33 of 128) and the last
    call on 16, against the per-token kernel."""
    x, g, _, _ = _case((1, t, h, d), t + chan, chan, scale=0.1)
    got = _fwd(x, g, chan)
    with _native.use_knobs(1, 0):
        exp = _fwd(x, g, chan)
    for name, a, e in zip(("o", "state"), got, exp):
        assert_f32_parity(a, e, name)


@pytest.mark.parametrize("chan", [False, True])
@pytest.mark.parametrize("dtype", ["fp32", "bf16"])
def test_views_at_odd_offsets_run_the_chunked_backward(dtype, chan):
    """Slices of packed buffers give the aligned tensors' gradients bit for bit (the per-token
    kernels' differ in rounding)."""
    x, g, go, gs = _case((2, 70, 3, 64), 31, chan, dtype)

    def shifted(t):
        return torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].copy_(t.flatten()).view(t.shape)

    def run(place):
        def qkv(name):
            bits = getattr(x, name + "_bits")
            return _dev(getattr(x, name)) if bits is None else torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda()

        ins = [place(qkv(n)) for n in "qkv"] + [_dev(x.beta), place(_dev(g)), _dev(x.s0)]
        res = kernels._GatedDeltaResidual(*ins, chunk=64)
        f = kernels.chunked_kda_rule_bwd if chan else kernels.chunked_gated_delta_rule_bwd
        return f(res, (place(_dev(go)), _dev(gs)))

    for name, a, b in zip(NAMES, run(shifted), run(lambda t: t)):
        assert torch.equal(a, b), name
