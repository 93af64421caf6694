"""The backbone over whole sequences in plain inference (MemoryPoolLM.apply
under no_grad): mpl_dense_layers against the oracle's layer_norm, dense,
gelu_tanh and silu and mpl_causal_attention against softmax attention, both in
fp64, around the edges of their tiles; and the fused forward against the
general path, which a call with gradients enabled takes."""

import numpy as np
import pytest
import torch

from model_amd import _lib
from model_amd.model import MemoryPoolLM, ModelConfig, _fused_forward_pays, causal_attention, dense_layers
from oracle import backbone as ob

pytestmark = pytest.mark.gpu

ACTS = {None: lambda v: v, "gelu_tanh": ob.gelu_tanh, "silu": ob.silu}


@pytest.mark.parametrize("rows,K,widths,acts,out_in,ln,mul,residual,joined", [
    (1, 4, [4], [None], False, False, False, False, False),              # the smallest of each
    (64, 64, [64], [None], False, False, False, True, False),            # one tile, one chunk
    (65, 68, [68], ["silu"], False, True, False, False, False),          # one past in rows, K and columns
    (63, 60, [60], ["gelu_tanh"], False, True, True, True, False),       # one short of each
    (200, 256, [256, 256, 256], [None, None, None], False, True, False, False, True),   # query, key, value
    (130, 256, [1024, 256], [None, "silu"], False, True, False, False, False),          # router and gate
    (129, 1024, [256], [None], False, False, False, True, False),        # feed-forward output
    (100, 300, [20, 4, 132], ["silu", None, "gelu_tanh"], False, True, False, False, False),
    (70, 128, [516], [None], True, True, False, False, False),           # embedding table layout
    (70, 36, [100], [None], True, False, True, True, False),
])
def test_dense_layers_match_oracle(gpu_lib, rows, K, widths, acts, out_in, ln, mul, residual, joined):
    """fp32 sums of K terms: within 2e-5 of the result's largest magnitude, as
    mpl_rows_linear."""
    rng = np.random.default_rng(rows * 31 + K)
    f32 = lambda *s: rng.standard_normal(s).astype(np.float32)  # noqa: E731
    x = f32(rows, K) * np.float32(1.5) + np.float32(0.3)
    Ws = [f32(n, K) * np.float32(K ** -0.5) if out_in else f32(K, n) * np.float32(K ** -0.5) for n in widths]
    bs = [f32(n) if i % 2 == 0 else None for i, n in enumerate(widths)]
    lnp = {"scale": 1 + np.float32(0.1) * f32(K), "bias": np.float32(0.1) * f32(K)} if ln else None
    m = f32(rows, K) if mul else None
    res = f32(rows, widths[0]) if residual else None
    cu = lambda t: None if t is None else torch.tensor(t, device="cuda")  # noqa: E731
    got = dense_layers(cu(x), [(cu(w), cu(b), a) for w, b, a in zip(Ws, bs, acts)], x_mul=cu(m), residual=cu(res),
                       ln=None if lnp is None else {k: cu(v) for k, v in lnp.items()}, out_in=out_in, joined=joined)
    a = x.astype(np.float64)
    if ln:
        a = ob.layer_norm(a, {k: v.astype(np.float64) for k, v in lnp.items()})
    if mul:
        a = a * m.astype(np.float64)
    want = []
    for w, b, act, n in zip(Ws, bs, acts, widths):
        w = w.astype(np.float64)
        y = ACTS[act](ob.dense(a, {"kernel": w.T if out_in else w, "bias": np.zeros(n) if b is None else b}))
        want.append(y + res if residual else y)
    if joined:
        want = [np.concatenate(want, 1)]
    for y, g in zip(want, got):
        np.testing.assert_allclose(g.cpu().numpy(), y, rtol=0, atol=2e-5 * np.abs(y).max())


@pytest.mark.parametrize("out_in,ln,mul", [(False, False, False), (True, False, False), (False, True, False),
                                           (False, False, True), (True, True, True)])
def test_dense_layers_every_chunk_count(gpu_lib, out_in, ln, mul):
    """The contraction runs in chunks of 32, a main loop of two at a time and
    up to five after it: every count from one chunk to eleven, whole and with
    a rest, on more row tiles than the 8 XCDs and a rest."""
    g = torch.Generator(device="cuda").manual_seed(5)
    R = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    rows, N = 64 * 9 + 5, 68
    for K in sorted({k for c in range(1, 12) for k in (32 * c - 28, 32 * c)}):
        x, w, b = R(rows, K), R(N, K) if out_in else R(K, N), R(N)
        m = R(rows, K) if mul else None
        lnp = {"scale": R(K), "bias": R(K)} if ln else None
        got, = dense_layers(x, [(w, b, None)], ln=lnp, x_mul=m, out_in=out_in)
        a = x.double()
        if ln:
            a = torch.nn.functional.layer_norm(a, (K,), lnp["scale"].double(), lnp["bias"].double(), 1e-6)
        a = a * m.double() if mul else a
        want = a @ (w.double().t() if out_in else w.double()) + b.double()
        # fp32 sums of K terms, as above
        assert float((got - want).abs().max()) <= 2e-5 * float(want.abs().max()), K


@pytest.mark.parametrize("B,T,H,hd", [(1, 1, 1, 32), (2, 31, 3, 32), (3, 32, 2, 64), (2, 33, 4, 64), (1, 100, 2, 128),
                                      (2, 129, 1, 64), (1, 300, 2, 32)])
def test_causal_attention_matches_softmax(gpu_lib, B, T, H, hd):
    """Scores of hd terms enter an exponential: an absolute error of hd * 2^-24
    times the largest |q||k| a score, the same relative error a weight; 4e-6
    covers it for these scores (|s| < 16) with the sums' own."""
    g = torch.Generator().manual_seed(T + hd)
    qkv = torch.randn((B, T, 3, H, hd), generator=g)
    qkv[:, T // 2:, 1] *= 3.0  # sharper rows: the running maximum moves between key blocks
    got = causal_attention(qkv.reshape(B, T, -1).cuda(), H, hd ** -0.5).cpu().double().reshape(B, T, H, hd)
    q, k, v = (qkv[:, :, i].double().permute(0, 2, 1, 3) for i in range(3))
    s = (q * hd ** -0.5) @ k.transpose(-1, -2).contiguous()
    s = s.masked_fill(~torch.ones((T, T), dtype=torch.bool).tril(), -float("inf"))
    want = (torch.softmax(s, -1) @ v).permute(0, 2, 1, 3)
    assert float((got - want).abs().max()) <= 4e-6 * max(1.0, float(s[s > -1e30].abs().max())) * float(v.abs().max())


def test_unsupported_shapes_are_reported(gpu_lib):
    L = _lib.lib()
    s = torch.cuda.current_stream().cuda_stream
    assert L.mpl_causal_attention(None, 1, 8, 2, 48, 1.0, None, s) == 4 and b"head_dim" in L.mpl_last_error()
    with pytest.raises(_lib.MplError, match="width"):
        dense_layers(torch.zeros((8, 8), device="cuda"), [(torch.zeros((8, 6), device="cuda"), None, None)])


@pytest.mark.parametrize("B,T,heads,memory_ffn,use_memory,pool_off", [
    (3, 40, 2, False, True, False), (1, 1, 4, True, True, False), (2, 65, 4, True, True, True),
    (2, 33, 2, False, False, False)])
def test_fused_forward_equals_general_path(gpu_lib, B, T, heads, memory_ffn, use_memory, pool_off):
    """fp32 tables, so that a change of rounding cannot move a selected slot
    but at a tie of its scores; the same fp32 rounding through 3 layers, 1e-4
    as the backbone's test against the oracle."""
    cfg = ModelConfig(vocab_size=400, max_len=80, d_model=128, n_layers=3, n_heads=heads, ffn_mult=2,
                      use_memory=use_memory, memory_layers=(0, 2), memory_ffn=memory_ffn, n_sub_keys=24, pool_heads=2,
                      d_key=32, d_value=64, top_k=8, values_dtype=torch.float32)
    model = MemoryPoolLM(cfg)
    params = model.init(3)
    tokens = torch.randint(0, 400, (B, T), generator=torch.Generator().manual_seed(1)).cuda()
    with torch.no_grad():
        assert model._fused_forward_ok(params["params"], tokens)
        got, aux = model.apply(params, tokens, pool_off=pool_off)
    want, aux2 = model.apply(params, tokens, pool_off=pool_off)  # gradients enabled: the general path
    assert not model._fused_forward_ok(params["params"], tokens)
    torch.testing.assert_close(got, want.detach(), rtol=1e-4, atol=1e-4)
    if use_memory and not pool_off:
        assert all(torch.equal(a, b) for a, b in zip(aux["slots"], aux2["slots"]))
    # transforms and modes take the general path
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.float16):
        assert not model._fused_forward_ok(params["params"], tokens)


def _small_model(**kw):
    cfg = ModelConfig(**{**dict(vocab_size=400, max_len=80, d_model=128, n_layers=2, n_heads=2, ffn_mult=2,
                                use_memory=True, memory_layers=(1,), memory_ffn=True, n_sub_keys=24, pool_heads=2,
                                d_key=32, d_value=64, top_k=8, values_dtype=torch.float32), **kw})
    model = MemoryPoolLM(cfg)
    tokens = torch.randint(0, cfg.vocab_size, (2, 33), generator=torch.Generator().manual_seed(2)).cuda()
    return model, model.init(4), tokens


def test_pool_off_without_memory_parameters(gpu_lib):
    """pool_off reads no parameter of the memory layers: they may be missing."""
    model, params, tokens = _small_model()
    want = model.apply(params, tokens, pool_off=True)[0].detach()  # gradients enabled: the general path
    bare = {k: v for k, v in params["params"].items() if k not in ("router_1", "mem_gate_1", "mem_out_1", "pool")}
    with torch.no_grad():
        assert model._fused_forward_ok(bare, tokens, True)
        got, aux = model.apply({"params": bare}, tokens, pool_off=True)
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4)


def test_shapes_the_general_path_refuses_stay_refused(gpu_lib):
    """A kernel of the right number of elements in another shape (saved as
    [out, in], say) is an error, not a product with its elements in another
    order."""
    for name, shape in (("ffn_in_0", (256, 128)), ("ffn_out_1", (128, 256)), ("router_1", (128, 2, 32)),
                        ("mem_gate_1", (64, 128)), ("mem_out_1", (128, 64))):
        model, params, tokens = _small_model()
        params["params"][name]["kernel"] = params["params"][name]["kernel"].reshape(shape)
        with torch.no_grad(), pytest.raises(RuntimeError):
            model.apply(params, tokens)
    for part in ("scale", "bias"):
        model, params, tokens = _small_model()
        params["params"]["ln_ffn_0"][part] = params["params"]["ln_ffn_0"][part][None]
        with torch.no_grad(), pytest.raises(RuntimeError):
            model.apply(params, tokens)


def test_shapes_the_general_path_broadcasts_are_taken(gpu_lib):
    """A gate of one column, biases of one element and a hidden layer whose
    width is no multiple of 4: accepted, with the general path's result."""
    model, params, tokens = _small_model()
    p = params["params"]
    g = torch.Generator(device="cuda").manual_seed(7)
    p["mem_gate_1"] = {"kernel": p["mem_gate_1"]["kernel"][:, :1].contiguous(), "bias": p["mem_gate_1"]["bias"][:1]}
    p["ffn_out_1"]["bias"] = torch.randn(1, generator=g, device="cuda")
    p["ffn_in_0"] = {"kernel": p["ffn_in_0"]["kernel"][:, :250].contiguous(), "bias": p["ffn_in_0"]["bias"][:250]}
    p["ffn_out_0"]["kernel"] = p["ffn_out_0"]["kernel"][:250]
    want = model.apply(params, tokens)[0].detach()
    with torch.no_grad():
        got = model.apply(params, tokens)[0]
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("vocab,dtype", [(401, torch.float32), (402, torch.float16), (400, torch.float16)])
def test_any_vocabulary(gpu_lib, vocab, dtype):
    """The tables are read by torch's own indexing and product, so a vocabulary
    that is no multiple of 4, or a table at an odd word, takes the fused
    launches too.  With fp16 pool tables, which the library stores by default,
    a last-bit difference of a query can move a component's fp16 rounding by
    a step: a score by 2^-11 * T * |q_i k_i| (T = 10, unit rows of 16: under
    1.5e-3), a weight by that share, a near tie's slot.  So those compare the
    tokens with the same slots, within 2e-3."""
    model, params, tokens = _small_model(vocab_size=vocab, values_dtype=dtype)
    p = params["params"]
    p["embed"]["embedding"] = torch.cat([p["pos_embed"].new_zeros(1), p["embed"]["embedding"].reshape(-1)])[1:]
    p["embed"]["embedding"] = p["embed"]["embedding"].reshape(vocab, 128)
    want, aux2 = model.apply(params, tokens)
    with torch.no_grad():
        assert model._fused_forward_ok(p, tokens)
        got, aux = model.apply(params, tokens)
    same = (aux["slots"][0].sort(-1).values == aux2["slots"][0].sort(-1).values).flatten(2).all(-1)
    assert bool(same.all()) if dtype == torch.float32 else float(same.float().mean()) > 0.8
    tol = 1e-4 if dtype == torch.float32 else 2e-3
    torch.testing.assert_close(got[same], want.detach()[same], rtol=tol, atol=tol)


def test_wide_short_calls_take_the_general_path(gpu_lib):
    """At widths where the library's products are faster than the fused ones
    only calls that win it back (long sequences, few tokens) are fused."""
    model, params, tokens = _small_model(d_model=2048, n_heads=32, n_layers=1, ffn_mult=1, memory_layers=())
    with torch.no_grad():
        assert not model._fused_forward_ok(params["params"], tokens)
    pays = [(128, 4, 64, 4096), (896, 7, 16, 512), (1024, 16, 1, 1024), (1024, 16, 16, 512), (1280, 20, 1, 128),
            (2048, 32, 2, 2048)]
    costs = [(1024, 8, 64, 256), (1280, 10, 16, 64), (1280, 10, 16, 1024), (2048, 32, 1, 16), (2048, 32, 4, 1024)]
    assert all(_fused_forward_pays(*c) for c in pays) and not any(_fused_forward_pays(*c) for c in costs)
