"""The whole-prompt pass on two-term fp16 planes: the exponents that a layer's activations get from its weights (launch_prefill_bounds) hold for weights of very
different sizes, are made again when a tensor is loaded again, and travel to handles that share the weights."""
import numpy as np
import pytest

import oracle
from golden_io import assert_model_close
from zig_gpt2_amd import gpt as zgpt
from zig_gpt2_amd import synth

pytestmark = pytest.mark.gpu


def uneven(cfg, seed, bf16):
    """Weights whose layers' activations lie many binades apart: large and small gains and biases, rows of a matrix far smaller than the others."""
    w = {k: np.array(v, np.float32) for k, v in synth.make_weights(cfg, seed=seed, bf16=bf16).items()}
    rng = np.random.default_rng(seed)
    for l in range(cfg.n_layer):
        p = f"h{l}."
        w[p + "ln_1_g"] *= np.float32(2.0 ** int(rng.integers(-6, 7)))
        w[p + "ln_2_g"] *= np.float32(2.0 ** int(rng.integers(-6, 4)))
        w[p + "ln_2_b"] += np.float32(0.5)
        w[p + "c_fc_w"] = w[p + "c_fc_w"].reshape(4 * cfg.n_embed, cfg.n_embed)
        w[p + "c_fc_w"][::3] *= np.float32(2.0 ** -14)
        v = w[p + "c_attn_w"].reshape(3, cfg.n_embed, cfg.n_embed)
        v[0] *= np.float32(0.25 / abs(w[p + "ln_1_g"]).max())  # (scores of an ordinary size)
        v[2, ::5] *= np.float32(2.0 ** 6)
        w[p + "c_attn_w"] = v.reshape(3 * cfg.n_embed, cfg.n_embed)
        if bf16:
            for k in ("c_fc_w", "c_attn_w"):
                bits = synth.to_bf16_bits(w[p + k])
                w[p + k] = (bits.astype(np.uint32) << 16).view(np.float32).reshape(w[p + k].shape)
    return w


@pytest.mark.parametrize("name,batch,n,bf16,route", [("tiny", 1, 33, True, 0), ("tiny3", 2, 47, False, 0), ("nano-char", 2, 129, True, 1), ("nano-char", 1, 70, False, 1),
                                                     ("xl-slice", 1, 95, True, 2), ("medium-slice", 1, 64, False, 2), ("xl-slice", 1, 40, False, 3)])
def test_weights_of_very_different_sizes(zg, name, batch, n, bf16, route):
    cfg = synth.CONFIGS[name]
    w = uneven(cfg, 61, bf16)
    m = zgpt.GPT(cfg, batch=batch, weights_f32=not bf16)
    m.load_weights(w)
    toks = np.stack([synth.rand_tokens(610 + b, n + 1, cfg.vocab_size) for b in range(batch)])
    zg.zg_debug_prefill_route(route, 0)
    try:
        lg = m.prefill(toks[:, :n]).copy()
    finally:
        zg.zg_debug_prefill_route(0, 0)
    nxt = m.forward(n + 1, toks[:, n])
    for b in range(batch):
        ref = oracle.GPT(cfg, w).forced_logits(toks[b], n - 1)
        assert_model_close(ref[0], lg[b], f"{name} uneven weights, row {b}")
        assert_model_close(ref[1], nxt[b], f"{name} uneven weights, decode, row {b}")
    m.close()


@pytest.mark.parametrize("batch,n", [(8, 250), (5, 255)])
def test_tiles_of_128_columns(zg, batch, n):
    """fp32 weights and one to two thousand rows: the ring kernel's 128 x 128 tiles (qkv with the cache append, GELU, slabs) against the persistent GEMM.
    Both are within some 5e-7 of the exact logits, in the 2-norm."""
    cfg = synth.CONFIGS["nano-char"]
    m = zgpt.GPT(cfg, batch=batch, weights_f32=True)
    m.load_weights(synth.make_weights(cfg, seed=64, bf16=False))
    toks = np.stack([synth.rand_tokens(640 + b, n + 1, cfg.vocab_size) for b in range(batch)])
    got = []
    for route in (0, 1):
        zg.zg_debug_prefill_route(route, 0)
        try:
            lg = m.prefill(toks[:, :n]).copy()
        finally:
            zg.zg_debug_prefill_route(0, 0)
        got.append(np.concatenate([lg, m.forward(n + 1, toks[:, n])]).astype(np.float64))
    m.close()
    assert np.linalg.norm(got[0] - got[1]) <= 2e-6 * np.linalg.norm(got[1])


def test_a_tensor_loaded_again(zg):
    cfg = synth.CONFIGS["tiny3"]
    toks = synth.rand_tokens(62, 40, cfg.vocab_size)
    m = zgpt.GPT(cfg)
    m.load_weights(synth.make_weights(cfg, seed=62, bf16=True))
    m.prefill([toks])
    w = uneven(cfg, 63, True)  # other planes, other exponents
    m.load_weights(w)
    other = zgpt.GPT(cfg, batch=2, share_weights_with=m)
    ref = oracle.GPT(cfg, w).forced_logits(toks, len(toks) - 1)[0]
    assert_model_close(ref, other.prefill(np.stack([toks, toks]))[1], "a handle that shares the weights")
    assert_model_close(ref, m.prefill([toks])[0], "loaded again")
    other.close()
    m.close()


def test_two_plane_handles_round_their_activations_to_16_bits(zg):
    """What ZG_GPT_PREFILL_2PLANE asks for: 2^-17 of an activation, beside the 2^-23 of the default."""
    cfg = synth.CONFIGS["nano-char"]
    w = synth.make_weights(cfg, seed=64, bf16=True)
    toks = synth.rand_tokens(640, 130, cfg.vocab_size)
    ref = oracle.GPT(cfg, w).forced_logits(toks, len(toks) - 1)[0].astype(np.float64)
    err = []
    for planes in (3, 2):
        m = zgpt.GPT(cfg, prefill_planes=planes)
        m.load_weights(w)
        err.append(np.linalg.norm(m.prefill([toks])[0] - ref) / np.linalg.norm(ref))
        m.close()
    assert err[0] < 2e-6 < err[1] < 1e-4, err


@pytest.mark.parametrize("name,batch,n,bf16,route,wgs", [("nano-char", 1, 70, True, 1, 0), ("nano-char", 1, 70, False, 1, 0), ("nano-char", 4, 250, True, 1, 16),
                                                         ("nano-char", 4, 250, False, 1, 16), ("nano-char", 2, 70, True, 2, 0), ("nano-char", 2, 70, False, 2, 0),
                                                         ("nano-char", 2, 70, True, 3, 0), ("nano-char", 2, 70, False, 3, 0)])
def test_rows_of_zeros_and_of_next_to_nothing(zg, monkeypatch, name, batch, n, bf16, route, wgs):
    """Outputs whose weights are all zero (pruned ones), or so small that nothing is left of them beside the bias, are the bias.  (16 workgroups: 24 tiles of the
    c_attn Linear, the last eight in halves that meet.)"""
    cfg = synth.CONFIGS[name]
    E = cfg.n_embed
    w = {k: np.array(v, np.float32) for k, v in synth.make_weights(cfg, seed=65, bf16=bf16).items()}
    rng = np.random.default_rng(65)
    for l in range(cfg.n_layer):
        for k, rows in (("c_attn", 3 * E), ("c_fc", 4 * E)):
            m = w[f"h{l}.{k}_w"].reshape(rows, E)
            for i, size in enumerate((0.0, 2.0 ** -140, 2.0 ** -118, 2.0 ** -100, 2.0 ** -60, 0.0)):
                m[i::23] *= np.float32(size)
            m[7::23] = 0.0
            w[f"h{l}.{k}_w"] = m
            w[f"h{l}.{k}_b"] = rng.normal(0.0, 0.05, rows).astype(np.float32)
        w[f"h{l}.c_proj_w"] = w[f"h{l}.c_proj_w"].reshape(E, E)
        w[f"h{l}.c_proj_w"][3] = 0.0
    if wgs:
        monkeypatch.setenv("ZGPT2_GEMM_WGS", str(wgs))
    m = zgpt.GPT(cfg, batch=batch, weights_f32=not bf16)
    m.load_weights(w)
    toks = np.stack([synth.rand_tokens(650 + b, n + 1, cfg.vocab_size) for b in range(batch)])
    zg.zg_debug_prefill_route(route, 0)
    try:
        lg = m.prefill(toks[:, :n]).copy()
    finally:
        zg.zg_debug_prefill_route(0, 0)
    nxt = m.forward(n + 1, toks[:, n])  # (the cache)
    m.close()
    for b in {0, batch - 1}:
        ref = oracle.GPT(cfg, w).forced_logits(toks[b], n - 1)
        assert_model_close(ref[0], lg[b], f"rows of zeros, row {b}")
        assert_model_close(ref[1], nxt[b], f"rows of zeros, decode, row {b}")


def exact_logits(cfg, w, toks):
    """The last position's logits in 64 bits."""
    E, H = cfg.n_embed, cfg.n_heads
    w = {k: np.asarray(v, np.float64) for k, v in w.items()}

    def norm(x, p):
        d = x - x.mean(-1, keepdims=True)
        return d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-5) * w[p + "_g"] + w[p + "_b"]

    n = len(toks)
    x = w["wte"].reshape(-1, E)[toks.astype(np.int64)] + w["wpe"].reshape(-1, E)[:n]
    for l in range(cfg.n_layer):
        p = f"h{l}."
        q, k, v = (norm(x, p + "ln_1") @ w[p + "c_attn_w"].reshape(3 * E, E).T + w[p + "c_attn_b"]).reshape(n, 3, H, E // H).transpose(1, 2, 0, 3)
        s = q @ k.transpose(0, 2, 1) / np.sqrt(E // H)
        s = np.where(np.tri(n, dtype=bool), s, -np.inf)
        s = np.exp(s - s.max(-1, keepdims=True))
        o = (s / s.sum(-1, keepdims=True) @ v).transpose(1, 0, 2).reshape(n, E)
        x = x + o @ w[p + "c_proj_w"].reshape(E, E).T + w[p + "c_proj_b"]
        h = norm(x, p + "ln_2") @ w[p + "c_fc_w"].reshape(4 * E, E).T + w[p + "c_fc_b"]
        h = 0.5 * h * (1.0 + np.tanh(0.7978845608 * (h + 0.044715 * h ** 3)))
        x = x + h @ w[p + "mlp_proj_w"].reshape(E, 4 * E).T + w[p + "mlp_proj_b"]
    return norm(x[-1:], "ln_f")[0] @ w["wte"].reshape(-1, E).T


@pytest.mark.parametrize("name,n,route", [("tiny", 33, 2), ("nano-char", 70, 1), ("nano-char", 70, 3), ("medium-slice", 40, 2)])
def test_rows_whose_mean_is_far_above_their_spread(zg, name, n, route):
    """A residual stream around 100 that varies by 0.02: E[x^2] - mean^2 has no correct digit in 32 bits, and a normed row could be any multiple of sqrt(E), beyond what
    the planes' exponent allows.  (The last bias takes the stream back: the head's own norm is the decode kernels'.)
    The bound: the mean's rounding is 2^-22 of 100, a thousandth of the spread."""
    cfg = synth.CONFIGS[name]
    w = {k: np.array(v, np.float32) for k, v in synth.make_weights(cfg, seed=66, bf16=True).items()}
    w["wpe"] = w["wpe"] + np.float32(100.0)
    for l in range(cfg.n_layer):
        for k in ("c_proj_w", "c_proj_b", "mlp_proj_w", "mlp_proj_b"):
            w[f"h{l}.{k}"] = w[f"h{l}.{k}"] * np.float32(2.0 ** -7)
    w["wpe"] = (synth.to_bf16_bits(w["wpe"]).astype(np.uint32) << 16).view(np.float32).reshape(w["wpe"].shape)
    w[f"h{cfg.n_layer - 1}.mlp_proj_b"] -= np.float32(100.0)
    toks = synth.rand_tokens(660, n, cfg.vocab_size)
    m = zgpt.GPT(cfg)
    m.load_weights(w)
    zg.zg_debug_prefill_route(route, 0)
    try:
        got = m.prefill([toks])[0].astype(np.float64)
    finally:
        zg.zg_debug_prefill_route(0, 0)
    m.close()
    ref = exact_logits(cfg, w, toks)
    assert np.linalg.norm(got - ref) <= 1e-2 * np.linalg.norm(ref)


def trained(cfg, seed, bf16, far):
    """Gains and rows that differ as a trained model's do: by factors of some e around the usual ones; a channel in a hundred has a gain `far` times the others' and
    weights that make up for it."""
    rng = np.random.default_rng(seed)
    E = cfg.n_embed
    w = {k: np.array(v, np.float32) for k, v in synth.make_weights(cfg, seed=seed, bf16=bf16).items()}
    for l in range(cfg.n_layer):
        p = f"h{l}."
        for q, behind, rows in (("ln_1", "c_attn", 3 * E), ("ln_2", "c_fc", 4 * E)):
            g = 0.4 * np.exp(rng.normal(0.0, 1.0, E))
            at = rng.permutation(E)[:max(1, E // 100)]
            g[at] *= far
            w[p + q + "_g"], w[p + q + "_b"] = g.astype(np.float32), rng.normal(0.0, 0.1, E).astype(np.float32)
            w[p + behind + "_w"] = w[p + behind + "_w"].reshape(rows, E)
            w[p + behind + "_w"][:, at] /= np.float32(far)
        for q, o, i in (("c_attn", 3 * E, E), ("c_fc", 4 * E, E), ("c_proj", E, E), ("mlp_proj", E, 4 * E)):
            m = w[p + q + "_w"].reshape(o, i) * np.exp(rng.normal(0.0, 0.7, o)).astype(np.float32)[:, None]
            if q == "c_attn":
                m[:2 * E] *= np.float32(0.5)  # (scores of an ordinary size)
            if bf16:
                m = (synth.to_bf16_bits(m).astype(np.uint32) << 16).view(np.float32).reshape(m.shape)
            w[p + q + "_w"], w[p + q + "_b"] = m, rng.normal(0.0, 0.2, o).astype(np.float32)
    return w


@pytest.mark.parametrize("far", [2.0 ** 5, 2.0 ** 8, 2.0 ** 10])
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("route", [1, 2, 3])
def test_gains_and_rows_that_differ_as_a_trained_models(zg, far, bf16, route):
    """The exponents' bounds stay so near to what such layers compute that two terms hold it.  The bound: exact planes of three terms are 1.7e-7 to 3.6e-7 off with these weights."""
    cfg = synth.CONFIGS["nano-char"]
    errs = []
    for seed in (67, 68, 69):
        w = trained(cfg, seed, bf16, far)
        toks = synth.rand_tokens(10 * seed, 100, cfg.vocab_size)
        m = zgpt.GPT(cfg, weights_f32=not bf16)
        m.load_weights(w)
        zg.zg_debug_prefill_route(route, 0)
        try:
            got = m.prefill([toks])[0].astype(np.float64)
        finally:
            zg.zg_debug_prefill_route(0, 0)
        m.close()
        ref = exact_logits(cfg, w, toks)
        errs.append(np.linalg.norm(got - ref) / np.linalg.norm(ref))
    assert max(errs) <= 4e-7, errs


@pytest.mark.parametrize("batch,n", [(1, 9), (2, 20), (1, 64)])
def test_short_prompts_of_small_models_have_the_last_bit_of_an_fp32_weight(zg, batch, n):
    """Outputs w - w of weights that two terms round up: nothing, where two planes leave the eighth that the 24th bit is worth."""
    cfg = synth.CONFIGS["nano-char"]
    E = cfg.n_embed
    w = {k: np.array(v, np.float32) for k, v in synth.make_weights(cfg, seed=70, bf16=False).items()}
    for l in range(cfg.n_layer):
        w[f"h{l}.ln_2_g"] = np.zeros(E, np.float32)
        w[f"h{l}.ln_2_b"] = np.ones(E, np.float32)
        m = np.zeros((4 * E, E), np.float32)
        m[np.arange(4 * E), np.arange(4 * E) % E] = np.float32(2.0 ** 20 * (1.0 + 4095 * 2.0 ** -23))
        w[f"h{l}.c_fc_w"], w[f"h{l}.c_fc_b"] = m, -m.max(1)
    m = zgpt.GPT(cfg, batch=batch, weights_f32=True)
    m.load_weights(w)
    toks = np.stack([synth.rand_tokens(700 + b, n, cfg.vocab_size) for b in range(batch)])
    for got, t in zip(m.prefill(toks).astype(np.float64), toks):
        ref = exact_logits(cfg, w, t)
        assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)
    m.close()
