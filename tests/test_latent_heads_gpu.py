"""Latent attention of portions over keys and values of the heads' own, in bf16 mode, where it can go wrong: rows around the edges of its blocks of 32 and
128 queries and tiles of 32 keys, behind histories, entries beyond the first 64, pages that are no whole tiles, heads that leave half a
workgroup, both rotations, the gate, the sink, latents of another layer, values that are not finite.  The oracles compute in fp64; the bounds are the
tier's for bf16 mode (lm_testlib)."""
import numpy as np
import pytest

import duvulix_oracle
import duvulix_testlib as dl
import lm_oracle
import lm_testlib as tl
import pemuvik_oracle
import pemuvik_testlib as pl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu
DIMS = dict(dim=64, vdim=64, rot_dim=32)


@pytest.fixture(params=["1", "4"])
def form(request, monkeypatch):
    monkeypatch.setenv("ZGPT2_LM_LATENT_HEADS", request.param)
    return request.param


def model(cfg, w, **kw):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), **{"dtype": "bfloat16", "max_tokens": 1024, "max_seqs": 4, **kw})
    m.load_weights(w)
    return m


def steps(m, toks, cuts):
    """Portions up to the positions of cuts, a row of them after the other: the logits of every step."""
    seqs, lo, out = [m.open() for _ in toks], [0] * len(toks), []
    for hi in cuts:
        out.append(m.step([(s, t[a:b], list(range(b - a))) for s, t, a, b in zip(seqs, toks, lo, hi)]))
        lo = hi
    for s in seqs:
        m.close_seq(s)
    return out


def of(refs, cuts):
    return [np.concatenate([r[a:b] for r, a, b in zip(refs, lo, hi)]) for lo, hi in zip([[0] * len(refs)] + cuts[:-1], cuts)]


@pytest.mark.parametrize("rank,heads", [(256, 3), (256, 2), (128, 5), (256, 1)])
def test_rows(form, monkeypatch, rank, heads):
    cfg = tl.config([tl.latent_layer(heads=heads, kv_rank=rank, q_rank=40, mlp=tl.dense_mlp(ff=96), **DIMS)], vocab=203, width=64)
    w = tl.weights(cfg, seed=rank)
    for rows in (9, 31, 32, 33, 127, 128, 129, 300):
        toks = [tl.tokens(rows, rows, cfg["vocab"])]
        ref = lm_oracle.Model(cfg, w).forward(toks[0])[0]
        m = model(cfg, w)
        got = steps(m, toks, [[rows]])[0]
        monkeypatch.setenv("ZGPT2_LM_LATENT_HEADS", "-1")
        other = steps(m, toks, [[rows]])[0]
        monkeypatch.setenv("ZGPT2_LM_LATENT_HEADS", form)
        m.close()
        tl.assert_close(got, ref, "bfloat16", (rank, heads, rows))
        assert not np.array_equal(got, other)  # (another order of roundings: it was this path that ran)


@pytest.mark.parametrize("page_tokens", [0, 48, 8])
def test_histories(form, page_tokens):
    cfg = tl.config([tl.latent_layer(heads=5, kv_rank=256, q_rank=40, mlp=tl.dense_mlp(ff=96), **DIMS)], vocab=203, width=64)
    w = tl.weights(cfg, seed=7)
    toks = [tl.tokens(80 + b, n, cfg["vocab"]) for b, n in enumerate((300, 97, 66))]
    refs = [lm_oracle.Model(cfg, w).forward(t)[0] for t in toks]
    cuts = [[33, 64, 31], [34, 95, 40], [163, 96, 65], [300, 97, 66]]
    m = model(cfg, w, page_tokens=page_tokens)
    for got, want in zip(steps(m, toks, cuts), of(refs, cuts)):
        tl.assert_close(got, want, "bfloat16", page_tokens)
    m.close()


def test_many_entries(form):
    cfg = tl.config([tl.latent_layer(heads=2, kv_rank=256, q_rank=40, mlp=tl.dense_mlp(ff=96), **DIMS)], vocab=203, width=64)
    w = tl.weights(cfg, seed=8)
    toks = [tl.tokens(b, 3 + b % 40, cfg["vocab"]) for b in range(70)]
    refs = [lm_oracle.Model(cfg, w).forward(t)[0] for t in toks]
    cuts = [[2] * 70, [len(t) for t in toks]]
    m = model(cfg, w, max_tokens=70 * 64, max_seqs=70, max_step_tokens=2048)
    for got, want in zip(steps(m, toks, cuts), of(refs, cuts)):
        tl.assert_close(got, want, "bfloat16")
    m.close()


def test_gate_and_other_layers_latents(form):
    cfg = dl.config([dl.latent_layer(heads=4, kv_rank=256, mlp=dl.dense(ff=64), **DIMS), dl.latent_layer(heads=3, kv_rank=256, kv_from=0, mlp=dl.dense(ff=64), **DIMS)],
                    vocab=203, width=64)
    w = dl.weights(cfg, seed=4)
    toks = [dl.tokens(90 + b, n, cfg["vocab"]) for b, n in enumerate((150, 97))]
    refs = [duvulix_oracle.forward(w, cfg, t) for t in toks]
    cuts = [[130, 33], [150, 97]]
    m = model(cfg, w)
    for got, want in zip(steps(m, toks, cuts), of(refs, cuts)):
        tl.assert_close(got, want, "bfloat16")
    m.close()


def test_sink(form):
    cfg = pl.config([pl.latent_layer(heads=4, kv_rank=256, mlp=pl.dense(ff=64), **DIMS)], vocab=203, width=64)
    w = pl.weights(cfg, seed=4)
    toks = [pl.tokens(90 + b, n, cfg["vocab"]) for b, n in enumerate((150, 97))]
    refs = [pemuvik_oracle.forward(w, cfg, t) for t in toks]
    cuts = [[130, 33], [150, 97]]
    m = model(cfg, w)
    for got, want in zip(steps(m, toks, cuts), of(refs, cuts)):
        tl.assert_close(got, want, "bfloat16")
    m.close()


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_values_that_are_not_finite(form, bad):
    """Rows in front of a token that is not finite, in its own tile too, are what they are without it; the others are not finite."""
    cfg = tl.config([tl.latent_layer(heads=3, kv_rank=256, q_rank=40, mlp=tl.dense_mlp(ff=96), **DIMS)], vocab=203, width=64)
    w = tl.weights(cfg, seed=3)
    toks = tl.tokens(5, 140, cfg["vocab"])
    toks[toks == 7] = 8
    ref = lm_oracle.Model(cfg, w).forward(toks)[0]
    toks[75] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = bad
    m = model(cfg, w)
    got = steps(m, [toks], [[140]])[0]
    m.close()
    tl.assert_close(got[:75], ref[:75], "bfloat16", bad)
    assert np.isnan(got[75:]).any(axis=1).all()


@pytest.mark.parametrize("rank,heads", [(256, 3), (128, 2), (256, 1)])
def test_32_bit(monkeypatch, rank, heads):
    """32-bit mode: rows around blocks and tiles, portions behind histories on pages that are no whole tiles."""
    cfg = tl.config([tl.latent_layer(heads=heads, kv_rank=rank, q_rank=40, mlp=tl.dense_mlp(ff=96), **DIMS)], vocab=203, width=64)
    w = tl.weights(cfg, seed=rank)
    m = model(cfg, w, dtype="float32", page_tokens=24)
    for rows in (9, 31, 32, 33, 128, 129, 300):
        toks = [tl.tokens(rows, rows, cfg["vocab"])]
        got = steps(m, toks, [[rows]])[0]
        monkeypatch.setenv("ZGPT2_LM_LATENT_HEADS", "-1")
        other = steps(m, toks, [[rows]])[0]
        monkeypatch.delenv("ZGPT2_LM_LATENT_HEADS")
        tl.assert_close(got, lm_oracle.Model(cfg, w).forward(toks[0])[0], "float32", (rank, heads, rows))
        assert not np.array_equal(got, other)  # (another order of sums: it was this path that ran)
    toks = [tl.tokens(80 + b, n, cfg["vocab"]) for b, n in enumerate((300, 97, 66))]
    refs = [lm_oracle.Model(cfg, w).forward(t)[0] for t in toks]
    cuts = [[33, 64, 31], [34, 95, 40], [163, 96, 65], [300, 97, 66]]
    for got, want in zip(steps(m, toks, cuts), of(refs, cuts)):
        tl.assert_close(got, want, "float32", cuts)
    m.close()


@pytest.mark.parametrize("design", ["gate", "sink"])
def test_32_bit_other_designs(design):
    if design == "gate":
        lib, oracle = dl, duvulix_oracle
        layers = [dl.latent_layer(heads=4, kv_rank=256, mlp=dl.dense(ff=64), **DIMS), dl.latent_layer(heads=3, kv_rank=256, kv_from=0, mlp=dl.dense(ff=64), **DIMS)]
    else:
        lib, oracle = pl, pemuvik_oracle
        layers = [pl.latent_layer(heads=4, kv_rank=256, mlp=pl.dense(ff=64), **DIMS)]
    cfg = lib.config(layers, vocab=203, width=64)
    w = lib.weights(cfg, seed=4)
    toks = [lib.tokens(90 + b, n, cfg["vocab"]) for b, n in enumerate((150, 97))]
    cuts = [[130, 33], [150, 97]]
    m = model(cfg, w, dtype="float32")
    for got, want in zip(steps(m, toks, cuts), of([oracle.forward(w, cfg, t) for t in toks], cuts)):
        tl.assert_close(got, want, "float32")
    m.close()


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_32_bit_values_that_are_not_finite(bad):
    cfg = tl.config([tl.latent_layer(heads=3, kv_rank=256, q_rank=40, mlp=tl.dense_mlp(ff=96), **DIMS)], vocab=203, width=64)
    w = tl.weights(cfg, seed=3)
    toks = tl.tokens(5, 140, cfg["vocab"])
    toks[toks == 7] = 8
    ref = lm_oracle.Model(cfg, w).forward(toks)[0]
    toks[75] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = bad
    m = model(cfg, w, dtype="float32")
    got = steps(m, [toks], [[140]])[0]
    m.close()
    tl.assert_close(got[:75], ref[:75], "float32", bad)
    assert np.isnan(got[75:]).any(axis=1).all()
