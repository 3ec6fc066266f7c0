"""The tiled products of the layered-model tier on sizes where they can go wrong: every tile form forced onto small ragged shapes
(rows around a tile's edge, K with a remainder behind the last K step, groups of experts that are empty or one row long)."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("form", ["128", "64", "32", ""])
@pytest.mark.parametrize("rows", [9, 33, 64, 129, 200])
def test_tile_forms(monkeypatch, form, rows, dtype):
    monkeypatch.setenv("ZGPT2_LM_GEMM_TILE", form) if form else monkeypatch.delenv("ZGPT2_LM_GEMM_TILE", raising=False)
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=68, mlp=tl.moe_mlp(ff=152, experts=7, top=2)),
                     tl.latent_layer(heads=2, dim=16, vdim=16, rot_dim=8, kv_rank=136, q_rank=40, mlp=tl.dense_mlp(ff=328))], vocab=203, width=136)
    w = tl.weights(cfg, seed=rows)
    toks = tl.tokens(70 + rows, rows, cfg["vocab"])
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=512, max_seqs=2)
    m.load_weights(w)
    s = m.open()
    got = m.step([(s, toks, list(range(rows)))])
    m.close()
    tl.assert_close(got, lm_oracle.Model(cfg, w).forward(toks)[0], dtype, (form, rows, dtype))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_values_that_are_not_finite(dtype, bad):
    """An activation that is not finite: the rows that see it are not finite, the others are what they are without it."""
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.dense_mlp(ff=328))], vocab=203, width=136)
    w = tl.weights(cfg, seed=3)
    toks = tl.tokens(5, 40, cfg["vocab"])
    toks[toks == 7] = 8
    ref = lm_oracle.Model(cfg, w).forward(toks)[0]
    toks[25] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = bad
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=512, max_seqs=2)
    m.load_weights(w)
    s = m.open()
    got = m.step([(s, toks, list(range(40)))])
    m.close()
    assert np.isnan(got[25:]).any(axis=1).all()
    tl.assert_close(got[:25], ref[:25], dtype, (bad, dtype))


@pytest.mark.parametrize("kv_rank,rot_dim", [(40, 6), (64, 32), (100, 20), (256, 32), (300, 12), (320, 64)])
def test_latent_tiles(kv_rank, rot_dim):
    """Latent attention of portions with every tile size (rows of no whole number of pieces among them): three sequences whose portions
    end around block and tile edges, behind histories of other lengths; five heads (the last group of four is one)."""
    cfg = tl.config([tl.latent_layer(heads=5, dim=16, vdim=16, rot_dim=rot_dim, rot_dims=rot_dim, kv_rank=kv_rank, q_rank=40, mlp=tl.dense_mlp(ff=96))],
                    vocab=203, width=64)
    w = tl.weights(cfg, seed=kv_rank)
    oracle = lm_oracle.Model(cfg, w)
    toks = [tl.tokens(80 + b, n, cfg["vocab"]) for b, n in enumerate((150, 97, 66))]
    refs = [oracle.forward(t)[0] for t in toks]
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="bfloat16", max_tokens=512, max_seqs=3)
    m.load_weights(w)
    seqs = [m.open() for _ in toks]
    cuts = [(33, 64, 150), (1, 96, 97), (31, 33, 66)]
    lo = [0, 0, 0]
    for step in range(3):
        hi = [c[step] for c in cuts]
        got = m.step([(s, t[a:b], list(range(b - a))) for s, t, a, b in zip(seqs, toks, lo, hi)])
        want = np.concatenate([r[a:b] for r, a, b in zip(refs, lo, hi)])
        tl.assert_close(got, want, "bfloat16", (kv_rank, step))
        lo = hi
    m.close()
