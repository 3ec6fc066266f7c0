"""32-bit products through the ring of K steps (rows of fp32, three terms made beside the products): both tile forms forced onto small ragged
shapes (rows and columns around a tile's edge, columns that are a multiple of four alone, one K step and odd numbers of them, groups of experts
that are empty or one row long, gathered rows, a matrix per head, gated results).  Infinite weights leave what a plain fp32 sum leaves."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def run(cfg, w, toks, dtype="float32"):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=512, max_seqs=2)
    m.load_weights(w)
    s = m.open()
    got = m.step([(s, toks, list(range(len(toks))))])
    m.close()
    return got


@pytest.mark.parametrize("form", ["2", "3", ""])
@pytest.mark.parametrize("rows", [9, 33, 64, 65, 129, 257])
def test_forms(monkeypatch, form, rows):
    monkeypatch.setenv("ZGPT2_LM_STREAM", form) if form else monkeypatch.delenv("ZGPT2_LM_STREAM", raising=False)
    for width, ff, eff, rank, experts in ((128, 64, 60, 64, 7), (192, 324, 192, 128, 3), (256, 576, 68, 256, 21)):
        cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.moe_mlp(ff=eff, experts=experts, top=2)),
                         tl.latent_layer(heads=3, dim=64, vdim=64, rot_dim=8, kv_rank=rank, q_rank=rank, mlp=tl.dense_mlp(ff=ff)),
                         tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.moe_mlp(ff=eff, experts=experts, top=1))], vocab=203, width=width)
        w = tl.weights(cfg, seed=rows + width)
        toks = tl.tokens(170 + rows, rows, cfg["vocab"])
        tl.assert_close(run(cfg, w, toks), lm_oracle.Model(cfg, w).forward(toks)[0], "float32", (form, rows, width))
    # (rounded rows, columns that are a multiple of four: no router that could flip)
    cfg = tl.config([tl.latent_layer(heads=3, dim=16, vdim=64, rot_dim=8, kv_rank=68, q_rank=68, mlp=tl.dense_mlp(ff=ff)) for ff in (4, 324)], vocab=203, width=192)
    w = tl.weights(cfg, seed=rows)
    toks = tl.tokens(270 + rows, rows, cfg["vocab"])
    tl.assert_close(run(cfg, w, toks, "bfloat16"), lm_oracle.Model(cfg, w).forward(toks)[0], "bfloat16", (form, rows))


@pytest.mark.parametrize("form", ["2", "3"])
def test_infinite_weights(monkeypatch, form):
    """Squared ReLU of minus infinity is zero and of infinity infinite: which rows stay finite tells the sums apart from NaN."""
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.dense_mlp(ff=320)) for _ in range(2)], vocab=203, width=128)
    w = tl.weights(cfg, seed=3)
    name = "l1.mlp.up"
    w[name] = w[name].copy()
    w[name][17, 5] = -np.inf
    toks = tl.tokens(6, 90, cfg["vocab"])
    monkeypatch.setenv("ZGPT2_LM_STREAM", "-1")
    ref = run(cfg, w, toks)
    monkeypatch.setenv("ZGPT2_LM_STREAM", form)
    got = run(cfg, w, toks)
    ok = np.isfinite(ref).all(axis=1)
    assert ok.any() and not ok.all() and (np.isfinite(got).all(axis=1) == ok).all()
    tl.assert_close(got[ok], ref[ok], "float32", form)


@pytest.mark.parametrize("rows", [40, 300, 505])
def test_toy_products_stay_on_the_fp32_instruction(monkeypatch, rows):
    """Products of fewer than 128 columns, the experts' gated ones among them: the same bits with the ring and without it, at any number of rows."""
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=32, mlp=tl.moe_mlp(ff=64, experts=6, top=4)) for _ in range(2)], vocab=203, width=64)
    w = tl.weights(cfg, seed=rows)
    toks = tl.tokens(370 + rows, rows, cfg["vocab"])
    monkeypatch.delenv("ZGPT2_LM_STREAM", raising=False)
    got = run(cfg, w, toks)
    monkeypatch.setenv("ZGPT2_LM_STREAM", "-1")
    assert np.array_equal(got, run(cfg, w, toks))
    tl.assert_close(got, lm_oracle.Model(cfg, w).forward(toks)[0], "float32", rows)
