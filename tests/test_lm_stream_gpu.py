"""Products of rounded rows through the ring of K steps: every tile form forced onto small ragged shapes (rows and columns around a tile's edge, one
K step to fewer and more than the ring holds, groups of experts that are empty or one row long, gathered rows, a matrix per head), results
as fp32 rows, rounded rows, squared and gated ones."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def run(cfg, w, toks):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="bfloat16", max_tokens=512, max_seqs=2)
    m.load_weights(w)
    s = m.open()
    got = m.step([(s, toks, list(range(len(toks))))])
    m.close()
    return got


@pytest.mark.parametrize("form", ["1", "2", "3", "4", ""])
@pytest.mark.parametrize("rows", [9, 33, 64, 65, 127, 129, 200, 257])
def test_forms(monkeypatch, form, rows):
    monkeypatch.setenv("ZGPT2_LM_STREAM", form) if form else monkeypatch.delenv("ZGPT2_LM_STREAM", raising=False)
    for width, ff, eff, rank, experts in ((64, 64, 64, 64, 7), (192, 320, 192, 128, 3), (128, 576, 72, 256, 21)):
        cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.moe_mlp(ff=eff, experts=experts, top=2)),
                         tl.latent_layer(heads=3, dim=16, vdim=64, rot_dim=8, kv_rank=rank, q_rank=rank, mlp=tl.dense_mlp(ff=ff)),
                         tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.moe_mlp(ff=eff, experts=experts, top=1))], vocab=203, width=width)
        w = tl.weights(cfg, seed=rows + width)
        toks = tl.tokens(70 + rows, rows, cfg["vocab"])
        tl.assert_close(run(cfg, w, toks), lm_oracle.Model(cfg, w).forward(toks)[0], "bfloat16", (form, rows, width))


@pytest.mark.parametrize("form", ["1", "2", "3"])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_values_that_are_not_finite(monkeypatch, form, bad):
    """A row that is not finite reaches no row in front of it (tiles repeat rows behind their edge)."""
    monkeypatch.setenv("ZGPT2_LM_STREAM", form)
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.dense_mlp(ff=320)),
                     tl.hgrn2_layer(heads=2, dim=24, vdim=64, mlp=tl.moe_mlp(ff=64, experts=3, top=1))], vocab=203, width=128)
    w = tl.weights(cfg, seed=3)
    toks = tl.tokens(5, 90, cfg["vocab"])
    toks[toks == 7] = 8
    ref = lm_oracle.Model(cfg, w).forward(toks)[0]
    toks[75] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = bad
    got = run(cfg, w, toks)
    assert np.isnan(got[75:]).any(axis=1).all()
    tl.assert_close(got[:75], ref[:75], "bfloat16", (form, bad))
