"""The choice of experts behind the norm in front of it (portions): numbers of experts up to and beyond what a wave keeps, widths at the edges of its pieces,
rows around a workgroup's, every number of choices, scores that tie and that are not numbers; bounds of the tier."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def run(cfg, w, toks, dtype):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=1024, max_seqs=2)
    m.load_weights(w)
    s = m.open()
    got = m.step([(s, toks, list(range(len(toks))))])
    m.close()
    return got


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("experts,top,width,rows", [(1, 1, 64, 9), (2, 2, 136, 65), (3, 1, 256, 64), (5, 3, 260, 100), (7, 2, 512, 33), (8, 2, 768, 130), (8, 8, 1024, 66), (6, 2, 1020, 20),
                                                   (9, 2, 64, 70), (16, 4, 128, 40)])
def test_experts(dtype, experts, top, width, rows):
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=16, vdim=16, mlp=tl.moe_mlp(ff=24, experts=experts, top=top))], vocab=101, width=width)
    w = tl.weights(cfg, seed=experts)
    toks = tl.tokens(rows, rows, cfg["vocab"])
    tl.assert_close(run(cfg, w, toks, dtype), lm_oracle.Model(cfg, w).forward(toks)[0], dtype, (experts, top, width, rows))


def test_ties_and_nan():
    """Equal scores: the experts of the lowest numbers; scores that are not numbers stay in range and in their rows."""
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=16, vdim=16, mlp=tl.moe_mlp(ff=24, experts=8, top=3))], vocab=101, width=64)
    w = tl.weights(cfg, seed=1)
    w["l0.mlp.router"] = np.zeros_like(w["l0.mlp.router"])
    w["l0.mlp.correction"] = np.zeros_like(w["l0.mlp.correction"])
    toks = tl.tokens(2, 40, cfg["vocab"])
    toks[toks == 7] = 8
    ref = lm_oracle.Model(cfg, w).forward(toks)[0]
    tl.assert_close(run(cfg, w, toks, "float32"), ref, "float32")
    toks[30] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = np.nan
    got = run(cfg, w, toks, "float32")
    tl.assert_close(got[:30], ref[:30], "float32")
    assert np.isnan(got[30]).any()
