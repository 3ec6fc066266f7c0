"""Rows of the residual stream between two sublayers: runs of rows that end inside, at and behind an entry's edge, widths with a remainder
behind the last 16-byte piece of a lane and widths in no whole pieces, one to four pieces a lane; decode steps of more rows than the
row-vector products take."""
import numpy as np
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def designs(width, dtype):
    def moe(**kw):  # in bf16 mode a rounded activation flips close calls of a router, one row in eight here: experts without a choice there
        return tl.moe_mlp(**{**kw, "experts": kw["top"]}) if dtype == "bfloat16" else tl.moe_mlp(**kw)

    tok = tl.config([tl.hgrn2_layer(heads=2, dim=16, vdim=24, mlp=moe(ff=24, experts=5, top=3)), tl.hgrn2_layer(heads=2, dim=8, vdim=8, mlp=tl.dense_mlp(ff=40)),
                     tl.latent_layer(heads=2, dim=16, vdim=16, rot_dim=8, kv_rank=32, q_rank=40, mlp=moe(ff=16, experts=4, top=2)),
                     tl.hgrn2_layer(heads=1, dim=16, vdim=24, mlp=moe(ff=24, experts=5, top=2))], vocab=203, width=width)
    duv = dl.config([dl.mamba_layer(mlp=dl.dense()), dl.attn_layer(mlp=None), dl.latent_layer(kv_rank=24, dim=8, vdim=16, rot_dim=8, mlp=dl.dense(ff=40))], width=width)
    return ((tok, tl.weights(tok, seed=width), lambda c, w, t: lm_oracle.Model(c, w).forward(t)[0], tl.tokens),
            (duv, dl.weights(duv, seed=width), lambda c, w, t: do.forward(w, c, t), dl.tokens))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("run", ["1", "3", "8"])  # (width 4: a norm of four values amplifies fp32 rounding to 2.6e-4 in any kernel)
@pytest.mark.parametrize("width", [8, 44, 50, 260, 520, 776, 1032])
def test_portions(monkeypatch, width, run, dtype):
    monkeypatch.setenv("ZGPT2_LM_NORM_RUN", run)
    for cfg, w, forward, tokens in designs(width, dtype):
        toks = [tokens(b, n, cfg["vocab"]) for b, n in enumerate((40, 27, 17))]
        refs = [forward(cfg, w, t) for t in toks]
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=256, max_seqs=3)
        m.load_weights(w)
        seqs = [m.open() for _ in toks]
        lo = [0, 0, 0]
        for hi in ((16, 1, 9), (17, 26, 10), (40, 27, 17)):
            got = m.step([(s, t[a:b], list(range(b - a))) for s, t, a, b in zip(seqs, toks, lo, hi)])
            tl.assert_close(got, np.concatenate([r[a:b] for r, a, b in zip(refs, lo, hi)]), dtype, (cfg["architecture"], width, run, hi))
            lo = hi
        m.close()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("rows", [9, 17])
@pytest.mark.parametrize("width", [48, 50])
def test_decode_steps_of_many_rows(width, rows, dtype):
    for cfg, w, forward, tokens in designs(width, dtype):
        toks = [tokens(50 + b, 5, cfg["vocab"]) for b in range(rows)]
        refs = [forward(cfg, w, t) for t in toks]
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=256, max_seqs=rows)
        m.load_weights(w)
        seqs = [m.open() for _ in toks]
        for i in range(5):
            got = m.step([(s, [t[i]], [0]) for s, t in zip(seqs, toks)])
            tl.assert_close(got, np.stack([r[i] for r in refs]), dtype, (cfg["architecture"], width, rows, i))
        m.close()
