"""The norm behind the gated recurrence's heads in the epilogue of its chunk kernel: heads of every width class (whole and partial waves of 32 channels,
no whole pieces of eight, wider than a workgroup, where the norm keeps its launch), chunks with a remainder, several entries; bounds of the tier."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("dim,vdim,heads", [(128, 128, 2), (64, 128, 1), (32, 96, 3), (16, 68, 2), (64, 8, 3), (24, 40, 2), (128, 32, 1), (20, 136, 2), (16, 4, 2)])
def test_heads(dtype, dim, vdim, heads):
    cfg = tl.config([tl.hgrn2_layer(heads=heads, dim=dim, vdim=vdim, mlp=tl.dense_mlp(ff=64))], vocab=101, width=64)
    w = tl.weights(cfg, seed=dim + vdim)
    toks = [tl.tokens(40 + b, n, cfg["vocab"]) for b, n in enumerate((130, 64, 33, 190))]
    refs = [lm_oracle.Model(cfg, w).forward(t)[0] for t in toks]
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=1024, max_seqs=4)
    m.load_weights(w)
    seqs, lo = [m.open() for _ in toks], [0] * 4
    for hi in ([65, 1, 33, 40], [130, 64, 33, 190]):
        entries = [(s, t[a:b], list(range(b - a))) for s, t, a, b in zip(seqs, toks, lo, hi) if b > a]
        tl.assert_close(m.step(entries), np.concatenate([r[a:b] for r, a, b in zip(refs, lo, hi)]), dtype, (dim, vdim, hi))
        lo = hi
    m.close()
