"""Steps of three to eight rows on the matrix cores: rows beyond 1024 columns on sixteen waves (remainders of a turn and of a wave's share, the longest
that fit and beyond them), the vocabulary's rows in turn (a ragged last tile, rows of one to four turns a wave), lists with as many assignments as
experts and more (several groups of eight on one expert) and with fewer."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def check(cfg, w, n, steps=2):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=512, max_seqs=8)
    m.load_weights(w)
    toks = [tl.tokens(60 + b, 3 + b + steps, cfg["vocab"]) for b in range(n)]
    refs = [lm_oracle.Model(cfg, w).forward(t)[0] for t in toks]
    seqs = [m.open() for _ in toks]
    m.step([(s, t[:len(t) - steps], []) for s, t in zip(seqs, toks)])
    for i in range(steps):
        at = [len(t) - steps + i for t in toks]
        got = m.step([(s, [t[k]], [0]) for s, t, k in zip(seqs, toks, at)])
        tl.assert_close(got, np.stack([r[k] for r, k in zip(refs, at)]), "float32", (n, i))
    m.close()


@pytest.mark.parametrize("n", [6, 8])
@pytest.mark.parametrize("ff", [1032, 1088, 2040, 2056, 3072, 4096, 4104])
def test_long_rows(ff, n):
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=16, vdim=16, mlp=tl.dense_mlp(ff=ff))], vocab=203, width=72)
    check(cfg, tl.weights(cfg, seed=ff), n)


@pytest.mark.parametrize("n", [3, 8])
@pytest.mark.parametrize("width,vocab", [(64, 16384), (72, 16401), (264, 20005), (520, 17003), (776, 16390), (1024, 33000)])
def test_many_rows(width, vocab, n):
    cfg = tl.config([tl.hgrn2_layer(heads=1, dim=16, vdim=16, mlp=tl.dense_mlp(ff=32))], vocab=vocab, width=width)
    check(cfg, tl.weights(cfg, seed=width), n, steps=1)


@pytest.mark.parametrize("n", [8, 5])
@pytest.mark.parametrize("experts,top,ff,width", [(1, 1, 40, 64), (2, 2, 72, 264), (16, 2, 64, 72), (5, 4, 264, 520), (3, 3, 136, 64), (24, 2, 64, 64)])
def test_lists(experts, top, ff, width, n):
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=16, vdim=16, mlp=tl.moe_mlp(ff=ff, experts=experts, top=top))], vocab=203, width=width)
    check(cfg, tl.weights(cfg, seed=experts + ff), n)
