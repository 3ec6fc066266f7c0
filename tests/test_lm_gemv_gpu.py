"""Products of decode steps of one and two sequences whose operands come in whole 16-byte pieces: rows of one, two and three pieces per
lane and their remainders, long rows split over the waves, activations on load, and the norms inside the product that reads them (an
odd and an even number of them in a step, and rows too long for it)."""
import numpy as np
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def check(cfg, w, refs, toks, n, dtype):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=256, max_seqs=2)
    m.load_weights(w)
    seqs = [m.open() for _ in range(n)]
    for i in range(len(toks[0])):
        got = m.step([(s, [t[i]], [0]) for s, t in zip(seqs, toks)])
        # (nothing is rounded in a step of few rows: the same sums in both modes)
        tl.assert_close(got, np.stack([r[i] for r in refs[:n]]), dtype, (n, i))
    m.close()


@pytest.mark.parametrize("width,ff", [(40, 1536), (512, 1544), (520, 2056), (1024, 4104), (1032, 520)])
@pytest.mark.parametrize("mlps", [(1, 1), (1, 0), (0, 1)])
def test_norms_inside_products(width, ff, mlps):
    cfg = dl.config([dl.mamba_layer(mlp=dl.dense(ff=ff) if mlps[0] else None), dl.attn_layer(mlp=None),
                     dl.latent_layer(kv_rank=24, dim=8, vdim=16, rot_dim=8, mlp=dl.dense(ff=ff) if mlps[1] else None)], width=width)
    w = dl.weights(cfg, seed=width)
    toks = [dl.tokens(3 + b, 6, cfg["vocab"]) for b in range(2)]
    refs = [do.forward(w, cfg, t) for t in toks]
    for n in (1, 2):
        check(cfg, w, refs, toks, n, "float32")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("ff", [24, 512, 520, 1032, 1528, 1544, 6160])
def test_activations_on_load(ff, dtype):
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=24, vdim=68, mlp=tl.moe_mlp(ff=ff, experts=5, top=2)),
                     tl.latent_layer(heads=2, dim=16, vdim=16, rot_dim=8, kv_rank=136, q_rank=40, mlp=tl.dense_mlp(ff=ff))], vocab=203, width=136)
    w = tl.weights(cfg, seed=ff)
    oracle = lm_oracle.Model(cfg, w)
    toks = [tl.tokens(20 + b, 5, cfg["vocab"]) for b in range(2)]
    refs = [oracle.forward(t)[0] for t in toks]
    for n in (1, 2):
        check(cfg, w, refs, toks, n, dtype)


@pytest.mark.parametrize("dim,vdim", [(1, 4), (16, 24), (100, 36), (128, 64), (129, 68), (160, 128), (256, 132), (24, 256), (40, 6), (40, 260)])
def test_one_token_of_the_recurrence(dim, vdim):
    """A token of every entry: states of fewer and more rows than the threads hold at a time, value widths around a row of lanes and beyond
    the kernel's."""
    cfg = tl.config([tl.hgrn2_layer(heads=3, dim=dim, vdim=vdim, mlp=tl.dense_mlp(ff=24))], vocab=97, width=48)
    w = tl.weights(cfg, seed=dim + vdim)
    oracle = lm_oracle.Model(cfg, w)
    toks = [tl.tokens(70 + b, 9, cfg["vocab"]) for b in range(2)]
    refs = [oracle.forward(t)[0] for t in toks]
    for n in (1, 2):
        check(cfg, w, refs, toks, n, "float32")


@pytest.mark.parametrize("width", [8, 136, 520, 1024, 1032, 44])
@pytest.mark.parametrize("experts,top", [(3, 2), (8, 2), (21, 5)])
def test_router_with_the_norms_in_front(width, experts, top):
    """Steps of few rows: the sum and norms inside the router's launch; fewer experts than waves, more, widths it leaves to two launches."""
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=16, vdim=24, mlp=tl.moe_mlp(ff=24, experts=experts, top=top)),
                     tl.hgrn2_layer(heads=2, dim=16, vdim=24, mlp=tl.moe_mlp(ff=24, experts=experts, top=top))], vocab=97, width=width)
    w = tl.weights(cfg, seed=width + experts)
    oracle = lm_oracle.Model(cfg, w)
    toks = [tl.tokens(90 + b, 5, cfg["vocab"]) for b in range(2)]
    refs = [oracle.forward(t)[0] for t in toks]
    for n in (1, 2):
        check(cfg, w, refs, toks, n, "float32")


@pytest.mark.parametrize("width,ff", [(136, 2047), (136, 2049), (520, 2051), (1032, 2054), (511, 1536), (513, 1536), (515, 1544), (518, 2056)])
def test_four_rows_a_wave(width, ff):
    """The products of the norms (ff rows) and of the polynomial (width rows) on either side of where four weight rows share what a row
    needs in front of them, with one to three left over."""
    cfg = dl.config([dl.mamba_layer(mlp=dl.dense(ff=ff)), dl.attn_layer(mlp=dl.dense(ff=ff))], width=width)
    w = dl.weights(cfg, seed=width + ff)
    toks = [dl.tokens(7 + b, 5, cfg["vocab"]) for b in range(2)]
    refs = [do.forward(w, cfg, t) for t in toks]
    for n in (1, 2):
        check(cfg, w, refs, toks, n, "float32")
