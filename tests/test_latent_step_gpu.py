"""Latent attention of decode steps in two launches (queries carried into the latent space by the attention's workgroups, key ranges merged
where the values are made): one and two ranges and all sixteen, edges of a range, the row's own token alone in its range; latents and rotary parts
at the kernels' edges and beyond them; layers that read another layer's latents; queries through a norm of their own; gates and sinks."""
import numpy as np
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
import lm_oracle
import lm_testlib as tl
import pemuvik_oracle as po
import pemuvik_testlib as pl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu

STARTS = [290, 15, 0, 256, 16, 255, 31, 1]  # tokens in front of the first step


def check(cfg, w, forward, n, dtype="float32", steps=3):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=1536, max_seqs=8)
    m.load_weights(w)
    starts = STARTS[:n]
    toks = [tl.tokens(40 + b, s + steps, cfg["vocab"]) for b, s in enumerate(starts)]
    refs = [forward(t) for t in toks]
    seqs = [m.open() for _ in starts]
    begun = [(s, t[:k], []) for s, t, k in zip(seqs, toks, starts) if k > 0]
    if begun:
        m.step(begun)
    for i in range(steps):
        got = m.step([(s, [t[k + i]], [0]) for s, t, k in zip(seqs, toks, starts)])
        tl.assert_close(got, np.stack([r[k + i] for r, k in zip(refs, starts)]), dtype, (n, i))
    m.close()


@pytest.mark.parametrize("n", [1, 2, 3, 8])
@pytest.mark.parametrize("dim,kv_rank,rot_dim,vdim", [(64, 256, 32, 64), (64, 8, 64, 5), (128, 320, 64, 132), (64, 512, 4, 8), (128, 64, 8, 17), (64, 136, 12, 33), (64, 520, 8, 8),
                                                      (72, 64, 8, 16)])
def test_projected_queries(dim, kv_rank, rot_dim, vdim, n):
    lat = dict(heads=3, dim=dim, vdim=vdim, rot_dim=rot_dim, kv_rank=kv_rank)
    cfg = dl.config([dl.latent_layer(mlp=dl.dense(ff=32), **lat), dl.latent_layer(kv_from=0, mlp=dl.dense(ff=32), **lat)], width=48)
    w = dl.weights(cfg, seed=dim + kv_rank)
    check(cfg, w, lambda t: do.forward(w, cfg, t), n)


@pytest.mark.parametrize("n", [1, 2, 3, 8])
@pytest.mark.parametrize("q_rank,rot_dims,kv_rank", [(384, 32, 256), (8, 16, 64), (1032, 0, 128), (1544, 32, 72), (40, 32, 40), (44, 32, 64)])
def test_queries_through_a_norm(q_rank, rot_dims, kv_rank, n):
    cfg = tl.config([tl.latent_layer(heads=2, dim=64, vdim=24, rot_dim=32, rot_dims=rot_dims, kv_rank=kv_rank, q_rank=q_rank, mlp=tl.dense_mlp(ff=32))], width=48)
    w = tl.weights(cfg, seed=q_rank)
    oracle = lm_oracle.Model(cfg, w)
    check(cfg, w, lambda t: oracle.forward(t)[0], n)


@pytest.mark.parametrize("n", [1, 8])
def test_looped_layers_file_their_own_latents(n):
    cfg = tl.config([tl.latent_layer(heads=2, dim=64, vdim=64, rot_dim=32, kv_rank=64, q_rank=64, mlp=tl.dense_mlp(ff=32)) for _ in range(2)], width=48,
                    loop={"start": 0, "stop": 2, "times": 2})
    w = tl.weights(cfg, seed=5)
    oracle = lm_oracle.Model(cfg, w)
    check(cfg, w, lambda t: oracle.forward(t)[0], n)


@pytest.mark.parametrize("n", [1, 2, 3, 8])
def test_sinks(n):
    cfg = pl.config([pl.latent_layer(heads=3, dim=64, vdim=20, rot_dim=16, kv_rank=72, mlp=pl.dense(ff=32)) for _ in range(2)], width=48)
    w = pl.weights(cfg, seed=9)
    check(cfg, w, lambda t: po.forward(w, cfg, t), n)


@pytest.mark.parametrize("page_tokens", [1, 3, 16, 0])
@pytest.mark.parametrize("dim,kv_rank,rot_dim", [(64, 64, 64), (64, 72, 8), (128, 512, 64)])
def test_long_ranges(dim, kv_rank, rot_dim, page_tokens):
    """Ranges of several turns of sixteen keys, whose pages are asked for a turn ahead: around whole turns, pages of one token to many."""
    lat = dict(heads=2, dim=dim, vdim=8, rot_dim=rot_dim, kv_rank=kv_rank)
    cfg = dl.config([dl.latent_layer(mlp=None, **lat)], width=32)
    w = dl.weights(cfg, seed=kv_rank)
    starts = [1279, 1023, 767, 800]
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=4224, max_seqs=4, page_tokens=page_tokens, max_step_tokens=1280)
    m.load_weights(w)
    toks = [tl.tokens(90 + b, s + 2, cfg["vocab"]) for b, s in enumerate(starts)]
    refs = [do.forward(w, cfg, t) for t in toks]
    seqs = [m.open() for _ in starts]
    for s, t, k in zip(seqs, toks, starts):
        m.step([(s, t[:k], [])])
    for i in range(2):
        for some in ([0], [1, 2, 3]):  # (more rows: the weights are asked for behind the row's position)
            got = m.step([(seqs[b], [toks[b][starts[b] + i]], [0]) for b in some])
            tl.assert_close(got, np.stack([refs[b][starts[b] + i] for b in some]), "float32", (i, some))
    m.close()


@pytest.mark.parametrize("n", [2, 6, 7, 8])
@pytest.mark.parametrize("heads,dim,kv_rank", [(13, 128, 512), (40, 64, 512), (64, 64, 256), (24, 128, 264)])
def test_weights_of_many_heads(heads, dim, kv_rank, n):
    """Around the rows x heads x weights from which the five launches take the step: both forms, one layer filing its latents for the next."""
    lat = dict(heads=heads, dim=dim, vdim=4, rot_dim=8, kv_rank=kv_rank)
    cfg = dl.config([dl.latent_layer(mlp=None, **lat), dl.latent_layer(kv_from=0, mlp=None, **lat)], width=32)
    w = dl.weights(cfg, seed=heads)
    check(cfg, w, lambda t: do.forward(w, cfg, t), n, steps=2)
