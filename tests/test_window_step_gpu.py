"""Attention of decode steps in two launches: shares of one key group and of many, the row's own token alone in its share, chunks that have just begun,
key heads read by one head to eight and by more, channels at the kernel's edges and beyond them, rotary pairs of both kinds and unrotated
channels, and windows with kept first tokens behind a preparation of their own."""
import numpy as np
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
import sanazen_oracle as so
import sanazen_testlib as sl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu

STARTS = [290, 15, 0, 256, 16, 255, 31, 1]  # tokens in front of the first step


def check(cfg, w, forward, tokens, n, steps=3):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=1536, max_seqs=8)
    m.load_weights(w)
    starts = STARTS[:n]
    toks = [tokens(40 + b, s + steps, cfg["vocab"]) for b, s in enumerate(starts)]
    refs = [forward(t) for t in toks]
    seqs = [m.open() for _ in starts]
    begun = [(s, t[:k], []) for s, t, k in zip(seqs, toks, starts) if k > 0]
    if begun:
        m.step(begun)
    for i in range(steps):
        got = m.step([(s, [t[k + i]], [0]) for s, t, k in zip(seqs, toks, starts)])
        want = np.stack([r[k + i] for r, k in zip(refs, starts)])
        # (fp32 sums through one layer: the layered tier's bound for 32-bit mode)
        assert np.abs(got - want).max() < 3e-5 * np.abs(want).max(), (n, i)
    m.close()


@pytest.mark.parametrize("n", [1, 3, 8])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,size,rot_dims", [(12, 3, 64, 64, 512, 64), (4, 4, 4, 4, 9, 4), (8, 1, 128, 36, 16, 64), (3, 1, 68, 128, 300, 6), (5, 5, 64, 132, 64, 10),
                                                                   (2, 1, 12, 8, 1, 12), (9, 1, 64, 64, 40, 64), (4, 2, 30, 8, 40, 30), (6, 1, 40, 6, 40, 0)])
def test_chunks(heads, kv_heads, dim, vdim, size, rot_dims, n):
    cfg = dl.config([dl.attn_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, size=size, rot_dims=rot_dims, scale=dim ** -0.5, mlp=dl.dense(ff=32))], width=48)
    w = dl.weights(cfg, seed=dim + vdim)
    check(cfg, w, lambda t: do.forward(w, cfg, t), dl.tokens, n)


@pytest.mark.parametrize("n", [1, 3, 8])
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,window,keep", [(4, 2, 64, 64, 40, 4), (2, 1, 8, 12, 17, 20), (3, 3, 128, 100, 0, 0), (8, 1, 16, 16, 300, 1)])
def test_windows_with_kept_tokens(heads, kv_heads, dim, vdim, window, keep, n):
    cfg = sl.config([sl.pair_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, window=window, keep_first=keep)])
    w = sl.weights(cfg, seed=dim + window)
    check(cfg, w, lambda t: so.forward(w, cfg, t)[0], sl.tokens, n)


@pytest.mark.parametrize("n", [1, 3])
@pytest.mark.parametrize("dim,vdim", [(8, 8), (68, 128)])
def test_scores_of_minus_infinity(dim, vdim, n):
    """Keys whose scores fall below what fp32 holds weigh nothing, a whole share of them too."""
    cfg = dl.config([dl.attn_layer(heads=2, kv_heads=1, dim=dim, vdim=vdim, size=None, rot_dims=0, scale=1.0, mlp=None)], vocab=89, width=48)
    w = dl.weights(cfg, seed=dim)
    q, k = (next(x for x in w if x.endswith(leaf)) for leaf in ("mix.q", "mix.k"))
    w["embed"] = w["embed"].copy()
    w["embed"][:, 0] = 0.0
    w["embed"][7, 0] = 1.0  # token 7: a key of -2^70 and more in its first channel
    w["embed"][:, 1] = 1.0  # every token: a query of 2^70 there
    w[q], w[k] = w[q].copy(), w[k].copy()
    w[q][0::dim] = 0.0
    w[q][0::dim, 1] = 2.0 ** 72
    w[k][0] = 0.0
    w[k][0, 0] = -(2.0 ** 72)
    w[q][:, 0] = 0.0
    w[k][1:, 0] = 0.0
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=1536, max_seqs=8)
    m.load_weights(w)
    toks = [dl.tokens(40 + b, 150 + 16 * b, cfg["vocab"]) for b in range(n)]
    for b, t in enumerate(toks):
        t[t == 7] = 8
        t[16:130 + b] = 7
    refs = [do.forward(w, cfg, t) for t in toks]
    seqs = [m.open() for _ in toks]
    m.step([(s, t[:-2], []) for s, t in zip(seqs, toks)])
    for i in (-2, -1):
        got = m.step([(s, [t[i]], [0]) for s, t in zip(seqs, toks)])
        want = np.stack([r[i] for r in refs])
        assert np.abs(got - want).max() < 3e-5 * np.abs(want).max(), (n, i)
    m.close()
