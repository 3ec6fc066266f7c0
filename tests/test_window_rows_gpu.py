"""Windowed attention of prompt portions in one launch: rows around a block's 32, portions behind a context of their own length, heads one to one
with key heads up to many on one (groups of one to four heads a workgroup, two to eight ranges of the keys), heads and values below and at the
kernel's 64 channels and beyond them, chunks and windows whose edges lie inside a block, kept tokens, capped scores, gated results, rounded results."""
import numpy as np
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
import lm_testlib as tl
import sanazen_oracle as so
import sanazen_testlib as sl
import vovalorn_oracle as vo
import vovalorn_testlib as vl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def check(cfg, w, forward, tokens, portions, dtype="float32"):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=1536, max_seqs=4)
    m.load_weights(w)
    toks = [tokens(40 + b, sum(p), cfg["vocab"]) for b, p in enumerate(portions)]
    refs = [forward(t) for t in toks]
    seqs = [m.open() for _ in portions]
    at = [0] * len(portions)
    for i in range(len(portions[0])):
        batch = [(s, t[k:k + p[i]], list(range(p[i]))) for s, t, k, p in zip(seqs, toks, at, portions) if p[i]]
        got = m.step(batch)
        want = np.concatenate([r[k:k + p[i]] for r, k, p in zip(refs, at, portions) if p[i]])
        if dtype == "float32":  # (fp32 sums through one layer: the layered tier's bound for 32-bit mode)
            assert np.abs(got - want).max() < 3e-5 * np.abs(want).max(), (i, np.abs(got - want).max() / np.abs(want).max())
        else:
            tl.assert_close(got, want, dtype, i)
        at = [k + p[i] for k, p in zip(at, portions)]
    m.close()


PORTIONS = [[(33, 64), (1, 32)], [(9, 130)], [(257, 31), (40, 9), (0, 65)]]


@pytest.mark.parametrize("portions", PORTIONS)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,size", [(12, 3, 64, 64, 512), (4, 4, 8, 4, 9), (6, 3, 32, 36, 16), (3, 1, 56, 64, 33), (5, 1, 64, 28, 64), (16, 1, 16, 12, 100), (4, 2, 72, 8, 40)])
def test_chunks(heads, kv_heads, dim, vdim, size, portions):
    cfg = dl.config([dl.attn_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, size=size, scale=dim ** -0.5, mlp=dl.dense(ff=32))], width=48)
    w = dl.weights(cfg, seed=dim + vdim)
    for dtype in ("float32", "bfloat16"):
        check(cfg, w, lambda t: do.forward(w, cfg, t), dl.tokens, portions, dtype)


@pytest.mark.parametrize("portions", PORTIONS)
@pytest.mark.parametrize("heads,kv_heads,dim,vdim,window,keep", [(4, 2, 64, 64, 40, 4), (2, 1, 8, 12, 17, 20), (3, 3, 24, 60, 0, 0), (8, 1, 16, 16, 300, 1), (4, 1, 32, 32, 1, 40)])
def test_windows_with_kept_tokens(heads, kv_heads, dim, vdim, window, keep, portions):
    cfg = sl.config([sl.pair_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=vdim, window=window, keep_first=keep)])
    w = sl.weights(cfg, seed=dim + window)
    check(cfg, w, lambda t: so.forward(w, cfg, t)[0], sl.tokens, portions)


@pytest.mark.parametrize("portions", PORTIONS)
@pytest.mark.parametrize("heads,kv_heads,dim,softcap", [(4, 2, 64, 8.0), (6, 2, 16, 0.0), (7, 1, 40, 3.0)])
def test_capped_scores(heads, kv_heads, dim, softcap, portions):
    cfg = vl.config([vl.attn_layer(heads=heads, kv_heads=kv_heads, dim=dim, softcap=softcap, mlp=vl.moe_mlp())])
    w = vl.weights(cfg, seed=dim)
    check(cfg, w, lambda t: vo.forward(w, cfg, t), vl.tokens, portions)


@pytest.mark.parametrize("n", [9, 33])
@pytest.mark.parametrize("heads,kv_heads,dim,size", [(5, 1, 64, None), (12, 2, 16, 100), (21, 3, 8, None), (3, 3, 32, 33)])
def test_many_sequences_of_one_row(heads, kv_heads, dim, size, n):
    """Blocks of one row each, beside one of many rows: workgroups of every number of heads, the last of a key head's with fewer."""
    cfg = dl.config([dl.attn_layer(heads=heads, kv_heads=kv_heads, dim=dim, vdim=12, size=size, scale=dim ** -0.5, mlp=dl.dense(ff=32))], width=48)
    w = dl.weights(cfg, seed=heads)
    for dtype in ("float32", "bfloat16"):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=8192, max_seqs=n, max_step_tokens=256)
        m.load_weights(w)
        starts = [(37 * b + 5) % 150 for b in range(n)]
        toks = [dl.tokens(40 + b, k + 45, cfg["vocab"]) for b, k in enumerate(starts)]
        refs = [do.forward(w, cfg, t) for t in toks]
        seqs = [m.open() for _ in toks]
        for s, t, k in zip(seqs, toks, starts):
            m.step([(s, t[:k], [])])
        for more in (1, 40):  # every sequence a row; then the last one forty of them
            got = m.step([(s, t[k:k + (more if b == n - 1 else 1)], [0]) for b, (s, t, k) in enumerate(zip(seqs, toks, starts))])
            want = np.stack([r[k] for r, k in zip(refs, starts)])
            if dtype == "float32":
                assert np.abs(got - want).max() < 3e-5 * np.abs(want).max(), more
            else:
                tl.assert_close(got, want, dtype, more)
            starts = [k + 1 for k in starts]
        m.close()


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("dim,vdim,size", [(16, 16, 128), (64, 64, 128), (32, 44, 40), (64, 28, 7)])
def test_values_that_are_not_finite(dim, vdim, size, dtype, bad):
    """A row that is not finite reaches the rows that see it and no others, those in front of it and of the next chunk in its block of 32 included."""
    cfg = dl.config([dl.attn_layer(heads=4, kv_heads=2, dim=dim, vdim=vdim, size=size, scale=dim ** -0.5, mlp=dl.dense(ff=32))], width=48)
    w = dl.weights(cfg, seed=3)
    toks = dl.tokens(5, 90, cfg["vocab"])
    toks[toks == 7] = 8
    ref = do.forward(w, cfg, toks)
    toks[75] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = bad
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=512, max_seqs=2)
    m.load_weights(w)
    got = m.step([(m.open(), toks, list(range(90)))])
    m.close()
    sees = np.array([r >= 75 and r // size == 75 // size for r in range(90)])
    assert not np.isfinite(got[sees]).any(axis=1).any() and np.isfinite(got[~sees]).all()
    if dtype == "float32":
        assert np.abs(got[~sees] - ref[~sees]).max() < 3e-5 * np.abs(ref).max()
    else:
        tl.assert_close(got[~sees], ref[~sees], dtype)
