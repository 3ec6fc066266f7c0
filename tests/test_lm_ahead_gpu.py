"""Generation that enqueues its steps ahead against the same steps taken one by one (use_graph=False takes them so): tokens of greedy and
sampled runs longer than the ring of steps in flight, pages that run over and go back to the pool behind windows, key-length buckets,
and a cache that is full half way."""
import numpy as np
import pytest

import duvulix_testlib as dl
import gupizen_testlib as gl
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu

DESIGNS = {
    "latent": (tl, tl.config([tl.hgrn2_layer(mlp=tl.moe_mlp()), tl.latent_layer(mlp=tl.dense_mlp())], vocab=97, width=48)),
    "chunks": (dl, dl.config([dl.attn_layer(mlp=dl.dense()), dl.attn_layer(size=5, mlp=None)], width=48)),
    "mixed": (dl, dl.config([dl.mamba_layer(mlp=dl.dense()), dl.latent_layer(mlp=dl.dense()), dl.attn_layer(mlp=None)], width=48)),
    "whole": (dl, dl.config([dl.attn_layer(size=None, mlp=dl.dense())], width=48)),
}


@pytest.mark.parametrize("n_seqs", [1, 3, 8])
@pytest.mark.parametrize("design", sorted(DESIGNS))
def test_tokens_of_steps_ahead(design, n_seqs):
    lib, cfg = DESIGNS[design]
    w = lib.weights(cfg, seed=7)
    prompts = [lib.tokens(b, 3 + 5 * b, cfg["vocab"]) for b in range(n_seqs)]
    runs = []
    for use_graph in (True, False):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=1024, max_seqs=8, page_tokens=8, use_graph=use_graph)
        m.load_weights(w)
        runs.append([m.generate(prompts, n, temp=t, seed=s) for n, t, s in ((1, 0.0, 0), (2, 0.0, 0), (9, 0.0, 0), (40, 0.0, 0), (40, 1.5, 5))])
        runs[-1].append(m.generate(prompts, 40))  # the slots and pages are all back
        m.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("page_tokens", [1, 3])
@pytest.mark.parametrize("design", sorted(DESIGNS))
def test_a_page_every_step(design, page_tokens):
    """Every sequence grows by a page with nearly every step in flight, and tables of windowed designs wrap round."""
    lib, cfg = DESIGNS[design]
    w = lib.weights(cfg, seed=11)
    prompts = [lib.tokens(b, 2 + 3 * b, cfg["vocab"]) for b in range(8)]
    runs = []
    for use_graph in (True, False):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=768, max_seqs=8, page_tokens=page_tokens, use_graph=use_graph)
        m.load_weights(w)
        runs.append([m.generate(prompts, 60), m.generate(prompts[::-1], 33, temp=1.0, seed=3)])
        m.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("page_tokens", [4, 5, 64])
@pytest.mark.parametrize("design", ["latent", "chunks"])
def test_steps_enqueued_four_at_a_time(design, page_tokens):
    """Lengths around whole fours, prompts that end anywhere in a page: fours, single steps, and both in turn."""
    lib, cfg = DESIGNS[design]
    w = lib.weights(cfg, seed=13)
    runs = []
    for use_graph in (True, False):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=512, max_seqs=4, page_tokens=page_tokens, use_graph=use_graph)
        m.load_weights(w)
        runs.append([m.generate([lib.tokens(b, n + b, cfg["vocab"]) for b in range(3)], new) for n, new in ((1, 5), (2, 6), (3, 7), (4, 8), (6, 9), (9, 21), (11, 38))])
        m.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


def test_key_buckets():
    lib, cfg = DESIGNS["whole"]
    w = lib.weights(cfg, seed=2)
    prompts = [lib.tokens(1, 500, cfg["vocab"])]
    runs = []
    for use_graph in (True, False):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=2048, max_seqs=2, use_graph=use_graph)
        m.load_weights(w)
        runs.append(m.generate(prompts, 30))
        m.close()
    assert np.array_equal(*runs)


def test_a_cache_that_is_full_half_way():
    lib, cfg = DESIGNS["latent"]
    w = lib.weights(cfg, seed=3)
    prompts = [lib.tokens(b, 6, cfg["vocab"]) for b in range(2)]
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=48, max_seqs=4, page_tokens=8)
    m.load_weights(w)
    want = m.generate(prompts, 17)
    with pytest.raises(Exception, match="pages needed|tokens in the cache"):
        m.generate(prompts, 60)
    assert np.array_equal(m.generate(prompts, 17), want)
    m.close()


def without_canon(layers, **kw):
    """Mixers with a convolution of their own behind a token shift (no convolution of the sublayers' inputs)."""
    cfg = gl.config(layers, **kw)
    del cfg["canon"]
    return cfg


CONVOLVED = {
    "delta": without_canon([gl.delta_layer(conv=4, mlp=gl.moe_mlp()), gl.delta_layer(conv=2, mlp=None)]),
    "parallel": without_canon([gl.parallel_layer(conv=4, mlp=gl.moe_mlp()), gl.parallel_layer(conv=2, mlp=None)]),
    "both": without_canon([gl.parallel_layer(conv=4, mlp=None), gl.delta_layer(conv=4, mlp=gl.moe_mlp()), gl.parallel_layer(conv=16, mlp=gl.moe_mlp())]),
    "one tap": without_canon([gl.delta_layer(conv=1, mlp=gl.moe_mlp())]),
}


@pytest.mark.parametrize("n_seqs", [1, 3, 8])
@pytest.mark.parametrize("design", sorted(CONVOLVED))
def test_convolutions_of_the_mixers(design, n_seqs):
    """A row's place inside its entry stays 0 through a generation: every token's convolution reads its own slot's tail."""
    cfg = CONVOLVED[design]
    w = gl.weights(cfg, seed=7)
    prompts = [gl.tokens(b, 1 + 3 * b, cfg["vocab"]) for b in range(n_seqs)]
    runs = []
    for use_graph in (True, False):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=1024, max_seqs=8, page_tokens=8, use_graph=use_graph)
        m.load_weights(w)
        runs.append([m.generate(prompts, n, temp=t, seed=s) for n, t, s in ((3, 0.0, 0), (40, 0.0, 0), (20, 1.5, 5), (40, 0.0, 0))])
        m.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


def against_single_steps(lib, cfg, dtype, n_seqs, n=24):
    w = lib.weights(cfg, seed=5)
    prompts = [lib.tokens(b, 2 + 4 * b, cfg["vocab"]) for b in range(n_seqs)]
    runs = []
    for use_graph in (True, False):
        m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype=dtype, max_tokens=1024, max_seqs=8, page_tokens=8, use_graph=use_graph)
        m.load_weights(w)
        runs.append([m.generate(prompts, n), m.generate(prompts[:1], n)])
        m.close()
    for a, b in zip(*runs):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n_seqs", [1, 3, 8])
@pytest.mark.parametrize("loop", [{"start": 0, "stop": 3, "times": 2}, {"start": 1, "stop": 2, "times": 3}, {"start": 2, "stop": 3, "times": 2}])
def test_looped_stacks(loop, n_seqs):
    cfg = tl.config([tl.hgrn2_layer(mlp=tl.moe_mlp()), tl.latent_layer(mlp=None), tl.hgrn2_layer(mlp=tl.dense_mlp())], width=48, loop=loop)
    cfg.update(logit_scale=0.5, logit_softcap=3.0)
    against_single_steps(tl, cfg, "float32", n_seqs)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [1020, 1024, 1028])
def test_widths_around_what_a_wave_holds(width, dtype):
    """Rows of more than 1024 columns are not handed on inside a step: the kernels of single steps there, links of a chain up to it."""
    for n_seqs in (1, 3):
        against_single_steps(tl, tl.config([tl.hgrn2_layer(mlp=tl.moe_mlp()), tl.latent_layer(mlp=tl.dense_mlp())], width=width), dtype, n_seqs)
        against_single_steps(dl, dl.config([dl.mamba_layer(mlp=dl.dense()), dl.attn_layer(mlp=None), dl.latent_layer(mlp=dl.dense())], width=width), dtype, n_seqs)
        against_single_steps(gl, without_canon([gl.delta_layer(mlp=gl.moe_mlp()), gl.parallel_layer(mlp=None)], width=width), dtype, n_seqs)


@pytest.mark.parametrize("design", sorted(DESIGNS) + sorted(CONVOLVED))
def test_bfloat16(design):
    lib, cfg = DESIGNS[design] if design in DESIGNS else (gl, CONVOLVED[design])
    against_single_steps(lib, cfg, "bfloat16", 8, 40)
