"""The recurrences with a decay per key channel in chunks of 64 tokens (lm_scan.hip), against the float64 oracles: head sizes around
the kernels' tiles, entries that end around blocks and chunks, gates from nearly one to nearly zero, values that are not finite."""
import numpy as np
import pytest

import lm_oracle
import lm_testlib as tl
import vovalorn_oracle
import vovalorn_testlib as vl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def steps(m, toks, cuts):
    """Feed every sequence up to its cut in each step (all of them in one call); the logits of all rows, per sequence."""
    seqs, lo, rows = [m.open() for _ in toks], [0] * len(toks), [[] for _ in toks]
    for cut in cuts:
        hi = [min(c, len(t)) for c, t in zip(cut, toks)]
        got = m.step([(s, t[a:b], list(range(b - a))) for s, t, a, b in zip(seqs, toks, lo, hi)])
        at = 0
        for i, (a, b) in enumerate(zip(lo, hi)):
            rows[i].append(got[at:at + b - a])
            at += b - a
        lo = hi
    for s in seqs:
        m.close_seq(s)
    return [np.concatenate(r) for r in rows]


def assert_rows_close(got, model, w, toks, what):
    """Every row within TOL, or within eight times what perturbing the embedding and the query map by one part in 2^24 does to it: where
    a head's q . k nearly cancels, the norm behind the head magnifies the rounding of its inputs (sequence 1, row 187 of the smallest
    heads at once forgotten: 3.6e-5 for a perturbation of 6e-8; the median row 5e-8)."""
    ref = model(w).forward(toks)[0]
    scale, moved = np.abs(ref).max(), np.zeros(len(ref))
    for seed in range(3):
        rng, near = np.random.default_rng(seed), dict(w)
        for name in ("embed", "l0.mix.q"):
            near[name] = np.asarray(w[name], np.float64) * (1 + 2.0**-24 * rng.standard_normal(w[name].shape))
        moved = np.maximum(moved, np.abs(model(near).forward(toks)[0] - ref).max(axis=1) / scale)
    err = np.abs(np.asarray(got, np.float64) - ref).max(axis=1) / scale
    assert (err < np.maximum(tl.TOL["float32"], 8 * moved)).all(), (what, err.max(), err.argmax())


CUTS = [(33, 1, 65), (97, 64, 66), (161, 192, 129), (200, 193, 200)]


@pytest.mark.parametrize("heads,dim,vdim", [(2, 16, 24), (1, 40, 72), (2, 64, 64), (1, 100, 130), (1, 128, 33), (2, 128, 128)])
@pytest.mark.parametrize("forget", ["slow", "mixed", "sudden"])
def test_hgrn2_chunks(heads, dim, vdim, forget):
    cfg = tl.config([tl.hgrn2_layer(heads=heads, dim=dim, vdim=vdim)], vocab=97, width=64)
    w = tl.weights(cfg, seed=dim + vdim, lower={"slow": (0.97, 1.0), "mixed": (0.0, 1.0), "sudden": (0.0, 1e-4)}[forget])
    if forget == "sudden":  # gates down to 1e-6: their products underflow within a block
        w["l0.mix.f.b"] = w["l0.mix.f.b"] - 10.0
    toks = [tl.tokens(90 + b, 200, cfg["vocab"]) for b in range(3)]
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=1024, max_seqs=3)
    m.load_weights(w)
    for got, t in zip(steps(m, toks, CUTS), toks):
        assert_rows_close(got, lambda v: lm_oracle.Model(cfg, v), w, t[: len(got)], (dim, vdim, forget))
    m.close()


@pytest.mark.parametrize("heads,dim,vdim", [(2, 12, 10), (1, 64, 96), (1, 72, 64), (2, 128, 128)])
@pytest.mark.parametrize("bias", [6.0, 0.0, -9.0])
def test_gla_chunks(heads, dim, vdim, bias):
    cfg = vl.config([vl.gla_layer(heads=heads, dim=dim, vdim=vdim, tau=2.0)])
    w = vl.weights(cfg, seed=dim + vdim)
    w["l0.mix.a2.b"] = w["l0.mix.a2.b"] + np.float32(bias)
    toks = [vl.tokens(95 + b, 200, cfg["vocab"]) for b in range(3)]
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=1024, max_seqs=3)
    m.load_weights(w)
    for got, t in zip(steps(m, toks, CUTS), toks):
        tl.assert_close(got, vovalorn_oracle.forward(w, cfg, t[: len(got)]), "float32", (dim, vdim, bias))
    m.close()


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("at", [64, 71, 90, 127])
def test_rows_in_front_of_a_value_that_is_not_finite(bad, at):
    cfg = tl.config([tl.hgrn2_layer(heads=2, dim=32, vdim=64)], vocab=97, width=64)
    w = tl.weights(cfg, seed=4)
    toks = tl.tokens(5, 150, cfg["vocab"])
    toks[toks == 7] = 8
    ref = lm_oracle.Model(cfg, w).forward(toks)[0]
    toks[at] = 7
    w["embed"] = w["embed"].copy()
    w["embed"][7, 3] = bad
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=512, max_seqs=1)
    m.load_weights(w)
    got = steps(m, [toks], [(150,)])[0]
    m.close()
    assert np.isnan(got[at:]).any(axis=1).all()
    tl.assert_close(got[:at], ref[:at], "float32", (bad, at))
