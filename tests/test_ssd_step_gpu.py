"""State space layers in decode steps: a token of every entry with the convolution inside, the norm where the output product reads its rows and
the convolution's tails moved on in that launch; states of fewer and more rows than the threads hold, columns at the edges of a workgroup's,
one tap to more than the kernel's, norms in parts and rows too long or too ragged for the product."""
import numpy as np
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 8])
@pytest.mark.parametrize("heads,vdim,state,groups,conv,norm_groups", [(24, 64, 128, 1, 4, 1), (4, 4, 1, 2, 1, 1), (6, 36, 33, 3, 2, 1), (2, 32, 256, 1, 3, 1), (4, 100, 96, 2, 4, 2),
                                                                      (3, 24, 32, 1, 7, 1), (4, 10, 64, 2, 4, 1), (1, 12, 40, 1, 4, 1), (33, 128, 64, 1, 4, 1), (8, 200, 17, 1, 4, 1)])
def test_one_token_of_every_entry(heads, vdim, state, groups, conv, norm_groups, n):
    cfg = dl.config([dl.mamba_layer(heads=heads, vdim=vdim, state=state, groups=groups, conv=conv, norm_groups=norm_groups, mlp=dl.dense(ff=32)) for _ in range(2)], width=48)
    w = dl.weights(cfg, seed=vdim + state)
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="float32", max_tokens=512, max_seqs=8)
    m.load_weights(w)
    starts, steps = [5, 0, 2, 40, 1, 3, 0, 9][:n], 5  # (more steps than taps reach back)
    toks = [dl.tokens(b, s + steps, cfg["vocab"]) for b, s in enumerate(starts)]
    refs = [do.forward(w, cfg, t) for t in toks]
    seqs = [m.open() for _ in starts]
    begun = [(s, t[:k], []) for s, t, k in zip(seqs, toks, starts) if k > 0]
    if begun:
        m.step(begun)
    for i in range(steps):
        got = m.step([(s, [t[k + i]], [0]) for s, t, k in zip(seqs, toks, starts)])
        want = np.stack([r[k + i] for r, k in zip(refs, starts)])
        # (fp32 sums through two layers: the layered tier's bound for 32-bit mode)
        assert np.abs(got - want).max() < 3e-5 * np.abs(want).max(), (n, i)
    m.close()


@pytest.mark.parametrize("n", [5, 6, 8])
@pytest.mark.parametrize("heads,vdim", [(16, 64), (86, 12), (16, 128), (32, 128), (129, 32)])
def test_norms_of_long_rows(heads, vdim, n):
    """Rows of up to 1024 columns are normed inside the product, longer ones in a launch in front of the product that splits them over sixteen waves."""
    test_one_token_of_every_entry(heads, vdim, 16, 1, 4, 1, n)
