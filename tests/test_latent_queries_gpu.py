"""Queries of latent attention in prompt portions, carried into the latent space and rotated in one launch: rows around a workgroup's 64, latents
of one piece of 64 columns and of more than a round of four waves, rotary parts without, with some and with all of their channels
rotated, pairs side by side and in halves, queries out of the fused projection, blocks of rows alone and in groups with a ragged last one."""
import pytest

import duvulix_oracle as do
import duvulix_testlib as dl
import lm_oracle
import lm_testlib as tl
from zig_gpt2_amd import lm

pytestmark = pytest.mark.gpu


def run(cfg, w, toks):
    m = lm.LayeredLM(lm.LMConfig.from_json(cfg), dtype="bfloat16", max_tokens=1280, max_seqs=2)
    m.load_weights(w)
    got = m.step([(m.open(), toks, list(range(len(toks))))])
    m.close()
    return got


@pytest.mark.parametrize("rows", [9, 63, 64, 65, 130])
@pytest.mark.parametrize("heads,dim,kv_rank,rot_dim,rot_dims", [(3, 64, 64, 8, 8), (2, 64, 256, 32, 32), (5, 128, 320, 64, 64), (1, 128, 128, 16, 0), (2, 64, 192, 32, 8)])
def test_portions(rows, heads, dim, kv_rank, rot_dim, rot_dims):
    lat = tl.latent_layer(heads=heads, dim=dim, vdim=24, rot_dim=rot_dim, rot_dims=rot_dims, kv_rank=kv_rank, q_rank=40, mlp=tl.dense_mlp(ff=32))
    cfg = tl.config([lat, lat], width=64)
    w = tl.weights(cfg, seed=rows + kv_rank)
    toks = tl.tokens(rows, rows, cfg["vocab"])
    tl.assert_close(run(cfg, w, toks), lm_oracle.Model(cfg, w).forward(toks)[0], "bfloat16", (rows, kv_rank))


@pytest.mark.parametrize("rows,rot_dim", [(33, 16), (129, 32), (64, 64), (70, 8)])
def test_projected_queries(rows, rot_dim):
    cfg = dl.config([dl.latent_layer(heads=2, dim=64, vdim=16, rot_dim=rot_dim, kv_rank=128, mlp=dl.dense(ff=32)),
                     dl.latent_layer(heads=2, dim=64, vdim=16, rot_dim=rot_dim, kv_rank=128, kv_from=0, mlp=dl.dense(ff=32))], width=64)
    w = dl.weights(cfg, seed=rows)
    toks = tl.tokens(rows, rows, cfg["vocab"])
    tl.assert_close(run(cfg, w, toks), do.forward(w, cfg, toks), "bfloat16", rows)


def test_groups_of_blocks():
    lat = tl.latent_layer(heads=130, dim=64, vdim=8, rot_dim=8, kv_rank=64, q_rank=40, mlp=tl.dense_mlp(ff=32))
    cfg = tl.config([lat], width=64)
    w = tl.weights(cfg, seed=4)
    toks = tl.tokens(8, 1030, cfg["vocab"])
    tl.assert_close(run(cfg, w, toks), lm_oracle.Model(cfg, w).forward(toks)[0], "bfloat16")
