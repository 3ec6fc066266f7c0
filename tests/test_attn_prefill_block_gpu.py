"""The causal prompt attention of a few prompts (blocks of 32 queries, their key tiles dealt over four waves) against float64 and against the kernel of
many prompts: tiles fewer than waves and one more, a last block of one query and of 32, sequences whose neighbours and caches hold NaN behind the
prompt, one key far above the rest in each wave's share."""
import numpy as np
import pytest
import torch

from test_attn_prefill_gpu import planes_to_f64, ref_attention
from zig_gpt2_amd import _lib, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 32, 33, 96, 97, 128, 129, 160, 161, 257, 289])
@pytest.mark.parametrize("cache", [False, True])
def test_blocks(zg, P, cache):
    B, H, ctx = 2, 2, P + 3
    E = 64 * H
    qkv = synth.fill_normal(5 + P, B * P * 3 * E, 0, 1.0).reshape(B * P, 3 * E)
    for t in range(7, P, 67):  # the running maximum moves by more than its deferral, in tiles of several waves
        qkv[t, E:E + 64] = 9.0 * np.sign(qkv[P - 1, :64])
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    qkv_d, kc, vc = dev(qkv), None, None
    if cache:
        x = qkv.reshape(B, P, 3, H, 64)
        full = np.full((2, B, H, ctx, 64), np.nan, np.float32)
        full[:, :, :, :P] = x[:, :, 1:].transpose(2, 0, 3, 1, 4)
        kc, vc = dev(full[0]), dev(full[1])
        qkv_d[:, E:] = float("nan")
    ref = ref_attention(qkv, B, P, E, H)
    err = []
    for groups in (0, 1):
        out = torch.zeros((B * P, 3 * E), dtype=torch.int16, device="cuda")
        torch.cuda.synchronize()
        _lib.check(zg.zg_debug_attn_prefill(qkv_d.data_ptr(), out.data_ptr(), B, P, E, H, kc.data_ptr() if cache else None, vc.data_ptr() if cache else None, ctx, None, 0, groups))
        torch.cuda.synchronize()
        got = planes_to_f64(out.cpu().numpy().view(np.uint16), E)
        assert np.isfinite(got).all()
        err.append(np.abs(got - ref).max() / np.abs(ref).max())
    # scores of up to 9 * 64 / 8 * 2: their 2^-23 relative error of split and products, some 70 * 2^-22, is the probabilities' own
    assert err[0] < 2e-5 and err[0] < 1.5 * err[1] + 1e-7, err
