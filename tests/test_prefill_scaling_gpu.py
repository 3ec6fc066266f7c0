"""One whole-prompt Linear and the prompt attention with exponents that lie binades above what the data need, as a model's do, whose weights they follow from: against
float64, with the bound that two fp16 terms of such exponents have.  (2^14 to 2^15 is where the largest value lies with no slack: what a term cannot hold is 2^(slack - 39) of it.)"""
import numpy as np
import pytest
import torch

from test_attn_prefill_gpu import ref_attention
from test_prefill_linear_gpu import bf16_round, gelu64, planes_to_f64, split3
from zig_gpt2_amd import _lib, synth

pytestmark = pytest.mark.gpu
dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("kernel", [1, 2, 3])
@pytest.mark.parametrize("slack", [0, 3, 8, 14, 20])
@pytest.mark.parametrize("M,N,K,epilogue", [(300, 768, 768, 1), (520, 384, 1536, 1), (600, 768, 256, 2), (257, 192, 128, 2)])
def test_linear(zg, kernel, slack, M, N, K, epilogue):
    x = synth.fill_normal(11, M * K, 0, 1.0).reshape(M, K)
    w = bf16_round(synth.fill_normal(12, N * K, 0, 0.05).reshape(N, K))
    bias = synth.fill_normal(13, N, 0, 0.1)
    c0 = synth.fill_normal(14, M * N, 0, 1.0).reshape(M, N)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    ref = x64 @ w64.T + bias
    a_d, w_d, b_d = dev(split3(x).view(np.int16)), dev(synth.to_bf16_bits(w).view(np.int16)), dev(bias)
    ws = torch.zeros(8 * M * N, dtype=torch.float32, device="cuda")
    c_d = dev(c0) if epilogue == 1 else torch.zeros((M, 3 * N), dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    _lib.check(zg.zg_debug_prefill_linear_at(a_d.data_ptr(), w_d.data_ptr(), b_d.data_ptr(), c_d.data_ptr(), M, N, K, epilogue, kernel, 0, ws.data_ptr(), ws.numel(), slack, 1, None))
    torch.cuda.synchronize()
    # the sums: 2^-23 of every product for the terms, 2^-24 for every addition of the matrix cores, what lies below the terms
    bound = (2.0 ** -23 + K / 8 * 2.0 ** -24) * (np.abs(x64) @ np.abs(w64).T) + 2.0 ** (slack - 39) * np.abs(x64).max() * np.abs(w64).sum(1)
    if epilogue == 1:
        got, ref = c_d.cpu().numpy().astype(np.float64), ref + c0
        bound = bound + 2.0 ** -22 * (np.abs(ref) + np.abs(c0) + np.abs(bias))
    else:
        got = planes_to_f64(c_d.cpu().numpy().view(np.uint16), N)
        most = np.linalg.norm(x64, axis=1).max() * np.linalg.norm(w64, axis=1).max() + np.abs(bias).max()
        # (the slope of GELU is below 1.13; its own 32-bit evaluation some 2^-21)
        bound = 1.13 * (bound + 2.0 ** -23 * np.abs(bias)) + 2.0 ** -21 * np.abs(ref) + 2.0 ** (slack - 39) * most
        ref = gelu64(ref)
    assert (np.abs(got - ref) <= bound).all(), (np.abs(got - ref) / bound).max()


@pytest.mark.parametrize("slack", [0, 3, 8, 14, 20])
@pytest.mark.parametrize("B,P,H,groups", [(2, 33, 2, 0), (1, 300, 4, 0), (1, 300, 4, 1), (2, 257, 3, 1)])
def test_attention(zg, slack, B, P, H, groups):
    E = 64 * H
    qkv = synth.fill_normal(31 + P, B * P * 3 * E, 0, 1.0).reshape(B * P, 3 * E)
    ref = ref_attention(qkv, B, P, E, H)
    qkv_d, out = dev(qkv), torch.zeros((B * P, 3 * E), dtype=torch.int16, device="cuda")
    torch.cuda.synchronize()
    _lib.check(zg.zg_debug_attn_prefill_at(qkv_d.data_ptr(), out.data_ptr(), B, P, E, H, None, None, 0, None, 0, groups, slack, 1, None))
    torch.cuda.synchronize()
    got = planes_to_f64(out.cpu().numpy().view(np.uint16), E)
    top = np.abs(qkv).max()
    # a score is off by what q and k lose in 64 products, an output by twice that of the values' spread, and by what v and it lose itself
    lost = 2.0 ** (slack - 39) * top
    assert np.abs(got - ref).max() <= 2e-6 * np.abs(ref).max() + lost * (2 * 64 * np.abs(qkv).mean() / 8 * 2 * top + 2)
