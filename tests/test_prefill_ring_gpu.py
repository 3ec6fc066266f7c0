"""The ring kernel of prompts of some hundred rows (prefill_ring.hip): Linear.forward of src/ops.zig:21-46 for M = batch x prompt
rows.  bf16 weights one Linear at a time against a float64 product of the same operands: single rows, ragged last tiles, one
K step, an odd number of them, tiles of 64 and of 128 rows, K slices.  fp32 weights (two planes, three or four products; three planes of a small model's) through whole
small models against the oracle, every Linear forced onto the ring."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from golden_io import assert_model_close, assert_ref_close
from test_prefill_linear_gpu import bf16_round, gelu64, planes_to_f64, split3
from zig_gpt2_amd import _lib, synth
from zig_gpt2_amd import gpt as zgpt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,epilogue", [
    (1, 64, 64, 0), (63, 128, 192, 0), (65, 192, 128, 2), (300, 768, 768, 1), (300, 768, 3072, 1), (300, 3072, 768, 2), (129, 1600, 320, 1), (577, 2048, 128, 2), (600, 1856, 64, 0)])
def test_ring_linear_matches_float64(zg, M, N, K, epilogue):
    x = synth.fill_normal(21, M * K, 0, 1.0).reshape(M, K)
    w = bf16_round(synth.fill_normal(22, N * K, 0, 0.05).reshape(N, K))
    bias = synth.fill_normal(23, N, 0, 0.1)
    c0 = synth.fill_normal(24, M * N, 0, 1.0).reshape(M, N)
    ref = x.astype(np.float64) @ w.astype(np.float64).T + bias
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    a_d, w_d, b_d = dev(split3(x).view(np.int16)), dev(synth.to_bf16_bits(w).view(np.int16)), dev(bias)
    ws = torch.zeros(4 * M * N, dtype=torch.float32, device="cuda")
    c_d = dev(c0) if epilogue == 1 else torch.zeros((M, 3 * N), dtype=torch.int16, device="cuda") if epilogue == 2 else torch.zeros((M, N), device="cuda")
    torch.cuda.synchronize()  # (the fills above run on torch's stream, the library launches on its own)
    _lib.check(zg.zg_debug_prefill_linear(a_d.data_ptr(), w_d.data_ptr(), b_d.data_ptr(), c_d.data_ptr(), M, N, K, epilogue, 3, 0, ws.data_ptr(), ws.numel()))
    torch.cuda.synchronize()
    name = C.create_string_buffer(128)
    _lib.check(zg.zg_debug_last_kernel(name, 128))
    assert name.value.decode().startswith("prefill_ring_kernel"), "the ring kernel did not run"
    got = c_d.cpu().numpy()
    if epilogue == 2:
        ref, got = gelu64(ref), planes_to_f64(got.view(np.uint16), N)
    assert_ref_close(ref + c0 if epilogue == 1 else ref, got, f"ring {M}x{N}x{K} epilogue {epilogue}", scale_floor=2e-6)


@pytest.mark.parametrize("name,batch,n,f32,kv_f16", [("tiny", 1, 1, True, False), ("tiny3", 3, 47, True, False), ("xl-slice", 1, 95, True, False), ("medium-slice", 2, 79, True, True),
                                                     ("nano-char", 4, 200, True, False), ("xl-slice", 7, 70, False, False), ("nano-char", 1, 255, False, True)])
def test_ring_prompt_matches_oracle(zg, name, batch, n, f32, kv_f16):
    cfg = synth.CONFIGS[name]
    w = synth.make_weights(cfg, seed=131, bf16=not f32)
    m = zgpt.GPT(cfg, batch=batch, weights_f32=f32, kv_f16=kv_f16)
    m.load_weights(w)
    toks = np.stack([synth.rand_tokens(1310 + b, n + 1, cfg.vocab_size) for b in range(batch)])
    _lib.check(zg.zg_debug_prefill_route(3, 0))
    try:
        lg = m.prefill(toks[:, :n]).copy()
    finally:
        _lib.check(zg.zg_debug_prefill_route(0, 0))
    nxt = m.forward(n + 1, toks[:, n])
    for b in {0, batch - 1}:
        ref = oracle.GPT(cfg, w).forced_logits(toks[b], n - 1)
        assert_model_close(ref[0], lg[b], f"{name} ring prefill row {b}")
        if not kv_f16:  # (fp16 caches: the next step reads them rounded)
            assert_model_close(ref[1], nxt[b], f"{name} decode on a ring prefill, row {b}")
    m.close()
