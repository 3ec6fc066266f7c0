"""Greedy decode as resident kernels (zig_gpt2_amd/csrc/decode_resident.hip: one sequence, decode_resident_batch.hip: two to eight)
against the launch chain they replace and the oracle: the edges of their shapes (64 positions of a workgroup, 64 steps of a launch,
vocabularies that do not divide by the 256 workgroups, XCDs with no, one and two heads, sequences a tile of terms is not filled by),
what a generation leaves behind, prompts token by token, values that are not finite, other streams, a withdrawn launch
(decode_rest.hip runs its steps) and a wait that runs out."""
import ctypes as C
import time

import numpy as np
import pytest

import oracle
from golden_io import assert_greedy_ids_match
from zig_gpt2_amd import _lib, synth
from zig_gpt2_amd import gpt as zgpt

pytestmark = pytest.mark.gpu

# n_embed 384 (6 heads: two XCDs without), 512 (8), 768 (12: XCDs with one and with two)
SHAPES = {
    "384": synth.GPTConfig(1031, 130, 2, 6, 384),
    "512": synth.GPTConfig(257, 129, 2, 8, 512),
    "768": synth.GPTConfig(65, 200, 3, 12, 768),
    "768-odd": synth.GPTConfig(12289, 66, 2, 12, 768),
}


def make(monkeypatch, cfg, w, resident, **kw):
    monkeypatch.setenv("ZGPT2_RESIDENT", str(int(resident)))
    m = zgpt.GPT(cfg, **kw)
    m.load_weights(w)
    return m


def last_kernel():
    name = C.create_string_buffer(160)
    _lib.check(_lib.load().zg_debug_last_kernel(name, 160))
    return name.value.decode()


def rel(a, b):
    return float(np.linalg.norm(np.float64(a) - np.float64(b)) / np.linalg.norm(np.float64(b)))


@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("f32", [False, True])
def test_same_tokens_and_state_as_the_launch_chain(zg, monkeypatch, name, f32):
    cfg = SHAPES[name]
    w = synth.make_weights(cfg, seed=31, bf16=not f32)
    res, chain = (make(monkeypatch, cfg, w, r, weights_f32=f32) for r in (True, False))
    ctx = cfg.context_size
    for plen, steps in ((1, 1), (1, 2), (3, ctx), (2, 64), (5, 65), (63, ctx), (64, ctx), (ctx - 1, ctx), (ctx, ctx), (9, 5)):
        p = [synth.rand_tokens(300 + plen, plen, cfg.vocab_size)]
        a, b = res.generate(p, steps), chain.generate(p, steps)
        if steps > plen:
            res.generate(p, steps)
            assert "decode_resident_kernel" in last_kernel()
        assert np.array_equal(a, b), (plen, steps)
        # the residual stream, the pick and the cache it leaves: fp32 sums in another order
        if steps > plen:
            assert rel(res.hidden(), chain.hidden()) < 2e-6, (plen, steps)
            assert np.array_equal(res.argmax(), chain.argmax())
        if steps < ctx:
            tok = a[:, -1]
            assert rel(res.forward(steps + 1, tok), chain.forward(steps + 1, tok)) < 2e-6, (plen, steps)
    res.close()
    chain.close()


@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("batch", [2, 3, 4, 5, 8])
def test_lock_step_batch_same_tokens_and_state_as_the_launch_chain(zg, monkeypatch, name, batch):
    cfg = SHAPES[name]
    w = synth.make_weights(cfg, seed=38, bf16=True)
    res, chain = (make(monkeypatch, cfg, w, r, batch=batch) for r in (True, False))
    ctx = cfg.context_size
    for plen, steps in ((1, 1), (2, 64), (6, ctx), (3, 65), (ctx, ctx)):
        p = [synth.rand_tokens(380 + plen + 7 * b, max(1, plen - b), cfg.vocab_size) for b in range(batch)]  # ragged
        a, b = res.generate(p, steps), chain.generate(p, steps)
        res.generate(p, steps)
        assert np.array_equal(a, b), (plen, steps)
        if steps > min(len(q) for q in p):
            assert "decode_resident_batch_kernel" in last_kernel()
            assert rel(res.hidden(), chain.hidden()) < 2e-6, (plen, steps)
            assert np.array_equal(res.argmax(), chain.argmax())
        if steps < ctx:
            assert rel(res.forward(steps + 1, a[:, -1]), chain.forward(steps + 1, a[:, -1])) < 2e-6, (plen, steps)
    res.close()
    chain.close()


@pytest.mark.parametrize("heads,batch,f32", [(6, 1, False), (8, 1, False), (8, 1, True), (6, 2, False), (6, 8, False), (8, 5, False), (8, 8, False)])
def test_contexts_of_2048(zg, monkeypatch, heads, batch, f32):
    """As many positions as the kernels take: 32 splits of a head, and in a batch eight chunks of a split and more."""
    cfg = synth.GPTConfig(301, 2048, 2, heads, 64 * heads)
    w = synth.make_weights(cfg, seed=42, bf16=not f32)
    res, chain = (make(monkeypatch, cfg, w, r, batch=batch, weights_f32=f32) for r in (True, False))
    for plen, steps in ((3, 2048), (1971, 2040), (1023, 1100)):
        p = [synth.rand_tokens(420 + plen + b, plen - b % 3, cfg.vocab_size) for b in range(batch)]
        a, b = res.generate(p, steps), chain.generate(p, steps)
        assert res.resident_stats()["ran"] and not chain.resident_stats()["ran"]
        assert np.array_equal(a, b), (plen, steps, np.argwhere(a != b)[:3])
        assert rel(res.hidden(), chain.hidden()) < 2e-6, (plen, steps)
        if steps < 2048:
            assert rel(res.forward(steps + 1, a[:, -1]), chain.forward(steps + 1, a[:, -1])) < 2e-6, (plen, steps)
    assert res.resident_stats()["rest_steps"] == 0
    res.close()
    chain.close()


def classes(a):
    return np.where(np.isnan(a), 3, np.where(np.isposinf(a), 1, np.where(np.isneginf(a), 2, 0)))


@pytest.mark.parametrize("batch", [1, 3, 8])
@pytest.mark.parametrize("where,what", [("k", np.inf), ("k", -np.inf), ("k", np.nan), ("v", np.inf), ("v", np.nan), ("k", 3e38), ("v", 3e38), ("wpe", np.inf),
                                        ("wpe", np.nan)])
def test_keys_and_values_that_are_not_finite(zg, monkeypatch, batch, where, what):
    """A channel of every key or value, or one position's whole row (from there on in the cache), not finite or at the end of the range:
    tokens and the class of every element of what is left are the chain's."""
    cfg = SHAPES["768"]
    w = dict(synth.make_weights(cfg, seed=43, bf16=True))
    if where == "wpe":
        w["wpe"] = w["wpe"].copy()
        w["wpe"][67, 5] = what
    else:
        w["h1.c_attn_b"] = w["h1.c_attn_b"].copy()
        w["h1.c_attn_b"][(768 if where == "k" else 1536) + 3 * 64 + 7] = what
    p = [synth.rand_tokens(430 + b, 2, cfg.vocab_size) for b in range(batch)]
    res, chain = (make(monkeypatch, cfg, w, r, batch=batch) for r in (True, False))
    for steps in (3, 90):
        a, b = res.generate(p, steps), chain.generate(p, steps)
        assert res.resident_stats()["ran"]
        assert np.array_equal(a, b), steps
        assert np.array_equal(classes(res.hidden()), classes(chain.hidden())), steps
        la, lb = res.forward(steps + 1, a[:, -1]), chain.forward(steps + 1, a[:, -1])
        assert np.array_equal(classes(la), classes(lb)), steps
    res.close()
    chain.close()


@pytest.mark.parametrize("batch", [2, 4, 5, 8])
def test_one_sequence_that_is_not_finite_stays_by_itself(zg, monkeypatch, batch):
    """A token whose embedding is NaN, in one sequence's prompt: the others' tokens, residual streams and logits are those of a batch without it, to the
    bit."""
    cfg = SHAPES["768"]
    w = dict(synth.make_weights(cfg, seed=44, bf16=True))
    w["wte"] = w["wte"].copy()
    w["wte"][64] = np.nan
    p = [synth.rand_tokens(440 + b, 2 + b % 2, 64) for b in range(batch)]
    m = make(monkeypatch, cfg, w, True, batch=batch)
    for bad in (0, batch - 1):
        rest = [b for b in range(batch) if b != bad]
        want, hid = m.generate(p, 100), m.hidden()
        lg = m.forward(101, want[:, -1])
        q = list(p)
        q[bad] = np.array([64, 3], np.uint64)
        got = m.generate(q, 100)
        assert m.resident_stats()["ran"]
        assert np.array_equal(got[rest], want[rest]) and np.array_equal(m.hidden()[rest], hid[rest])
        assert not got[bad, 2:].any() and np.isnan(m.hidden()[bad]).all()
        assert np.array_equal(m.forward(101, got[:, -1])[rest], lg[rest], equal_nan=True)
    m.close()


@pytest.mark.parametrize("batch", [1, 3])
def test_tokens_of_the_oracle(zg, monkeypatch, batch):
    cfg = SHAPES["384"]
    w = synth.make_weights(cfg, seed=32, bf16=True)
    m = make(monkeypatch, cfg, w, True, batch=batch)
    prompts = [synth.rand_tokens(321 + b, 3 - b, cfg.vocab_size) for b in range(batch)]
    ids = m.generate(prompts, cfg.context_size)
    assert "decode_resident_" in last_kernel()
    for p, got in zip(prompts, ids):
        ref, lg = oracle.GPT(cfg, w).generate_greedy(p, cfg.context_size, want_logits=True)
        top = np.sort(lg, axis=1)
        assert_greedy_ids_match(ref[len(p):], got[len(p):], top[:, -1], top[:, -2], "resident decode")
    m.close()


@pytest.mark.parametrize("batch", [1, 5])
def test_nan_logits_pick_index_zero(zg, monkeypatch, batch):
    """As the chain: logits that are all NaN pick index 0, and the next generation on repaired weights is clean."""
    cfg = SHAPES["768"]
    w = synth.make_weights(cfg, seed=33, bf16=True)
    m = make(monkeypatch, cfg, w, True, batch=batch)
    p = [synth.rand_tokens(331 + b, 2, cfg.vocab_size) for b in range(batch)]
    want = m.generate(p, 70)
    bad = dict(w)
    bad["ln_f_g"] = np.full_like(w["ln_f_g"], np.nan)
    m.load_weights(bad)
    assert not m.generate(p, 70)[:, 2:].any()
    m.load_weights(w)
    assert np.array_equal(m.generate(p, 70), want)
    m.close()


@pytest.mark.parametrize("batch", [1, 2])
def test_withdrawn_launch_runs_on_the_chain(zg, monkeypatch, batch):
    """No patience at the start: every workgroup leaves before it has touched anything, and the steps run on what workgroups there are, in
    front of the end of the stream.  The handle then stays on the chain for some generations."""
    cfg = SHAPES["768"]
    w = synth.make_weights(cfg, seed=34, bf16=True)
    p = [synth.rand_tokens(341 + b, 5, cfg.vocab_size) for b in range(batch)]
    chain = make(monkeypatch, cfg, w, False, batch=batch)
    want = chain.generate(p, 150)
    hid = chain.hidden()
    monkeypatch.setenv("ZGPT2_RESIDENT_WITHDRAW", "0")
    m = make(monkeypatch, cfg, w, True, batch=batch)
    assert np.array_equal(m.generate(p, 150), want)
    assert m.resident_stats()["ran"]
    for _ in range(8):
        assert np.array_equal(m.generate(p, 150), want)
        assert not m.resident_stats()["ran"]
    m.generate_enqueue(p, 150)  # tried again, withdrawn again
    assert rel(m.hidden(), hid) < 2e-6
    assert np.array_equal(m.generate_fetch(150), want)
    m.close()
    chain.close()


@pytest.mark.parametrize("name,batch,f32", [("384", 1, False), ("512", 1, True), ("768-odd", 1, False), ("768", 1, True), ("384", 8, False), ("768", 3, False)])
@pytest.mark.parametrize("launch", [0, 1, 2])
def test_launch_withdrawn_behind_others(zg, monkeypatch, name, batch, f32, launch):
    """The first, second or third launch of a generation withdraws, its followers leave at once, and the steps that are missing have run when
    the stream has: no call makes up for them.  Tokens, residual stream, pick, logits and cache are the chain's."""
    import torch

    c = SHAPES[name]
    cfg = synth.GPTConfig(c.vocab_size, 215, c.n_layer, c.n_heads, c.n_embed)
    w = synth.make_weights(cfg, seed=39, bf16=not f32)
    p = [synth.rand_tokens(390 + b, 2 + (3 * b) % 7, cfg.vocab_size) for b in range(batch)]  # ragged; no prompt pass
    steps = 210  # four launches
    chain = make(monkeypatch, cfg, w, False, batch=batch, weights_f32=f32)
    want = chain.generate(p, steps)
    monkeypatch.setenv("ZGPT2_RESIDENT_START", str(1 << 20))  # (0.7 s: not for those behind a withdrawn one)
    monkeypatch.setenv("ZGPT2_RESIDENT_WITHDRAW", str(launch))
    m = make(monkeypatch, cfg, w, True, batch=batch, weights_f32=f32)
    t0 = time.perf_counter()
    m.generate_enqueue(p, steps)
    torch.cuda.synchronize()
    assert time.perf_counter() - t0 < 0.6
    st = m.resident_stats()
    assert st["ran"] and st["rest_steps"] == steps - 64 * launch and st["rest_workgroups"] >= 1, st
    assert np.array_equal(m.generate_fetch(steps), want)
    assert rel(m.hidden(), chain.hidden()) < 2e-6
    assert np.array_equal(m.argmax(), chain.argmax())
    tok = want[:, -1]
    assert rel(m.forward(steps + 1, tok), chain.forward(steps + 1, tok)) < 2e-6
    m.close()
    chain.close()


@pytest.mark.parametrize("name,batch,f32", [("384", 1, False), ("768", 1, True), ("512", 8, False), ("768-odd", 2, False)])
def test_rest_on_the_workgroups_that_came_first(zg, monkeypatch, name, batch, f32):
    """The list of members closed at once: any number of workgroups, another one every time, run the steps."""
    cfg = SHAPES[name]
    w = synth.make_weights(cfg, seed=45, bf16=not f32)
    p = [synth.rand_tokens(450 + b, 1 + b % 4, cfg.vocab_size) for b in range(batch)]
    chain = make(monkeypatch, cfg, w, False, batch=batch, weights_f32=f32)
    want = chain.generate(p, 40)
    monkeypatch.setenv("ZGPT2_RESIDENT_WITHDRAW", "0")
    monkeypatch.setenv("ZGPT2_REST_PATIENCE", "0")
    members = []
    for _ in range(6):
        m = make(monkeypatch, cfg, w, True, batch=batch, weights_f32=f32)
        assert np.array_equal(m.generate(p, 40), want), members
        st = m.resident_stats()
        assert st["rest_steps"] == 40
        members.append(st["rest_workgroups"])
        assert rel(m.hidden(), chain.hidden()) < 2e-6 and np.array_equal(m.argmax(), chain.argmax())
        m.close()
    print("members", members)
    chain.close()


@pytest.mark.parametrize("name,batch,f32", [("384", 1, False), ("768", 1, True), ("384", 6, False), ("768", 2, False)])
@pytest.mark.parametrize("withdraw", [-1, 0, 1])
def test_prompts_token_by_token(zg, monkeypatch, name, batch, f32, withdraw):
    """Handles without the prompt pass: launches that end inside the prompts, whole launches of nothing else, the first pick behind them."""
    cfg = SHAPES[name]
    w = synth.make_weights(cfg, seed=46, bf16=not f32)
    chain = make(monkeypatch, cfg, w, False, batch=batch, weights_f32=f32, prefill=False)
    monkeypatch.setenv("ZGPT2_RESIDENT_WITHDRAW", str(withdraw))
    for plen, steps in ((70, 64), (70, 65), (70, 70), (64, 71), (129, 130), (129, 128), (128, 130)):
        res = make(monkeypatch, cfg, w, True, batch=batch, weights_f32=f32, prefill=False)
        p = [synth.rand_tokens(460 + plen + b, plen - 5 * (b % 3), cfg.vocab_size) for b in range(batch)]
        a, b = res.generate(p, steps), chain.generate(p, steps)
        st = res.resident_stats()
        assert st["ran"] and st["rest_steps"] == (0 if withdraw < 0 or 64 * withdraw >= steps else steps - 64 * withdraw), st
        assert np.array_equal(a, b), (plen, steps)
        assert rel(res.hidden(), chain.hidden()) < 2e-6, (plen, steps)
        if steps > min(len(q) for q in p):
            assert np.array_equal(res.argmax(), chain.argmax())
        if steps < cfg.context_size:
            assert rel(res.forward(steps + 1, a[:, -1]), chain.forward(steps + 1, a[:, -1])) < 2e-6, (plen, steps)
        res.close()
    chain.close()


@pytest.mark.parametrize("batch", [1, 5])
def test_beside_other_streams(zg, monkeypatch, batch):
    """Generations beside matrix products on another stream, whose workgroups want most of a compute unit's LDS, and beside a handle with a
    stream and a thread of its own: the tokens of each on its own, whichever way the steps ran; a product waits for one launch at most."""
    import threading

    import torch

    cfg = synth.GPTConfig(1031, 256, 12, 12, 768)
    w = synth.make_weights(cfg, seed=40, bf16=True)
    p = [synth.rand_tokens(400 + b, 4 + b, cfg.vocab_size) for b in range(batch)]
    m, own = make(monkeypatch, cfg, w, True, batch=batch), make(monkeypatch, cfg, w, True, batch=batch, own_stream=True)
    want = m.generate(p, 256)
    assert m.resident_stats()["ran"] and np.array_equal(own.generate(p, 256), want) and not own.resident_stats()["ran"]
    side = torch.cuda.Stream()
    a = torch.randn(2048, 2048, device="cuda").to(torch.bfloat16)
    ref = a @ a
    torch.cuda.synchronize()
    got = []

    def run():
        for _ in range(3):
            got.append(own.generate(p, 256))

    t = threading.Thread(target=run)
    t.start()
    waits = []
    for _ in range(6):
        m.generate_enqueue(p, 256)
        for _ in range(40):
            t0 = time.perf_counter()
            with torch.cuda.stream(side):
                c = a @ a
                done = torch.cuda.Event()
                done.record(side)
            done.synchronize()
            waits.append(time.perf_counter() - t0)
        assert np.array_equal(m.generate_fetch(256), want)
    t.join()
    assert len(got) == 3 and all(np.array_equal(g, want) for g in got)
    assert torch.equal(c, ref)
    print(f"products waited {1e3 * np.median(waits):.2f} ms, {1e3 * max(waits):.2f} at most; {m.resident_stats()}")
    m.close()
    own.close()


@pytest.mark.parametrize("batch", [1, 4])
def test_wait_that_runs_out_fails_the_call(zg, monkeypatch, batch):
    cfg = SHAPES["512"]
    w = synth.make_weights(cfg, seed=35, bf16=True)
    p = [synth.rand_tokens(351, 2, cfg.vocab_size)] * batch
    monkeypatch.setenv("ZGPT2_TAG_SPIN_LIMIT", "0")
    m = make(monkeypatch, cfg, w, True, batch=batch)
    monkeypatch.delenv("ZGPT2_TAG_SPIN_LIMIT")
    with pytest.raises(_lib.ZgError, match="timed out"):
        m.generate(p, 129)
    m.close()


def test_vocabulary_beyond_the_offsets_stays_on_the_chain(zg):
    """1.4 million tokens of 768 columns: more than 32-bit offsets reach.  The launch chain takes them, as before."""
    import torch

    cfg = synth.GPTConfig(1_400_000, 8, 2, 12, 768)
    m = zgpt.GPT(cfg, prefill=False)
    g = torch.Generator(device="cuda")
    g.manual_seed(41)
    w = {name: torch.randn(shape, generator=g, device="cuda") * 0.02 + mean for name, shape, mean, _ in synth.tensor_specs(cfg)}
    torch.cuda.synchronize()  # (made on torch's stream)
    m.load_weights(w)
    ids = m.generate([[5]], 6)[0]
    assert not m.resident_stats()["ran"]
    x = torch.from_numpy(m.hidden()).cuda()  # of the last step: its pick is the largest product with the normed row
    x = (x - x.mean()) / torch.sqrt(x.var(correction=0) + 1e-5) * w["ln_f_g"] + w["ln_f_b"]
    logits = x @ w["wte"].to(torch.bfloat16).to(torch.float32).T
    assert float(logits[0, int(ids[-1])]) >= float(logits.max()) - 1e-4
    m.close()


def test_what_the_chain_keeps(zg, monkeypatch):
    """Narrow caches, several sequences with fp32 weights, sampling, no graph, one layer: the launch chain, as before."""
    cfg = SHAPES["512"]
    w = synth.make_weights(cfg, seed=36, bf16=True)
    for kw in ({"kv_f16": True}, {"kv_b24": True}, {"use_graph": False}, {"batch": 2, "weights_f32": True}):
        m = make(monkeypatch, cfg, w, True, **kw)
        m.generate([synth.rand_tokens(361, 2, cfg.vocab_size)] * m.batch, 20)
        assert "decode_resident" not in last_kernel(), kw
        m.close()
    one = synth.GPTConfig(257, 129, 1, 8, 512)
    m = make(monkeypatch, one, synth.make_weights(one, seed=37, bf16=True), True)
    m.generate([synth.rand_tokens(361, 2, one.vocab_size)], 20)
    assert "decode_resident" not in last_kernel()
    m.close()
    m = make(monkeypatch, cfg, w, True)
    m.generate_sample([synth.rand_tokens(361, 2, cfg.vocab_size)], 20, 0.8, seed=3)
    assert "decode_resident" not in last_kernel()
    m.close()
