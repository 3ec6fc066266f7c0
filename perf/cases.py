"""What the framework is timed on: the work its users have it do, through its public entry points.

Six kinds of case, over the three tiers:

  linear         ops.Linear.forward on device buffers: one row (a token at a time) to 8192 rows (a batch of prompts), fp32.
  gpt_generate   GPT.generate (greedy, GPT-2 layer shapes), then GPT.forward of the last token for the next token's logits.
  gpt_prompt     GPT.prefill: a batch of prompts in one pass, logits of the last position.
  lm_generate    LayeredLM.generate (greedy), then one step over the whole text: the logits a caller scores the answer with.
  lm_prompt      LayeredLM.step over whole prompts, logits of every prompt's last position.
  lm_portions    LayeredLM.step as a continuous-batching server calls it: prompts of different lengths fed in portions, sequences
                 that are through with their prompt decoding a token beside them.

Sizes are those of this repository's configurations and benchmark: GPT-2 124M, XL and the char model; the layered stacks of
width 768 x 12 layers ("small") and 1024 x 24 ("medium").  Checkpoints do not exist offline: weights are drawn on the GPU, once
per model, with the traits of trained ones that matter here (branch gains of 1 / sqrt(2 layers), balanced experts with routers
that are sure of most tokens, a head that is sure of most next tokens); the seed of a case draws its inputs.
"""
import math

import numpy as np
import torch

from zig_gpt2_amd import _lib, gpt, lm, ops, synth

DEV = "cuda"


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # a few rows through one Linear of the op tier (a caller that batches eight tokens): launch and completion latency
        {"name": "linear_8x768x3072", "kind": "linear", "m": 8, "k": 768, "n": 3072},
        # the MLP's up-projection over eight prompts at once
        {"name": "linear_8192x768x3072", "kind": "linear", "m": 8192, "k": 768, "n": 3072},
        # the char model answering one short prompt: the smallest generation there is
        {"name": "gpt_char_generate", "kind": "gpt_generate", "model": "nano-char", "prompts": 1, "prompt_len": 16, "steps": 96, "weights": "bf16"},
        # the headline path: one sequence from its first token on
        {"name": "gpt_124m_generate_1", "kind": "gpt_generate", "model": "124M", "prompts": 1, "prompt_len": 1, "steps": 256, "weights": "bf16"},
        # eight answers in lock step behind prompts of different lengths
        {"name": "gpt_124m_generate_8", "kind": "gpt_generate", "model": "124M", "prompts": 8, "prompt_len": 75, "steps": 256, "weights": "bf16"},
        # one ordinary prompt on an ordinary (fp32) checkpoint
        {"name": "gpt_124m_prompt_1x300_f32", "kind": "gpt_prompt", "model": "124M", "prompts": 1, "prompt_len": 300, "weights": "f32"},
        # eight full contexts
        {"name": "gpt_124m_prompt_8x1023", "kind": "gpt_prompt", "model": "124M", "prompts": 8, "prompt_len": 1023, "weights": "bf16"},
        # a dense layered stack answering one user
        {"name": "duvulix_generate_1", "kind": "lm_generate", "design": "Duvulix", "size": "small", "prompts": 1, "prompt_len": 21, "new": 64, "dtype": "bfloat16"},
        # a stack with experts answering eight users in one batch
        {"name": "tokosun_generate_8", "kind": "lm_generate", "design": "Tokosun", "size": "small", "prompts": 8, "prompt_len": 37, "new": 48, "dtype": "bfloat16"},
        # a server's iterations: ragged prompts in portions of 256 tokens beside decoding sequences
        {"name": "duvulix_portions_8", "kind": "lm_portions", "design": "Duvulix", "size": "small", "prompts": 8, "prompt_len": 700, "portion": 256,
         "dtype": "bfloat16"},
        # a prompt on the 32-bit option
        {"name": "tokosun_prompt_1x333_f32", "kind": "lm_prompt", "design": "Tokosun", "size": "small", "prompts": 1, "prompt_len": 333, "dtype": "float32"},
        # eight full contexts on the medium stack with experts
        {"name": "tokosun_medium_prompt_8x1023", "kind": "lm_prompt", "design": "Tokosun", "size": "medium", "prompts": 8, "prompt_len": 1023,
         "dtype": "bfloat16"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "gpt_generate", "gpt_prompt", "lm_generate", "lm_prompt", "lm_prompt", "lm_portions"])
    if kind == "linear":
        e = rng.choice([384, 768, 1600])
        k, n = rng.choice([(e, 3 * e), (e, e), (e, 4 * e), (4 * e, e), (e, 65), (e, 1031)])
        return {"kind": kind, "m": _log_int(rng, 1, 8192), "k": k, "n": n}
    if kind == "gpt_generate":
        model, most = rng.choice([("nano-char", 240), ("124M", 240), ("xl", 24)])
        prompts = _log_int(rng, 1, 8 if model != "xl" else 4)
        steps = _log_int(rng, 12, most)
        return {"kind": kind, "model": model, "prompts": prompts, "prompt_len": _log_int(rng, 1, max(1, steps // 2)), "steps": steps,
                "weights": "bf16" if model == "xl" else rng.choice(["bf16", "bf16", "f32"])}
    if kind == "gpt_prompt":
        model, most = rng.choice([("nano-char", 255), ("124M", 1023), ("xl", 700)])
        return {"kind": kind, "model": model, "prompts": _log_int(rng, 1, 8 if model != "xl" else 2), "prompt_len": _log_int(rng, 9, most),
                "weights": "bf16" if model == "xl" else rng.choice(["bf16", "f32"])}
    design, size = rng.choice(["Tokosun", "Duvulix"]), rng.choice(["small", "small", "medium"])
    prompts = _log_int(rng, 1, 8)
    if kind == "lm_generate":
        return {"kind": kind, "design": design, "size": size, "prompts": prompts, "prompt_len": _log_int(rng, 1, 200),
                "new": _log_int(rng, 8, 48 if size == "small" else 20), "dtype": "bfloat16"}
    if kind == "lm_prompt":
        dtype = rng.choice(["bfloat16", "bfloat16", "float32"])
        most = 1023 if dtype == "bfloat16" else max(20, 600 // prompts)
        return {"kind": kind, "design": design, "size": "small" if dtype == "float32" else size, "prompts": prompts, "prompt_len": _log_int(rng, 9, most), "dtype": dtype}
    return {"kind": kind, "design": design, "size": size, "prompts": prompts, "prompt_len": _log_int(rng, 40, 700), "portion": rng.choice([64, 100, 256]),
            "dtype": "bfloat16"}


# ------------------------------------------------------------------------------------------------ models a program keeps
SIZES = {"small": (768, 12), "medium": (1024, 24)}
VOCAB = 50257
_models, _weights, _started = {}, {}, []


def _start():
    if not _started:
        _lib.check(_lib.load().zg_init(0))
        _started.append(True)


def _generator(*key):
    g = torch.Generator(device=DEV)
    g.manual_seed(sum(int(v) * m for v, m in zip(key, (1, 1_000_003, 7_919, 104_729))) % (1 << 62))
    return g


def _bf16(t):
    return t.to(torch.bfloat16).to(torch.float32)


def gpt_weights(model, kind):
    """GPT-2's initial distribution; "f32": an ordinary checkpoint, "bf16": one whose matrices are bf16-representable."""
    cfg, g, w = synth.CONFIGS[model], _generator(17, list(synth.CONFIGS).index(model)), {}
    for name, shape, mean, _ in synth.tensor_specs(cfg):
        t = torch.randn(shape, generator=g, device=DEV) * 0.02 + mean
        w[name] = _bf16(t) if kind == "bf16" else t
    return w


def gpt_model(case):
    key = (case["model"], case["prompts"], case["weights"])
    if key not in _models:
        _start()
        m = gpt.GPT(synth.CONFIGS[case["model"]], batch=case["prompts"], weights_f32=case["weights"] == "f32")
        m.load_weights(gpt_weights(case["model"], case["weights"]))
        _models[key] = m
    return _models[key]


def lm_config(design, size):
    """The stacks of the repository's benchmark: the two designs of the layered tier that between them have a matrix-state
    recurrence, a state space, latent attention, attention in chunks, dense feed-forwards of both kinds and experts."""
    width, n_layers = SIZES[size]
    heads = width // 64
    if design == "Tokosun":
        rec = dict(mixer="hgrn2", heads=width // 128, dim=128, vdim=128)
        att = dict(mixer="latent_attention", heads=heads, dim=64, vdim=64, rot_dim=32, kv_rank=256, q_rank=384, scale=96 ** -0.5, rot_dims=32, rot_base=10000.0,
                   rot_scaling={"factor": 4.0, "original": 2048, "fast": 32.0, "slow": 1.0})
        dense, moe = dict(ff="dense", ff_width=4 * width), dict(ff="moe", ff_width=width, experts=8, top=2)
        order = [dict(rec, **dense), dict(att, **moe), dict(att, **moe), dict(rec, **moe)]
        return lm.LMConfig(vocab=VOCAB, width=width, layers=[lm.LayerSpec(**order[i % 4]) for i in range(n_layers)], norm_eps=1e-6)
    dense = dict(ff="dense", ff_width=4 * width, dense_act="polynorm", rot_halves=True)
    ssm = dict(mixer="ssd", heads=2 * width // 64, vdim=64, dim=128, kv_heads=1, conv=4, norm_groups=1, **dense)
    lat = dict(mixer="latent_attention", heads=heads, dim=64, vdim=64, rot_dim=32, kv_rank=256, scale=96 ** -0.5, rot_dims=32, rot_base=10000.0, head_gate=True,
               **dense)
    att = dict(mixer="rotary_attention", heads=heads, kv_heads=heads // 4, dim=64, vdim=64, scale=64 ** -0.5, chunk=512, rot_dims=64, rot_base=10000.0,
               rot_scaling={"factor": 8.0, "original": 1024, "fast": 24.0, "slow": 2.0}, **dense)
    layers = [lm.LayerSpec(**[ssm, lat, dict(lat, kv_from=i - 1), att][i % 4]) for i in range(n_layers)]
    return lm.LMConfig(vocab=VOCAB, width=width, layers=layers, norm_eps=1e-6, architecture="Duvulix")


def lm_weights(design, size):
    """name -> fp32 tensor on the GPU; matrices are bf16-representable.  Tokens come in kinds, a kind's embedding leans towards
    two directions, and a layer's router sends a direction to an expert of its own: the load is balanced and most choices are
    clear.  The head prefers one successor per token clearly enough that the greedy choice is seldom close."""
    cfg = lm_config(design, size)
    W, L = cfg.width, len(cfg.layers)
    g = _generator(29, list(SIZES).index(size), len(design))

    def normal(*shape):
        return torch.randn(shape, generator=g, device=DEV)

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=g, device=DEV) * (hi - lo) + lo

    directions = torch.linalg.qr(normal(W, 8))[0].T.contiguous()
    own = normal(VOCAB, W)
    first = torch.randint(0, 8, (VOCAB,), generator=g, device=DEV)
    second = (first + torch.randint(1, 8, (VOCAB,), generator=g, device=DEV)) % 8
    successor = torch.randperm(VOCAB, generator=g, device=DEV)
    w = {}
    for name, shape in cfg.tensor_shapes().items():
        last = name.split(".", 1)[-1]
        if name == "embed":
            t = 1.5 * (own + 0.35 * math.sqrt(W) * (directions[first] + 0.6 * directions[second]))
        elif name == "head":
            t = 0.02 * normal(*shape)
            t[successor] += 7.68 / W * own
        elif last == "mlp.router":
            t = 0.3 * directions[torch.randperm(8, generator=g, device=DEV)] + 0.002 * normal(*shape)
        elif last in ("norm1b", "norm2b"):
            t = 1.0 / math.sqrt(2 * L) - 1.0 + 0.03 * normal(*shape)
        elif last in ("norm1", "norm2", "norm") and len(shape) == 1:
            t = 0.1 * normal(*shape)
        elif last == "shift":
            t = uniform(shape, 0.0, 0.5)
        elif last == "mlp.correction":
            t = 0.01 * normal(*shape)
        elif last == "mlp.act":
            t = torch.tensor([0.5, 0.3, 0.2, 0.05], device=DEV)
        elif last == "mix.lower":
            t = uniform(shape, 0.3, 0.98)
        elif last == "mix.f.b":
            t = 1.0 + 0.5 * normal(*shape)
        elif last == "mix.A_log":
            t = torch.log(uniform(shape, 1.0, 16.0))
        elif last == "mix.dt_bias":
            t = torch.log(torch.expm1(torch.exp(uniform(shape, math.log(1e-3), math.log(0.1)))))
        elif last == "mix.conv":
            t = 0.4 * normal(*shape)
        elif last == "mix.conv.b":
            t = 0.1 * normal(*shape)
        elif last in ("mix.D", "mix.norm", "mix.dq.norm", "mix.dkv.norm"):
            t = 1.0 + 0.1 * normal(*shape)
        else:
            assert len(shape) == 2, name
            t = 0.02 * normal(*shape)
        w[name] = _bf16(t) if len(shape) == 2 else t.to(torch.float32)
    return w


def lm_model(case):
    key = (case["design"], case["size"], case["dtype"])
    if key not in _models:
        _start()
        m = lm.LayeredLM(lm_config(case["design"], case["size"]), dtype=case["dtype"], max_tokens=8 * 1024 + 64, max_seqs=8, max_step_tokens=8 * 1024)
        m.load_weights({n: t.cpu().numpy() for n, t in lm_weights(case["design"], case["size"]).items()})
        _models[key] = m
    return _models[key]


# ------------------------------------------------------------------------------------------------ inputs
def _tokens(seed, vocab, *shape):
    return np.random.default_rng([int(seed), 5]).integers(0, vocab, shape)


def _ragged(case, seed):
    """Prompts of case["prompts"] different lengths, the longest of case["prompt_len"] tokens."""
    B, n = case["prompts"], case["prompt_len"]
    vocab = synth.CONFIGS[case["model"]].vocab_size if "model" in case else VOCAB
    lens = [max(1, n - (b * n) // (2 * B)) for b in range(B)]
    t = _tokens(seed, vocab, B, n)
    return [t[b, : lens[b]].astype(np.uint64 if "model" in case else np.int32) for b in range(B)]


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "linear":
        _start()
        g = _generator(seed, case["m"], case["n"])
        m, k, n = case["m"], case["k"], case["n"]
        w, b = torch.randn(n, k, generator=g, device=DEV) * 0.02, torch.randn(n, generator=g, device=DEV) * 0.02
        s.update(layer=ops.Linear(k, n, w, b), x=torch.randn(m, k, generator=g, device=DEV), y=torch.empty(m, n, device=DEV))
    elif kind == "gpt_generate":
        s.update(model=gpt_model(case), prompts=_ragged(case, seed))
    elif kind == "gpt_prompt":
        m = gpt_model(case)
        s.update(model=m, tokens=_tokens(seed, m.config.vocab_size, case["prompts"], case["prompt_len"]).astype(np.uint64))
    elif kind == "lm_prompt":
        s.update(model=lm_model(case), tokens=_tokens(seed, VOCAB, case["prompts"], case["prompt_len"]).astype(np.int32))
    else:
        s.update(model=lm_model(case), prompts=_ragged(case, seed))
        if kind == "lm_portions":
            s.update(rounds=_rounds(s["prompts"], case["portion"], _tokens(seed + 1, VOCAB, case["prompts"], 64).astype(np.int32)))
    return s


def _rounds(prompts, portion, answers):
    """The steps of a server that feeds every prompt `portion` tokens at a time and lets sequences decode meanwhile, until the
    last prompt is through: per step [(sequence number, its tokens, places whose logits are asked for)]."""
    fed, said, rounds = [0] * len(prompts), [0] * len(prompts), []
    while any(f < len(p) for f, p in zip(fed, prompts)):
        entries = []
        for b, p in enumerate(prompts):
            if fed[b] < len(p):
                t = p[fed[b]: fed[b] + portion]
                fed[b] += len(t)
                entries.append((b, t, [len(t) - 1] if fed[b] == len(p) else []))
            else:
                entries.append((b, answers[b, said[b] % 64: said[b] % 64 + 1], [0]))
                said[b] += 1
        rounds.append(entries)
    return rounds


# ------------------------------------------------------------------------------------------------ one pass
def run(state):
    kind, m = state["case"]["kind"], state.get("model")
    if kind == "linear":
        state["layer"].forward(state["x"], state["y"])
        return state["y"]
    if kind == "gpt_generate":
        steps = state["case"]["steps"]
        tokens = m.generate(state["prompts"], steps)
        return {"tokens": tokens, "logits": m.forward(steps + 1, tokens[:, -1])}
    if kind == "gpt_prompt":
        return m.prefill(state["tokens"])
    if kind == "lm_prompt":
        seqs = [m.open() for _ in state["tokens"]]
        logits = m.step([(s, t, [len(t) - 1]) for s, t in zip(seqs, state["tokens"])])
        for s in seqs:
            m.close_seq(s)
        return logits
    if kind == "lm_generate":
        tokens = m.generate(state["prompts"], state["case"]["new"])
        seqs = [m.open() for _ in tokens]
        logits = m.step([(s, np.concatenate([p, t]), [len(p) + len(t) - 1]) for s, p, t in zip(seqs, state["prompts"], tokens)])
        for s in seqs:
            m.close_seq(s)
        return {"tokens": tokens, "logits": logits}
    seqs = [m.open() for _ in state["prompts"]]
    out = [m.step([(seqs[b], t, want) for b, t, want in entries]) for entries in state["rounds"]]
    for s in seqs:
        m.close_seq(s)
    return [o for o in out if o.size]


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _lm_matrices(cfg):
    """(elements of every matrix but the embedding, elements a token multiplies with, the head's among both)."""
    stored = used = 0
    for name, shape in cfg.tensor_shapes().items():
        if len(shape) != 2 or name == "embed":
            continue
        n = shape[0] * shape[1]
        lay = cfg.layers[int(name[1: name.index(".")])] if name.startswith("l") else None
        stored += n
        used += n * lay.top / lay.experts if ".mlp.e" in name else n
    return stored, used


def _lm_attention(cfg, pairs):
    """Multiply-adds of the attention layers: `pairs` (query, key) pairs of one sequence, scores and weighted sum per head."""
    return sum(lay.heads * (lay.dim + lay.rot_dim + lay.vdim) * pairs for lay in cfg.layers if "attention" in lay.mixer)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + n * k + n + m * n), "flops": 2 * m * n * k}
    if "model" in case:
        c, B, wb = synth.CONFIGS[case["model"]], case["prompts"], 2 if case["weights"] == "bf16" else 4
        E, L, V = c.n_embed, c.n_layer, c.vocab_size
        block = 12 * L * E * E
        if kind == "gpt_prompt":
            n = case["prompt_len"]
            return {"bytes": wb * (block + V * E) + 8 * B * n * E * L + 4 * B * V, "flops": 2 * B * (n * block + V * E) + 4 * B * L * E * n * (n + 1) // 2}
        lens = [len(p) for p in _ragged(case, 0)]
        steps = case["steps"] - min(lens) + 2  # the prompts in one pass, then a pass per token, then the logits
        keys = sum(t for n in lens for t in range(n, case["steps"] + 2))
        rows = sum(case["steps"] + 1 - n for n in lens)
        return {"bytes": steps * wb * (block + V * E) + 8 * E * L * keys + 4 * B * V,
                "flops": 2 * (rows * (block + V * E) + sum(lens) * block) + 4 * L * E * keys}
    cfg = lm_config(case["design"], case["size"])
    stored, used = _lm_matrices(cfg)
    head = VOCAB * cfg.width
    B = case["prompts"]
    if kind == "lm_prompt":
        n = case["prompt_len"]
        return {"bytes": 2 * stored + 4 * B * VOCAB, "flops": 2 * (B * n * (used - head) + B * head) + 2 * _lm_attention(cfg, B * n * (n + 1) // 2)}
    if kind == "lm_generate":
        lens, new = [len(p) for p in _ragged(case, 0)], case["new"]
        rows, touched = B * new, min(stored, used * B)
        pairs = 2 * sum((n + new) * (n + new + 1) // 2 for n in lens)
        return {"bytes": 2 * (touched * (new - 1) + 2 * stored) + 4 * B * VOCAB,
                "flops": 2 * (rows * used + (2 * sum(lens) + rows) * (used - head) + B * head) + 2 * _lm_attention(cfg, pairs)}
    rounds = _rounds(_ragged(case, 0), case["portion"], np.zeros((B, 64), np.int32))
    rows, wants = sum(len(t) for r in rounds for _, t, _ in r), sum(len(w) for r in rounds for _, _, w in r)
    pairs = sum(n * (n + 1) // 2 for n in [len(p) for p in _ragged(case, 0)])
    return {"bytes": 2 * stored * len(rounds) + 4 * wants * VOCAB, "flops": 2 * (rows * (used - head) + wants * head) + 2 * _lm_attention(cfg, pairs)}


def tolerance(case):
    """About four times the error against 64 bits that was measured (in brackets)."""
    if case["kind"] == "linear":  # fp32 operands and sums (1.6e-7)
        return {"rel": 1e-6, "max": 1e-5}
    if "model" in case or case["dtype"] == "float32":  # fp32 activations and sums through a whole model (2e-7 to 6e-7; GPT-2 XL has 48 layers)
        return {"rel": 4e-6, "max": 4e-5, "differ": 0.01}
    return {"rel": 6e-3, "max": 4e-2, "differ": 0.01}  # activations rounded to bf16 in front of a prompt's matrix products (1.6e-3)


# ------------------------------------------------------------------------------------------------ the same in 64 bits
F = torch.float64


def _d(t):
    return t.to(F)


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        s = prepare(case, seed)
        return _d(s["x"]) @ _d(s["layer"].weight).T + _d(s["layer"].bias)
    with torch.no_grad():
        if kind == "gpt_prompt":
            m = synth.CONFIGS[case["model"]]
            tokens = _tokens(seed, m.vocab_size, case["prompts"], case["prompt_len"])
            return GptExact(case).forward(torch.as_tensor(tokens, device=DEV))[:, -1].cpu().numpy()
        if kind == "gpt_generate":
            return GptExact(case).generate(_ragged(case, seed), case["steps"])
        if kind == "lm_prompt":
            tokens = torch.as_tensor(_tokens(seed, VOCAB, case["prompts"], case["prompt_len"]), device=DEV)
            return lm_exact(case, tokens, torch.full((case["prompts"], 1), case["prompt_len"] - 1, device=DEV))[:, 0].cpu().numpy()
        prompts = _ragged(case, seed)
        if kind == "lm_generate":
            return _lm_generate_exact(case, prompts)
        rounds = _rounds(prompts, case["portion"], _tokens(seed + 1, VOCAB, case["prompts"], 64).astype(np.int32))
        text, asked = [[] for _ in prompts], []
        for entries in rounds:
            asked.append([(b, len(text[b]) + w) for b, t, want in entries for w in want])
            for b, t, _ in entries:
                text[b] += t.tolist()
        tokens, flat = _padded(text), [a for r in asked for a in r]
        most = max(sum(1 for c in flat if c[0] == b) for b in range(len(text)))
        at = torch.zeros(len(text), most, dtype=torch.int64)
        place, count = {}, [0] * len(text)
        for b, pos in flat:
            at[b, count[b]] = pos
            place[b, pos] = count[b]
            count[b] += 1
        logits = lm_exact(case, tokens, at.to(DEV)).cpu().numpy()
        return [np.stack([logits[b, place[b, pos]] for b, pos in r]) for r in asked if r]


def _padded(rows):
    n = max(len(r) for r in rows)
    return torch.as_tensor([list(map(int, r)) + [0] * (n - len(r)) for r in rows], device=DEV)


class GptExact:
    """GPT-2 over whole sequences and, with kept keys and values, a token at a time."""

    def __init__(self, case):
        self.c = synth.CONFIGS[case["model"]]
        self.w = {k: _d(v) for k, v in gpt_weights(case["model"], case["weights"]).items()}

    def forward(self, tokens, at=0, cache=None):
        c, w = self.c, self.w
        B, n = tokens.shape
        H, E = c.n_heads, c.n_embed

        def norm(x, name):
            x = x - x.mean(-1, keepdim=True)
            return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w[name + "_g"] + w[name + "_b"]

        x = w["wte"][tokens] + w["wpe"][at: at + n]
        for l in range(c.n_layer):
            p = f"h{l}."
            q, k, v = (norm(x, p + "ln_1") @ w[p + "c_attn_w"].T + w[p + "c_attn_b"]).reshape(B, n, 3, H, E // H).permute(2, 0, 3, 1, 4)
            if cache is not None:
                cache[l][0][:, :, at: at + n], cache[l][1][:, :, at: at + n] = k, v
                k, v = cache[l][0][:, :, : at + n], cache[l][1][:, :, : at + n]
            s = q @ k.transpose(-1, -2).contiguous() / math.sqrt(E // H)
            if n > 1:
                s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -math.inf)
            o = (torch.softmax(s, -1) @ v.contiguous()).transpose(1, 2).reshape(B, n, E)
            x = x + o @ w[p + "c_proj_w"].T + w[p + "c_proj_b"]
            h = norm(x, p + "ln_2") @ w[p + "c_fc_w"].T + w[p + "c_fc_b"]
            h = 0.5 * h * (1.0 + torch.tanh(0.7978845608 * (h + 0.044715 * h ** 3)))
            x = x + h @ w[p + "mlp_proj_w"].T + w[p + "mlp_proj_b"]
        return norm(x[:, -1:], "ln_f") @ w["wte"].T

    def generate(self, prompts, steps):
        """The reference's loop: position s takes the prompt's token, or the last one (behind the prompt: its last token again)."""
        c, B = self.c, len(prompts)
        cache = [[torch.zeros(B, c.n_heads, steps + 1, c.n_embed // c.n_heads, dtype=F, device=DEV) for _ in (0, 1)] for _ in range(c.n_layer)]
        given, lens = _padded(prompts), torch.as_tensor([len(p) for p in prompts], device=DEV)
        last, out = given[:, 0], []
        for s in range(steps + 1):
            inside = s < lens
            fed = torch.where(inside, given[:, min(s, given.shape[1] - 1)], last)
            logits = self.forward(fed[:, None], s, cache)[:, 0]
            last = torch.where(inside, fed, logits.argmax(-1))
            out.append(last)
        return {"tokens": torch.stack(out[:steps], 1).cpu().numpy().astype(np.uint64), "logits": logits.cpu().numpy()}


def _unit(v, eps=1e-6):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)


def _rotate(v, lay, positions):
    """v [B, n, heads, channels]: the first rot_dims channels turned as pairs, interleaved or in halves."""
    d, base = lay.rot_dims, lay.rot_base
    f = np.array([base ** (-2.0 * i / d) for i in range(d // 2)])
    amp, sc = 1.0, lay.rot_scaling
    if sc:
        corr = lambda turns: d * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(corr(sc["fast"])), 0), min(math.ceil(corr(sc["slow"])), d - 1)
        ramp = np.clip((np.arange(d // 2) - lo) / max(hi - lo, 0.001), 0.0, 1.0)
        f, amp = f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
    # (an angle is the 32-bit product of position and frequency by definition)
    a = _d(positions.to(torch.float32)[:, None] * torch.as_tensor(f, device=DEV).to(torch.float32)[None])[None, :, None]
    c, s, out = torch.cos(a) * amp, torch.sin(a) * amp, v.clone()
    i, j = (slice(0, d // 2), slice(d // 2, d)) if lay.rot_halves else (slice(0, d, 2), slice(1, d, 2))
    out[..., i], out[..., j] = v[..., i] * c - v[..., j] * s, v[..., j] * c + v[..., i] * s
    return out


def _attend(q, k, v, scale, seen):
    """q [B, n, H, D], k [B, n, H, D], v [B, n, H, V], seen [n, n]."""
    s = q.permute(0, 2, 1, 3).contiguous() @ k.permute(0, 2, 3, 1).contiguous() * scale
    return (torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v.permute(0, 2, 1, 3).contiguous()).permute(0, 2, 1, 3)


def _mixer(lay, w, u, pos, latents, li):
    B, n, _ = u.shape
    H, D, V, R = lay.heads, lay.dim, lay.vdim, lay.rot_dim
    seen = pos[None, :] <= pos[:, None]
    if lay.mixer == "hgrn2":
        q = torch.nn.functional.silu(u @ w["q"].T).reshape(B, n, H, D)
        v = (u @ w["v"].T).reshape(B, n, H, V)
        f = (w["lower"] + (1.0 - w["lower"]) * torch.sigmoid(u @ w["f"].T + w["f.b"])).reshape(B, n, H, D, 1)
        S, o = torch.zeros(B, H, D, V, dtype=F, device=DEV), torch.empty(B, n, H, V, dtype=F, device=DEV)
        for t in range(n):
            S = torch.lerp(v[:, t, :, None, :].expand_as(S), S, f[:, t])
            o[:, t] = (q[:, t, :, None, :] @ S)[:, :, 0]
        return (_unit(o) * w["norm"]).reshape(B, n, H * V) @ w["o"].T
    if lay.mixer == "latent_attention":
        q = u @ w["q"].T if not lay.q_rank else (_unit(u @ w["dq"].T) * w["dq.norm"]) @ w["uq"].T
        q = q.reshape(B, n, H, D + R)
        if lay.kv_from is None:
            t = u @ w["dkv"].T
            latents[li] = _unit(t[..., : lay.kv_rank]) * w["dkv.norm"], _rotate(t[..., None, lay.kv_rank:], lay, pos)
        c, kr = latents[li if lay.kv_from is None else lay.kv_from]
        k = torch.cat([(c @ w["uk"].T).reshape(B, n, H, D), kr.expand(B, n, H, R)], -1)
        o = _attend(torch.cat([q[..., :D], _rotate(q[..., D:], lay, pos)], -1), k, (c @ w["uv"].T).reshape(B, n, H, V), lay.scale, seen)
        if lay.head_gate:
            o = o * torch.sigmoid(u @ w["g"].T)[..., None]
        return o.reshape(B, n, H * V) @ w["o"].T
    if lay.mixer == "rotary_attention":
        G = lay.kv_heads
        q, k = _rotate((u @ w["q"].T).reshape(B, n, H, D), lay, pos), _rotate((u @ w["k"].T).reshape(B, n, G, D), lay, pos)
        v = (u @ w["v"].T).reshape(B, n, G, V)
        seen = seen & (pos[None, :] // lay.chunk == pos[:, None] // lay.chunk)
        o = _attend(q, k.repeat_interleave(H // G, 2), v.repeat_interleave(H // G, 2), lay.scale, seen)
        return o.reshape(B, n, H * V) @ w["o"].T
    inner, N = H * V, D  # state space, one group of B and C
    t = u @ w["in"].T
    z, xbc, dt = t[..., :inner], t[..., inner: 2 * inner + 2 * N], torch.nn.functional.softplus(t[..., 2 * inner + 2 * N:] + w["dt_bias"])
    taps = lay.conv
    full = torch.cat([torch.zeros(B, taps - 1, xbc.shape[-1], dtype=F, device=DEV), xbc], 1)
    xbc = torch.nn.functional.silu(sum(full[:, j: j + n] * w["conv"][:, j] for j in range(taps)) + w["conv.b"])
    x, bm, cm = xbc[..., :inner].reshape(B, n, H, V), xbc[..., inner: inner + N], xbc[..., inner + N:]
    decay = torch.exp(-torch.exp(w["A_log"]) * dt)
    S, y = torch.zeros(B, H, N, V, dtype=F, device=DEV), torch.empty(B, n, H, V, dtype=F, device=DEV)
    xd = x * dt[..., None]
    for i in range(n):
        S = decay[:, i, :, None, None] * S + bm[:, i, None, :, None] * xd[:, i, :, None, :]
        y[:, i] = (cm[:, i, None, None, :] @ S)[:, :, 0]
    y = (y + w["D"][:, None] * x).reshape(B, n, inner) * torch.nn.functional.silu(z)
    return _unit(y) * w["norm"] @ w["o"].T


def _feed_forward(lay, w, g):
    if lay.ff == "dense":
        z = g @ w["up"].T
        if lay.dense_act == "polynorm":
            a = w["act"]
            z = a[0] * _unit(z) + a[1] * _unit(z ** 2) + a[2] * _unit(z ** 3) + a[3]
        else:
            z = torch.relu(z) ** 2
        return z @ w["down"].T
    score = torch.softmax(g @ w["router"].T, -1)
    pick = torch.topk(score + w["correction"], lay.top, -1).indices
    gate = torch.zeros_like(score).scatter(-1, pick, score.gather(-1, pick))
    y = torch.zeros_like(g)
    for e in range(lay.experts):
        rows = gate[..., e] > 0
        if bool(rows.any()):
            h = g[rows]
            h = torch.nn.functional.silu(h @ w[f"e{e}.gate"].T) * (h @ w[f"e{e}.up"].T)
            y[rows] += gate[..., e][rows][:, None] * (h @ w[f"e{e}.down"].T)
    return y


def lm_exact(case, tokens, at):
    """Logits [B, places, vocab] of the positions `at` [B, places] of tokens [B, n]."""
    cfg = lm_config(case["design"], case["size"])
    key = (case["design"], case["size"])
    if key not in _weights:
        _weights.clear()
        _weights[key] = lm_weights(*key)
    w = _weights[key]
    pos, latents = torch.arange(tokens.shape[1], device=DEV), {}
    x = _d(w["embed"][tokens])
    for i, lay in enumerate(cfg.layers):
        p = f"l{i}."
        mine = {n[len(p):]: _d(t) for n, t in w.items() if n.startswith(p)}
        sub = lambda s: {n[len(s):]: t for n, t in mine.items() if n.startswith(s)}  # noqa: E731
        u = _unit(x) * (1.0 + mine["norm1"])
        if "shift" in mine:
            u = u + (torch.cat([torch.zeros_like(u[:, :1]), u[:, :-1]], 1) - u) * mine["shift"]
        x = x + _unit(_mixer(lay, sub("mix."), u, pos, latents, i)) * (1.0 + mine["norm1b"])
        x = x + _unit(_feed_forward(lay, sub("mlp."), _unit(x) * (1.0 + mine["norm2"]))) * (1.0 + mine["norm2b"])
    x = torch.gather(x, 1, at[..., None].expand(-1, -1, x.shape[-1]))
    return (_unit(x) * (1.0 + _d(w["final.norm"]))) @ _d(w["head"]).T


def _lm_generate_exact(case, prompts):
    """The greedy text is the one that agrees with its own argmax everywhere: guesses are corrected until nothing changes."""
    lens, new = [len(p) for p in prompts], case["new"]
    at = torch.as_tensor([[n - 1 + i for i in range(new + 1)] for n in lens], device=DEV)
    text = [p.tolist() + [0] * new for p in prompts]
    for _ in range(new + 1):
        logits = lm_exact(case, _padded(text), at)
        picks = logits.argmax(-1)[:, :new].cpu().numpy()
        if all(t[n:] == r.tolist() for t, n, r in zip(text, lens, picks)):
            break
        text = [t[:n] + r.tolist() for t, n, r in zip(text, lens, picks)]
    return {"tokens": picks.astype(np.int32), "logits": logits[:, -1].cpu().numpy()}
