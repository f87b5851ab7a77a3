"""The work that is timed: what a serving program has this engine do, step by step.

A case is one call pattern on one model:

* ``decode``: one decode step of ``requests`` running requests (the replayed graph: model and sampling);
* ``prompt``: ``prompts`` new requests, their whole prompts in one step, a row of logits for each, and their release;
* ``mixed``: continuous batching's ordinary step, the first portion of new prompts beside ``requests`` running requests;
* ``generate``: prompts in, token ids out, through ``ContinuousBatchEngine``.

Lengths are ragged as they are in a running batch: request i of n holds ``context * (1 - i / (2 n))`` tokens, and
prompts shrink in the same way.  The models are the benchmark's layer sizes: Llama 3.2 1B whole, some of the layers
of 3B and 8B, and two designs whose mixers differ from the Llama's, at the benchmark's four layers: Rorevik (capped
attention beside a state-space mixer, a delta rule with a decay per channel) and Dokanex (attention through a latent,
attention within chunks).  Designs with routed experts are not here: which experts a token takes turns on the last
bit of a 16-bit activation where two scores are close, so two correct implementations differ there by more than any
tolerance on the logits could tell from a mistake.  Their attention, products and norms are the ones timed here.

Decoding requests are fed given tokens, so that a step's inputs do not hang on the choice of the step before it; the
step samples all the same.  Token ids are compared in float32 only: in bfloat16 the best two of 128,256 logits of a
random model change places by rounding in about one row of thirty.
"""
from __future__ import annotations

import math

import torch

VOCAB = 128256
GROWTH = 4096        # tokens that the running requests of a state may still generate

SIZES = {
    "1b": dict(width=2048, heads=32, kv_heads=8, head_dim=64, ff=8192, rope_factor=32.0, tied=True),
    "3b": dict(width=3072, heads=24, kv_heads=8, head_dim=128, ff=8192, rope_factor=32.0, tied=True),
    "8b": dict(width=4096, heads=32, kv_heads=8, head_dim=128, ff=14336, rope_factor=8.0, tied=False),
}
LLAMA_LAYERS = {"1b": 16, "3b": 8, "8b": 8}
LLAMA_EPS, LLAMA_THETA, LLAMA_ORIGINAL = 1e-5, 500000.0, 8192


def _case(kind, design, size, dtype="bfloat16", requests=0, context=0, prompts=0, tokens=0, new_tokens=0, name=None):
    case = dict(kind=kind, design=design, size=size, dtype=dtype, layers=LLAMA_LAYERS[size] if design == "llama" else 4,
                requests=requests, context=context, prompts=prompts, tokens=tokens, new_tokens=new_tokens)
    return dict(case, name=name) if name else case


def listed():
    return [
        # one user of a chat, early in a conversation: the smallest step, all latency
        _case("decode", "llama", "1b", requests=1, context=150, name="decode_one_user"),
        # a small batch with some thousand tokens each: the benchmark's headline step
        _case("decode", "llama", "1b", requests=8, context=4000, name="decode_batch_8"),
        # a full server: many requests of unlike lengths, keys and values outweigh the weights
        _case("decode", "llama", "1b", requests=64, context=4000, name="decode_batch_64"),
        # a short question: time to the first token
        _case("prompt", "llama", "1b", prompts=1, tokens=100, name="prompt_100"),
        # a full step of the default token budget: one document
        _case("prompt", "llama", "1b", prompts=1, tokens=2048, name="prompt_2048"),
        # continuous batching: a new request's first portion beside running requests, at 8B layer sizes
        _case("mixed", "llama", "8b", requests=31, context=2000, prompts=1, tokens=512, name="mixed_step_8b"),
        # the engine from end to end on the float32 path: eight short prompts of unlike length, greedy
        _case("generate", "llama", "1b", dtype="float32", prompts=8, tokens=60, new_tokens=16, name="generate_float32"),
        # three prompts in one step on the float32 path
        _case("prompt", "llama", "1b", dtype="float32", prompts=3, tokens=517, name="prompt_float32"),
        # a state-space mixer and a delta rule: states instead of growing caches
        _case("decode", "rorevik", "1b", requests=12, context=3000, name="rorevik_decode_12"),
        _case("prompt", "rorevik", "1b", prompts=1, tokens=2048, name="rorevik_prompt_2048"),
        # long documents on attention through a latent, whose cache is small enough for them
        _case("decode", "dokanex", "1b", requests=4, context=16000, name="dokanex_decode_long"),
        _case("prompt", "dokanex", "1b", prompts=2, tokens=1501, name="dokanex_prompt_2"),
    ]


def _spread(rng, low, high):
    """A whole number between ``low`` and ``high``, even over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    largest = max(work(c)["flops"] for c in listed() if c["dtype"] == "bfloat16")
    while True:
        kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "prompt", "mixed", "generate"])
        design = "llama" if kind == "generate" else rng.choice(["llama", "llama", "rorevik", "dokanex"])
        size = "1b" if kind == "generate" else rng.choice(["1b", "1b", "3b", "8b"] if design == "llama" else ["1b", "1b", "3b"])
        wide = kind == "generate" or (design == "llama" and size == "1b" and kind != "mixed" and rng.random() < 0.2)
        case = _case(kind, design, size, dtype="float32" if wide else "bfloat16")
        if kind in ("decode", "mixed"):
            case["requests"] = _spread(rng, 1, 64)
            case["context"] = _spread(rng, 16, min(16384, (8192 if wide else 131072) // case["requests"]))
        if kind == "prompt":
            case["prompts"] = _spread(rng, 1, 8)
            case["tokens"] = _spread(rng, 16, (1024 if wide else 3000) // case["prompts"])
        if kind == "mixed":
            case["prompts"], case["tokens"] = 1, _spread(rng, 16, 512)
        if kind == "generate":
            case["prompts"], case["tokens"], case["new_tokens"] = _spread(rng, 1, 8), _spread(rng, 8, 100), _spread(rng, 4, 16)
        if wide or work(case)["flops"] <= largest:
            return case


# ------------------------------------------------------------------------------------------------ models
def _llama_config(c):
    z = SIZES[c["size"]]
    return dict(
        architectures=["LlamaForCausalLM"], hidden_size=z["width"], intermediate_size=z["ff"], num_hidden_layers=c["layers"],
        num_attention_heads=z["heads"], num_key_value_heads=z["kv_heads"], head_dim=z["head_dim"], vocab_size=VOCAB,
        max_position_embeddings=131072, rms_norm_eps=LLAMA_EPS, rope_theta=LLAMA_THETA, tie_word_embeddings=z["tied"],
        rope_scaling=dict(rope_type="llama3", factor=z["rope_factor"], low_freq_factor=1.0, high_freq_factor=4.0,
                          original_max_position_embeddings=LLAMA_ORIGINAL), torch_dtype=c["dtype"])


def _rorevik_config(c):
    z, positions = SIZES[c["size"]], _longest(c)
    w, hd = z["width"], z["head_dim"]
    left = dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=hd, vdim=hd, scale=hd ** -0.5, softcap=30.0, rot={"base": 500000.0, "dims": hd // 2})
    right = dict(heads=w // 64, vdim=64, state=128, groups=1, norm_groups=1, conv=4)
    delta = dict(heads=w // 128, kv_heads=w // 128, dim=128, vdim=128, conv=4, decay_rank=128, gate_rank=128)
    mlp = {"kind": "dense", "ff": z["ff"], "limit": 7.0}
    both = {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0}, "mlp": mlp}
    return {"architecture": "Rorevik", "vocab": VOCAB, "width": w, "max_positions": positions, "embedding": {"scale": w ** 0.5},
            "norm": {"eps": 1e-5}, "layers": [{"type": "channel_delta", "mixer": delta, "mlp": mlp} if i % 3 == 2 else both for i in range(c["layers"])]}


def _dokanex_config(c):
    z = SIZES[c["size"]]
    w, hd = z["width"], z["head_dim"]
    latent = dict(heads=16, dim=128, rot_dim=64, vdim=w // 16, q_rank=w * 3 // 8, kv_rank=192, scale=192 ** -0.5,
                  rot={"base": 500000.0, "dims": 64, "scaling": {"factor": 8.0, "original": 1024, "fast": 32.0, "slow": 1.0}})
    chunk = dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=hd, vdim=hd, scale=hd ** -0.5, softcap=30.0, mask={"size": 1024})
    layers = []
    for i in range(c["layers"]):
        mixer = latent if i % 4 < 2 else chunk if i % 4 == 2 else dict(chunk, kv_from=i - 1)
        layers.append({"type": "latent_attention" if i % 4 < 2 else "attention", "mixer": mixer, "mlp": {"kind": "dense", "ff": z["ff"]}})
    return {"architecture": "Dokanex", "vocab": VOCAB, "width": w, "embedding": {"scale": w ** 0.5}, "norm": {"eps": 1e-5},
            "logit_softcap": 30.0, "layers": layers}


def _config(c):
    return {"llama": _llama_config, "rorevik": _rorevik_config, "dokanex": _dokanex_config}[c["design"]](c)


def _shapes(c):
    """The tensors of the case's model: name -> (shape, what kind of number it holds)."""
    cfg, w, ff = _config(c), SIZES[c["size"]]["width"], SIZES[c["size"]]["ff"]
    out = {}

    def add(prefix, kind="matrix", **named):
        for n, s in named.items():
            out[prefix + n.replace("__", ".")] = (s if isinstance(s, tuple) else (s,), kind)

    if c["design"] == "llama":
        q, kv = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
        add("model.", embed_tokens__weight=(VOCAB, w))
        for i in range(c["layers"]):
            p = f"model.layers.{i}."
            add(p, "norm", input_layernorm__weight=w, post_attention_layernorm__weight=w)
            add(p, self_attn__q_proj__weight=(q, w), self_attn__k_proj__weight=(kv, w), self_attn__v_proj__weight=(kv, w),
                self_attn__o_proj__weight=(w, q), mlp__gate_proj__weight=(ff, w), mlp__up_proj__weight=(ff, w), mlp__down_proj__weight=(w, ff))
        add("model.", "norm", norm__weight=w)
        if not cfg["tie_word_embeddings"]:
            add("", lm_head__weight=(VOCAB, w))
        return out
    add("", embed=(VOCAB, w))
    add("", "norm", final__norm=w)
    if c["design"] == "rorevik":
        add("", pos=(cfg["max_positions"], w), head=(VOCAB, w))
        add("", "norm", embed__norm=w)
    for i, layer in enumerate(cfg["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        add(p, "norm", norm1=w, norm2=w)
        add(p + "mlp.", gate=(ff, w), up=(ff, w), down=(w, ff))
        if c["design"] == "rorevik":
            add(p + "mlp.", "small", gate__b=ff, up__b=ff, down__b=w)
        if layer["type"] == "parallel":
            a, s = m["left"], m["right"]
            inner, mixed = s["heads"] * s["vdim"], s["heads"] * s["vdim"] + 2 * s["groups"] * s["state"]
            add(p + "mix.left.", q=(a["heads"] * a["dim"], w), k=(a["kv_heads"] * a["dim"], w), v=(a["kv_heads"] * a["vdim"], w), o=(w, a["heads"] * a["vdim"]))
            add(p + "mix.right.", **{"in": (inner + mixed + s["heads"], w), "o": (w, inner)})
            add(p + "mix.right.", "taps", conv=(mixed, s["conv"]))
            add(p + "mix.right.", "small", conv__b=mixed)
            add(p + "mix.right.", "step", dt_bias=s["heads"])
            add(p + "mix.right.", "rate", A_log=s["heads"])
            add(p + "mix.right.", "norm", D=s["heads"], norm=inner)
        elif layer["type"] == "channel_delta":
            k, v, h = m["kv_heads"] * m["dim"], m["heads"] * m["vdim"], m["heads"]
            add(p + "mix.", q=(k, w), k=(k, w), v=(v, w), b=(h, w), a1=(m["decay_rank"], w), a2=(h * m["dim"], m["decay_rank"]),
                g1=(m["gate_rank"], w), g2=(v, m["gate_rank"]), o=(w, v))
            add(p + "mix.", "taps", q__conv=(k, m["conv"]), k__conv=(k, m["conv"]), v__conv=(v, m["conv"]))
            add(p + "mix.", "step", dt_bias=h * m["dim"])
            add(p + "mix.", "rate", A_log=h)
            add(p + "mix.", "norm", norm=m["vdim"])
        elif layer["type"] == "latent_attention":
            h, r = m["heads"], m["kv_rank"]
            add(p + "mix.", dq=(m["q_rank"], w), uq=(h * (m["dim"] + m["rot_dim"]), m["q_rank"]), dkv=(r + m["rot_dim"], w),
                uk=(h * m["dim"], r), uv=(h * m["vdim"], r), o=(w, h * m["vdim"]))
            add(p + "mix.", "norm", dq__norm=m["q_rank"], dkv__norm=r)
        else:
            add(p + "mix.", q=(m["heads"] * m["dim"], w), g=(m["heads"], w), o=(w, m["heads"] * m["vdim"]))
            add(p + "mix.", "one", sink=m["heads"])
            if "kv_from" not in m:
                add(p + "mix.", k=(m["kv_heads"] * m["dim"], w), v=(m["kv_heads"] * m["vdim"], w))
    return out


def _tensors(c, g):
    """Random weights with the spreads that such tensors have: matrices N(0, 0.02) at a width of 2,048 and smaller
    by the root of the width beyond it, norms around 1, decays and step sizes over the ranges that state-space and
    delta-rule mixers start from."""
    dtype = getattr(torch, c["dtype"])
    matrix = 0.02 * math.sqrt(2048 / SIZES[c["size"]]["width"])
    out = {}
    for name, (shape, kind) in sorted(_shapes(c).items()):
        if kind in ("norm", "rate", "step"):
            u = torch.rand(shape, generator=g, device="cuda")
            t = 0.5 + u if kind == "norm" else torch.log(1.0 + 15.0 * u) if kind == "rate" else torch.log(torch.expm1(torch.exp(math.log(1e-3) + u * math.log(1e2))))
        else:
            t = torch.randn(shape, generator=g, device="cuda") * {"matrix": matrix, "small": 0.1, "taps": 0.5, "one": 1.0}[kind]
        out[name] = t.to(dtype)
    return out


# ------------------------------------------------------------------------------------------------ inputs
def _ragged(n, longest):
    return [max(1, longest - longest * i // (2 * n)) for i in range(n)]


def _longest(c):
    return max(c["context"] + GROWTH + 1 if c["requests"] else 0, c["tokens"] + c["new_tokens"] + 1)


def _inputs(c, seed):
    """(weights, what the running requests hold, the tokens they are fed from then on, the prompts)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    weights = _tensors(c, g)
    ids = lambda *shape: torch.randint(0, VOCAB, shape, generator=g, device="cuda").tolist()
    held = [ids(n) for n in _ragged(c["requests"], c["context"])]
    fed = ids(GROWTH, c["requests"]) if c["requests"] else []
    return weights, held, fed, [ids(n) for n in _ragged(c["prompts"], c["tokens"])]


def prepare(case, seed):
    from photon_infer_amd import ContinuousBatchEngine, EngineOptions, ModelRunner, StepEntry
    from photon_infer_amd.registry import config_from_dict

    weights, held, fed, prompts = _inputs(case, seed)
    room = sum(len(h) + GROWTH + 16 for h in held) + sum(len(p) + case["new_tokens"] + 16 for p in prompts)
    options = EngineOptions(dtype=case["dtype"], max_batch=case["requests"] + case["prompts"], max_cache_tokens=room,
                            max_model_len=_longest(case), keep_logits=True)
    runner = ModelRunner(None, options, config=config_from_dict(_config(case)), tensors=weights)
    running = [f"running {i}" for i in range(len(held))]
    for rid, tokens in zip(running, held):
        runner.admit(rid)
        for at in range(0, len(tokens), 2048):
            runner.step([StepEntry(rid, tokens[at:at + 2048])])
    state = dict(case=case, runner=runner, running=running, fed=fed, at=0, prompts=prompts)
    if case["kind"] == "decode":           # a server's graph for this batch is there before the step in question
        run(state)
    if case["kind"] == "generate":
        state["engine"] = ContinuousBatchEngine(None, runner=runner)
    return state


def run(state):
    from photon_infer_amd import StepEntry

    case, runner = state["case"], state["runner"]
    if case["kind"] == "generate":
        return [torch.tensor(ids) for ids in state["engine"].generate(state["prompts"], max_new_tokens=case["new_tokens"], ignore_eos=True)]
    entries = []
    if state["running"]:
        entries = [StepEntry(rid, [tok], [0]) for rid, tok in zip(state["running"], state["fed"][state["at"]])]
        state["at"] += 1
    if case["kind"] == "decode":
        none = [0.0] * len(entries)
        ids = runner.decode_step(entries, none, none)
        return {"logits": runner.decode_logits, "ids": ids} if case["dtype"] == "float32" else {"logits": runner.decode_logits}
    fresh = [f"new {i}" for i in range(len(state["prompts"]))]
    for rid in fresh:
        runner.admit(rid)
    logits = runner.step([StepEntry(rid, p, [len(p) - 1]) for rid, p in zip(fresh, state["prompts"])] + entries)
    for rid in fresh:
        runner.release(rid)
    return logits


# ------------------------------------------------------------------------------------------------ what a pass needs
def _per_token(c):
    """(weights that every token is multiplied with, over all layers; bytes of keys, values or latents it leaves; pair flops per
    seen key; flops of the recurrences per token; bytes of the states a request holds)."""
    cfg, e = _config(c), 2 if c["dtype"] == "bfloat16" else 4
    matrices = sum(math.prod(s) for n, (s, k) in _shapes(c).items() if k == "matrix" and len(s) == 2 and s[0] != VOCAB and n != "pos")
    if c["design"] == "llama":
        h, g, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        return matrices, c["layers"] * 2 * g * d * e, c["layers"] * 4 * h * d, 0, 0
    left, pair, flops, states = 0, 0, 0, 0
    for layer in cfg["layers"]:
        m = layer["mixer"]
        if layer["type"] == "parallel":
            left, pair = left + 2 * m["left"]["kv_heads"] * m["left"]["dim"] * e, pair + 4 * m["left"]["heads"] * m["left"]["dim"]
            size = m["right"]["heads"] * m["right"]["state"] * m["right"]["vdim"]
            flops, states = flops + 5 * size, states + 4 * size
        elif layer["type"] == "channel_delta":
            size = m["heads"] * m["dim"] * m["vdim"]
            flops, states = flops + 7 * size, states + 4 * size
        elif layer["type"] == "latent_attention":
            left, pair = left + (m["kv_rank"] + m["rot_dim"]) * e, pair + 2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
        else:       # attention within chunks: counted by the chunk's share in work()
            left += 0 if "kv_from" in m else 2 * m["kv_heads"] * m["dim"] * e
    return matrices, left, pair, flops, states


def work(case):
    c, e = case, 2 if case["dtype"] == "bfloat16" else 4
    width = SIZES[c["size"]]["width"]
    matrices, left, pair, recurrence, states = _per_token(c)
    fed = [(n, 1) for n in _ragged(c["requests"], c["context"])] + [(0, n) for n in _ragged(c["prompts"], c["tokens"])]
    steps = [fed]
    if c["kind"] == "generate":
        steps += [[(n + i, 1) for n in _ragged(c["prompts"], c["tokens"])] for i in range(c["new_tokens"] - 1)]
    nbytes = flops = 0.0
    for step in steps:
        nbytes += (matrices + VOCAB * width) * e
        for before, new in step:
            seen = new * before + new * (new + 1) / 2
            flops += 2.0 * new * matrices + new * recurrence + pair * seen + 2.0 * VOCAB * width
            nbytes += (before + new) * left + new * width * e + VOCAB * 4 + states * (2 if before else 1)
            if c["design"] == "dokanex":
                z = SIZES[c["size"]]
                lengths = [(before + new) % 1024 or 1024] if new == 1 else [1024] * (new // 1024) + [new % 1024]
                flops += 2 * 4.0 * z["heads"] * z["head_dim"] * sum(n if new == 1 else n * (n + 1) / 2 for n in lengths)
                if new == 1:        # of the keys and values only the chunk's are read
                    nbytes -= (before + new - lengths[0]) * 2 * z["kv_heads"] * z["head_dim"] * e
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # against 64 bits the float32 path is off by 9e-6 (sixteen layers, a few hundred tokens) and the bfloat16 path by
    # 0.019 (the Llama's sixteen layers) or 0.005 (four layers of the others); "max" is five such deviations and more
    if case["dtype"] == "float32":
        return {"rel": 4e-5, "max": 1e-3, "differ": 0.01}
    return {"rel": 0.03 if case["design"] == "llama" else 0.02, "max": 0.3}


# ------------------------------------------------------------------------------------------------ in 64 bits
def _norm(x, w, eps):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, angles, mult=1.0, halves=False):
    """x [T, heads, dim]: the first 2 * angles.shape[1] features turned in pairs, neighbours or (``halves``) a half apart."""
    n = angles.shape[1]
    c, s = torch.cos(angles)[:, None] * mult, torch.sin(angles)[:, None] * mult
    y = x.clone()
    a, b = (slice(0, n), slice(n, 2 * n)) if halves else (slice(0, 2 * n, 2), slice(1, 2 * n, 2))
    y[..., a], y[..., b] = x[..., a] * c - x[..., b] * s, x[..., a] * s + x[..., b] * c
    return y


def _attend(q, k, v, scale, cap=None, chunk=None, sink=None):
    """One sequence, causal: q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H, dv]."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    at, out = torch.arange(T, device=q.device), []
    kt, vt = k.permute(1, 2, 0), v.permute(1, 0, 2)
    for i in range(0, T, 512):
        n, end = min(512, T - i), min(T, i + 512)
        lo = 0 if not chunk else i // chunk * chunk
        qi = q[i:end].reshape(n, G, H // G, -1).permute(1, 2, 0, 3).reshape(G, H // G * n, -1)
        s = (qi.contiguous() @ kt[..., lo:end].contiguous()).view(H, n, end - lo).mul_(scale)
        if cap:
            s = s.div_(cap).tanh_().mul_(cap)
        hidden = at[None, lo:end] > at[i:end, None]
        if chunk:
            hidden = hidden | (at[None, lo:end] // chunk != at[i:end, None] // chunk)
        s.masked_fill_(hidden, -math.inf)
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink.view(H, 1, 1))
        p = s.sub_(top).exp_()
        den = p.sum(-1, keepdim=True)
        if sink is not None:
            den = den + torch.exp(sink.view(H, 1, 1) - top)
        o = (p.view(G, -1, end - lo) @ vt[:, lo:end].contiguous()).view(H, n, -1) / den
        out.append(o.transpose(0, 1))
    return torch.cat(out)


def _conv(seqs, w, b=None):
    out = []
    for u in seqs:
        taps = w.shape[1]
        padded = torch.cat([u.new_zeros(taps - 1, u.shape[1]), u])
        y = sum(padded[j:j + u.shape[0]] * w[:, j] for j in range(taps))
        out.append(_silu(y if b is None else y + b))
    return out


def _side_by_side(seqs):
    return torch.nn.utils.rnn.pad_sequence(seqs, batch_first=True)


def _back(padded, seqs):
    return [padded[i, :len(s)] for i, s in enumerate(seqs)]


def _state_space(seqs, m, W):
    H, P, N, inner = m["heads"], m["vdim"], m["state"], m["heads"] * m["vdim"]
    proj = [h @ W("in").T for h in seqs]
    xbc = _conv([p[:, inner:2 * inner + 2 * N] for p in proj], W("conv"), W("conv.b"))
    dt = _side_by_side([torch.nn.functional.softplus(p[:, 2 * inner + 2 * N:] + W("dt_bias")) for p in proj])       # [R, T, H]
    u = _side_by_side(xbc)
    x, B, C = u[..., :inner].unflatten(-1, (H, P)), u[..., inner:inner + N], u[..., inner + N:]                     # one group
    keep = torch.exp(-torch.exp(W("A_log")) * dt)
    S, y = u.new_zeros(u.shape[0], H, P, N), torch.empty_like(x)
    for t in range(u.shape[1]):
        S = S * keep[:, t, :, None, None] + (dt[:, t, :, None] * x[:, t])[..., None] * B[:, t, None, None, :]
        y[:, t] = torch.matmul(S, C[:, t, None, :, None])[..., 0]
    y = (y + W("D")[:, None] * x).flatten(-2)
    out = [a * _silu(p[:, :inner]) for a, p in zip(_back(y, proj), proj)]
    return [_norm(a, W("norm"), 1e-5) @ W("o").T for a in out]


def _channel_delta(seqs, m, W):
    H, d, dv = m["heads"], m["dim"], m["vdim"]
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    q, k, v = (_side_by_side(_conv([h @ W(n).T for h in seqs], W(n + ".conv"))).unflatten(-1, (H, -1)) for n in "qkv")
    q, k = unit(q) * d ** -0.5, unit(k)
    beta = _side_by_side([torch.sigmoid(h @ W("b").T) for h in seqs])
    a = _side_by_side([torch.nn.functional.softplus(h @ W("a1").T @ W("a2").T + W("dt_bias")) for h in seqs]).unflatten(-1, (H, d))
    decay = torch.exp(-torch.exp(W("A_log"))[:, None] * a)
    S, o = q.new_zeros(q.shape[0], H, d, dv), torch.empty_like(v)
    for t in range(q.shape[1]):
        S = S * decay[:, t, ..., None]
        u = beta[:, t, :, None] * (v[:, t] - torch.matmul(k[:, t, :, None, :], S)[..., 0, :])
        S = S + k[:, t, ..., None] * u[..., None, :]
        o[:, t] = torch.matmul(q[:, t, :, None, :], S)[..., 0, :]
    out = []
    for one, h in zip(_back(_norm(o, W("norm"), 1e-5), seqs), seqs):
        out.append((one * torch.sigmoid(h @ W("g1").T @ W("g2").T).unflatten(-1, (H, dv))).flatten(-2) @ W("o").T)
    return out


def _ramped(dims, rot):
    """The rotation's frequencies, slowed by a ramp over the pairs, and the factor on cosines and sines."""
    f, s = [rot["base"] ** (-2.0 * i / dims) for i in range(dims // 2)], rot["scaling"]
    where = lambda turns: dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))
    lo, hi = max(math.floor(where(s["fast"])), 0), min(math.ceil(where(s["slow"])), dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [a / s["factor"] * r + a * (1.0 - r) for a, r in zip(f, ramp)], 0.1 * math.log(s["factor"]) + 1.0


def _llama_frequencies(size):
    z, out = SIZES[size], []
    for j in range(z["head_dim"] // 2):
        f = LLAMA_THETA ** (-2.0 * j / z["head_dim"])
        turns = LLAMA_ORIGINAL * f / (2.0 * math.pi)
        s = min(max((turns - 1.0) / 3.0, 0.0), 1.0)
        out.append((1.0 - s) * f / z["rope_factor"] + s * f)
    return out


def _forward(c, weights, sequences):
    """Logits [sequences, vocabulary] of every sequence's last token."""
    cfg, z = _config(c), SIZES[c["size"]]
    w, hd, H, G = z["width"], z["head_dim"], z["heads"], z["kv_heads"]
    made = {}

    def W(name):            # a layer's tensors in 64 bits, kept until the next layer
        if name not in made:
            made[name] = weights[name].double()
        return made[name]

    ids = [torch.tensor(s, device="cuda") for s in sequences]
    at = [torch.arange(len(s), device="cuda", dtype=torch.float64) for s in ids]
    angles = lambda p, f: p[:, None] * torch.tensor(f, device="cuda", dtype=torch.float64)
    llama = c["design"] == "llama"
    table = weights["model.embed_tokens.weight" if llama else "embed"]
    x = [table[s].double() for s in ids]
    if llama:
        # the model's definition has frequencies and angles in 32 bits
        f32 = torch.tensor(_llama_frequencies(c["size"]), dtype=torch.float64).float().cuda()
        turns = [(p.float()[:, None] * f32).double() for p in at]
    else:
        x = [a * cfg["embedding"]["scale"] for a in x]
    if c["design"] == "rorevik":
        x = [_norm(a + weights["pos"][:len(a)].double(), W("embed.norm"), 1e-5) for a in x]
    kept = {}
    for i in range(c["layers"]):
        made.clear()
        p = f"model.layers.{i}." if llama else f"l{i}."
        L = lambda n, p=p: W(p + n)
        h = [_norm(a, L("input_layernorm.weight" if llama else "norm1"), 1e-5) for a in x]
        kind = "llama" if llama else cfg["layers"][i]["type"]
        m = None if llama else cfg["layers"][i]["mixer"]
        heads = lambda a, n: a.unflatten(-1, (n, -1))
        if kind == "llama":
            o = []
            for a, t in zip(h, turns):
                q, k, v = (heads(a @ L(f"self_attn.{n}_proj.weight").T, s) for n, s in (("q", H), ("k", G), ("v", G)))
                o.append(_attend(_turn(q, t, halves=True), _turn(k, t, halves=True), v, hd ** -0.5).flatten(1) @ L("self_attn.o_proj.weight").T)
        elif kind == "parallel":
            f = [500000.0 ** (-2.0 * j / (hd // 2)) for j in range(hd // 4)]
            o = _state_space(h, m["right"], lambda n: L("mix.right." + n))
            for r, (a, t) in enumerate(zip(h, at)):
                q, k, v = (heads(a @ L("mix.left." + n).T, s) for n, s in (("q", H), ("k", G), ("v", G)))
                t = angles(t, f)
                o[r] = o[r] + _attend(_turn(q, t), _turn(k, t), v, hd ** -0.5, cap=30.0).flatten(1) @ L("mix.left.o").T
        elif kind == "channel_delta":
            o = _channel_delta(h, m, lambda n: L("mix." + n))
        elif kind == "latent_attention":
            n, d, rank = m["heads"], m["dim"], m["kv_rank"]
            f, mult = _ramped(m["rot_dim"], m["rot"])
            o = []
            for a, t in zip(h, at):
                t = angles(t, f)
                q = heads(_norm(a @ L("mix.dq").T, L("mix.dq.norm"), 1e-5) @ L("mix.uq").T, n)
                down = a @ L("mix.dkv").T
                latent, rot = _norm(down[:, :rank], L("mix.dkv.norm"), 1e-5), _turn(down[:, None, rank:], t, mult)
                q = torch.cat([q[..., :d], _turn(q[..., d:], t, mult)], -1)
                k = torch.cat([heads(latent @ L("mix.uk").T, n), rot.expand(-1, n, -1)], -1)
                o.append(_attend(q, k, heads(latent @ L("mix.uv").T, n), m["scale"]).flatten(1) @ L("mix.o").T)
        else:
            if "kv_from" not in m:
                kept = {r: (_norm(heads(a @ L("mix.k").T, G), None, 1e-5), heads(a @ L("mix.v").T, G)) for r, a in enumerate(h)}
            o = []
            for r, a in enumerate(h):
                q = _norm(heads(a @ L("mix.q").T, H), None, 1e-5)
                y = _attend(q, *kept[r], m["scale"], cap=30.0, chunk=1024, sink=L("mix.sink"))
                o.append((y * torch.sigmoid(a @ L("mix.g").T)[..., None]).flatten(1) @ L("mix.o").T)
        x = [a + b for a, b in zip(x, o)]
        del h, o
        for r, a in enumerate(x):
            y = _norm(a, L("post_attention_layernorm.weight" if llama else "norm2"), 1e-5)
            names = [f"mlp.{n}_proj.weight" if llama else f"mlp.{n}" for n in ("gate", "up", "down")]
            g, u = y @ L(names[0]).T, y @ L(names[1]).T
            if c["design"] == "rorevik":
                g, u = torch.clamp(g + L("mlp.gate.b"), max=7.0), torch.clamp(u + L("mlp.up.b"), min=-7.0, max=7.0)
                x[r] = a + (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ L(names[2]).T + L("mlp.down.b")
            else:
                x[r] = a + (_silu(g) * u) @ L(names[2]).T
    made.clear()
    last = torch.stack([a[-1] for a in x])
    del x
    last = _norm(last, W("model.norm.weight" if llama else "final.norm"), 1e-5)
    head = weights["lm_head.weight"] if llama and not z["tied"] else weights["head"] if c["design"] == "rorevik" else table
    logits = last @ head.double().T
    return 30.0 * torch.tanh(logits / 30.0) if c["design"] == "dokanex" else logits


def exact(case, seed):
    weights, held, fed, prompts = _inputs(case, seed)
    if case["kind"] == "generate":          # token ids only: none of them is a rounded number
        return None
    if case["kind"] == "prompt":
        return _forward(case, weights, prompts)
    # a decode state has taken its first step when it is handed over
    steps = 2 if case["kind"] == "decode" else 1
    running = [h + [row[i] for row in fed[:steps]] for i, h in enumerate(held)]
    matrices = _per_token(case)[0]
    if 2.0 * matrices * sum(len(s) for s in running) > 6e14:        # over some 15 seconds in 64 bits
        return None
    if case["kind"] == "mixed":
        return _forward(case, weights, prompts + running)
    logits = _forward(case, weights, running)
    return {"logits": logits, "ids": None} if case["dtype"] == "float32" else {"logits": logits}
