"""Workloads that stand for the use of this engine, for timing and for comparing results.

A case names a model shape, how the model is used and the sizes of that use. The uses:

- "prompt": prompts come in as one step, the logits behind each prompt's last token are wanted, the requests end
  (what scoring a prompt, or the first token of an answer, costs).
- "decode": requests that already hold a context take ``steps`` single-token steps, launched the way the engine and
  the benchmark launch them (the next step before the last one is collected).
- "job": the two together from start to end: prompts in, ``steps`` tokens decoded, the requests end.
- "mixed": continuous batching: ``batch`` requests decode while the portions of one new prompt come in beside them.

The tokens of every step are given (as in a trace replay), so that two implementations go through the same contexts,
and every step's logits are returned. The shapes are those of the benchmark (``bench.py``) and of the tests; the
weights are random, drawn by the package's own law for every tensor.
"""
import math
import re

import torch

DEVICE = "cuda:0" if torch.cuda.is_available() else "cpu"
F64 = torch.float64


# ------------------------------------------------------------------------------------------- model shapes
def _qwen(layers, width, heads, kv_heads, ff, tied=False, vocab=151936, head_dim=128, longest=40960):
    return {"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "vocab_size": vocab, "hidden_size": width,
            "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": kv_heads,
            "head_dim": head_dim, "intermediate_size": ff, "max_position_embeddings": longest, "rms_norm_eps": 1e-6,
            "rope_theta": 1e6, "tie_word_embeddings": tied}


def _kofipel(layers, width):
    heads, ff = width // 128, {2048: 8192, 4096: 12288}[width]
    mix = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128}
    mlp = {"kind": "dense", "ff": ff}
    delta = {"type": "channel_delta", "mlp": mlp, "mixer": dict(mix, conv=4, rank=64)}
    attn = {"type": "attention", "mlp": mlp,
            "mixer": dict(mix, scale=128 ** -0.5, softcap=30.0, mask={"size": 1024, "keep_first": 64},
                          rot={"base": 1e6, "dims": 128})}
    return {"architecture": "Kofipel", "vocab": 32000, "width": width, "norm": {"eps": 1e-6}, "canon": {"taps": 4},
            "token_side": {"dim": 32}, "layers": [attn if i % 4 == 3 else delta for i in range(layers)]}


def _rupezen(layers, width):
    heads, ff = width // 128, {2048: 8192, 4096: 12288}[width]
    layer = {"type": "attention",
             "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 64, "vdim": 128, "diff": 0.5, "scale": 64 ** -0.5,
                       "mask": {"size": 4096}, "rot": {"base": 1e6, "dims": 32}},
             "mlp": {"kind": "moe", "expert": {"ff": ff // 4},
                     "router": {"experts": 32, "top": 4, "groups": {"count": 4, "keep": 2}}}}
    mid = layers // 2
    return {"architecture": "Rupezen", "vocab": 32000, "width": width, "norm": {"eps": 1e-6}, "residual_mult": 0.5,
            "loop": {"start": mid - 1, "stop": mid + 1, "times": 2}, "layers": [layer] * layers}


_STRETCH = {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}


def _safilorn(layers, width):
    heads, ff = width // 128, {2048: 8192, 4096: 12288}[width]
    latent = {"type": "latent_attention",
              "mixer": {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 1536, "kv_rank": 512,
                        "scale": 192 ** -0.5, "rot": {"base": 1e6, "dims": 64, "scaling": _STRETCH}}}
    gla = {"type": "gla", "mixer": {"heads": heads, "dim": 128, "vdim": 128, "tau": 16.0, "rank": 64}}
    dense = {"kind": "dense", "ff": ff}
    moe = {"kind": "moe", "expert": {"ff": ff // 4, "limit": 7.0}, "router": {"experts": 32, "top": 4}}
    return {"architecture": "Safilorn", "vocab": 32000, "width": width, "norm": {"eps": 1e-6},
            "embedding": {"scale": width ** 0.5},
            "layers": [dict(latent if i % 4 == 3 else gla, mlp=moe if i % 2 else dense) for i in range(layers)]}


def _fefulorn(layers, width):
    heads, ff = width // 128, {2048: 8192, 4096: 12288}[width]
    ssm = {"type": "mamba2", "mixer": {"heads": width // 64, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}}
    latent = {"type": "latent_attention",
              "mixer": {"heads": heads, "dim": 128, "vdim": 128, "q_rank": 1536, "kv_rank": 512, "scale": 128 ** -0.5,
                        "mask": {"size": 4096}}}
    attn = {"type": "attention",
            "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                      "mask": {"size": 1024}, "rot": {"base": 1e6, "dims": 64, "scaling": {"factor": 2.0}}, "v_mix": True}}
    moe = {"kind": "moe", "expert": {"ff": ff // 4, "limit": 7.0},
           "router": {"experts": 32, "top": 4, "groups": {"count": 4, "keep": 2}}, "shared": {"ff": ff // 4, "limit": 7.0}}
    kinds = [ssm, ssm, ssm, latent, ssm, ssm, ssm, attn]
    return {"architecture": "Fefulorn", "vocab": 32000, "width": width, "norm": {"eps": 1e-6},
            "embedding": {"scale": width ** 0.5}, "logit_scale": 1.0,
            "layers": [dict(kinds[i % 8], mlp=moe) for i in range(layers)]}


def _mepolix(layers, width):
    heads, ff = width // 128, {2048: 8192, 4096: 12288}[width]
    mix = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128}
    mlp = {"kind": "dense", "ff": ff}
    delta = {"type": "delta", "mlp": mlp, "mixer": dict(mix, conv=4)}
    both = {"type": "parallel", "mlp": mlp,
            "mixer": {"left": dict(mix, scale=128 ** -0.5, rot={"base": 1e6, "dims": 128, "scaling": _STRETCH}),
                      "right": {"width": width, "blocks": width // 128, "conv": 4}, "left_scale": 0.8, "right_scale": 1.2}}
    return {"architecture": "Mepolix", "vocab": 32000, "width": width, "norm": {"eps": 1e-6}, "logit_softcap": 30.0,
            "layers": [both if i % 4 == 3 else delta for i in range(layers)]}


def _mapalorn(layers, width):
    heads, ff = width // 128, {2048: 8192, 4096: 12288}[width]
    latent = {"type": "latent_attention",
              "mixer": {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
                        "rot": {"base": 1e6, "dims": 64}}}
    attn = {"type": "attention",
            "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                      "rot": {"base": 1e6, "dims": 128}}}
    moe = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 32, "top": 4}, "shared": {"ff": ff // 4}}
    kinds = [latent, latent, latent, attn]
    return {"architecture": "Mapalorn", "vocab": 32000, "width": width, "norm": {"eps": 1e-6},
            "layers": [dict(kinds[i % 4], mlp=moe if i else {"kind": "dense", "ff": ff, "limit": 7.0}) for i in range(layers)],
            "loop": {"start": 2, "stop": 3, "times": 2}}


_DESIGNS = {"kofipel": _kofipel, "rupezen": _rupezen, "safilorn": _safilorn, "fefulorn": _fefulorn,
            "mepolix": _mepolix, "mapalorn": _mapalorn}
_QWEN = {"qwen3_small": dict(width=512, heads=8, kv_heads=2, ff=1536, vocab=4096, head_dim=64),
         "qwen3_4b": dict(width=2560, heads=32, kv_heads=8, ff=9728, tied=True),
         "qwen3_8b": dict(width=4096, heads=32, kv_heads=8, ff=12288)}


def _config(case):
    """config.json of the case's model."""
    if case["model"] in _QWEN:
        return _qwen(case["layers"], **_QWEN[case["model"]])
    return _DESIGNS[case["model"]](case["layers"], case["width"])


def _runs(raw):
    """The layers' numbers in the order they run."""
    if "num_hidden_layers" in raw:
        return list(range(raw["num_hidden_layers"]))
    n, loop = len(raw["layers"]), raw.get("loop")
    if not loop:
        return list(range(n))
    return list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], n))


def _case(name, model, use, layers, batch, prompt, steps=0, width=0, dtype="bfloat16", spread=0.0, portion=0):
    case = {"model": model, "width": width, "layers": layers, "use": use, "dtype": dtype, "batch": batch,
            "prompt": prompt, "spread": spread, "steps": steps, "portion": portion}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest calls: one request on a small model, where launches and the host count
        _case("small_decode_b1", "qwen3_small", "decode", 4, 1, 60, steps=8),
        # the benchmark's headline: eight requests over contexts of 2,048 tokens
        _case("8b_decode_b8", "qwen3_8b", "decode", 36, 8, 2048, steps=4),
        # many requests of uneven lengths (a rollout's full batch)
        _case("8b_decode_b64", "qwen3_8b", "decode", 12, 64, 500, steps=4, spread=0.4),
        # the benchmark's prompt
        _case("8b_prompt_2048", "qwen3_8b", "prompt", 36, 1, 2048),
        # continuous batching: requests decode while a newcomer's prompt comes in by portions
        _case("4b_mixed", "qwen3_4b", "mixed", 36, 24, 450, steps=3, spread=0.5, portion=512),
        # the 32-bit mode, which checks are run in
        _case("8b_fp32_job", "qwen3_8b", "job", 4, 3, 211, steps=4, dtype="float32", spread=0.2),
        # the other designs, from prompt to the last token: one long prompt, several uneven ones, a full batch of short ones
        _case("kofipel_job_b1", "kofipel", "job", 8, 1, 2048, steps=6, width=4096),
        _case("mepolix_job_b4", "mepolix", "job", 8, 4, 701, steps=6, width=4096, spread=0.3),
        _case("safilorn_job_b1", "safilorn", "job", 8, 1, 2333, steps=8, width=2048),
        _case("fefulorn_job_b8", "fefulorn", "job", 8, 8, 250, steps=4, width=4096, spread=0.3),
        _case("rupezen_job_b64", "rupezen", "job", 6, 64, 33, steps=4, width=2048, spread=0.3),
        _case("mapalorn_job_b4", "mapalorn", "job", 7, 4, 777, steps=6, width=4096, spread=0.3),
    ]


def _cost(case):
    """About what a pass takes, in milliseconds at rates that ordinary steps reach."""
    w = work(case)
    return w["bytes"] / 4e9 + w["flops"] / 5e11


def draw(rng):
    """Another case of the same kinds: any of the models, any use, sizes spread evenly over their logarithms."""
    most = 0.6 * max(_cost(c) for c in listed())
    while True:
        case = _any(rng)
        if _cost(case) <= most:
            return case


def _any(rng):
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    spread = rng.choice([0.0, 0.2, 0.5])
    kind = rng.randrange(10)
    if kind == 0:
        return _case(None, "qwen3_small", "decode", rng.randint(2, 6), between(1, 16), between(5, 900), rng.randint(4, 10), spread=spread)
    if kind == 1:
        batch = between(1, 64)
        return _case(None, "qwen3_8b", "decode", rng.randint(6, 16), batch, between(64, min(4000, 32000 // batch)),
                     rng.randint(2, 5), spread=spread)
    if kind == 2:
        batch = between(1, 4)
        return _case(None, "qwen3_8b", "prompt", rng.randint(8, 24), batch, between(40, 5000 // batch), spread=spread)
    if kind == 3:
        return _case(None, "qwen3_4b", "mixed", rng.randint(8, 24), between(2, 32), between(100, 700), rng.randint(2, 4),
                     spread=spread, portion=between(100, 1000))
    if kind == 4:
        return _case(None, "qwen3_8b", "job", rng.randint(2, 4), between(1, 6), between(30, 300), rng.randint(2, 6),
                     dtype="float32", spread=spread)
    model = rng.choice(sorted(_DESIGNS))
    width = rng.choice([2048, 4096])
    layers = 6 if model == "rupezen" else rng.choice([4, 8]) if model != "mapalorn" else rng.randint(4, 7)
    batch = between(1, 64)
    return _case(None, model, rng.choice(["job", "job", "prompt", "decode"]), layers, batch,
                 between(20, 3000) if batch == 1 else between(12, max(16, 3000 // batch)), rng.randint(3, 8), width=width, spread=spread)


# ------------------------------------------------------------------------------------------- inputs
def _lengths(case):
    """Tokens of every request's prompt: around ``prompt``, apart by up to ``spread`` of it."""
    n, p, s = case["batch"], case["prompt"], case["spread"]
    if n == 1 or not s:
        return [p] * n
    return [max(2, int(round(p * (1.0 + s * (2.0 * ((i * 37) % n) / (n - 1) - 1.0))))) for i in range(n)]


def _room(case):
    """Tokens a request may hold: its prompt and, for requests that live on from pass to pass, what they grow by."""
    longest = max(_lengths(case))
    return longest + (2000 if case["use"] in ("decode", "mixed") else case["steps"] + 1)


def _tokens(case, seed):
    """The token ids that requests are given, [requests + newcomer, room]."""
    vocab = _vocab(_config(case))
    gen = torch.Generator().manual_seed(int(seed) + 1)
    return torch.randint(0, vocab, (case["batch"] + 1, max(_room(case), case["steps"] * case["portion"])), generator=gen)


def _vocab(raw):
    return raw.get("vocab_size") or raw["vocab"]


def _weights(case, seed):
    """The model's tensors by name, on the device. What ends a sublayer (its last matrix, or the norm behind it) is a
    quarter of its usual size: as in trained models, a sublayer changes the stream by a part of what it holds."""
    import return_amd.models  # noqa: F401
    from return_amd.config import lookup_architecture
    from return_amd.weights import random_weights
    raw = _config(case)
    cls, build_spec = lookup_architecture((raw.get("architectures") or [raw.get("architecture")])[0])
    cfg = cls.from_dict(raw)
    width = raw.get("hidden_size") or raw["width"]
    scaled = (raw.get("embedding") or {}).get("scale", 1.0)
    weights = random_weights(build_spec(cfg), seed=int(seed), std=0.02 if width > 1000 else 0.04, embedding_std=1.0 / scaled,
                             dtype=case["dtype"], device=DEVICE, generator_device=DEVICE)
    # (one expert of many counts for less: in two implementations a token's last expert may differ when two scores
    # nearly tie. The Mapalorn design adds its experts up without weights.)
    routed = 1 / 64 if case["model"] == "mapalorn" else 1 / 16
    for name, w in weights.items():
        if re.search(r"(mix\.|left\.|right\.)o$|down$|(o|down)_proj\.weight$|side\.norm$", name):
            w.mul_(routed if re.search(r"\.e\d+\.", name) else 1 / 4)
        elif case["model"] == "mepolix" and re.search(r"\.norm[12]$", name):
            w.mul_(0.25)
        elif case["model"] == "safilorn" and re.search(r"\.norm[12]b$", name):
            w.sub_(0.75)                       # (this design's norms multiply by one and the weight)
    return cfg, weights


def prepare(case, seed):
    from return_amd.config import EngineConfig
    from return_amd.engine import ModelRunner
    cfg, weights = _weights(case, seed)
    lengths, most = _lengths(case), 0
    n, room = case["batch"] + 1, _room(case) + 16
    step = max(sum(lengths), case["batch"] + case["portion"], 64)
    most = case["batch"] * room + case["steps"] * case["portion"] + 64
    runner = ModelRunner(config=cfg, weights=weights, engine_config=EngineConfig(
        dtype=case["dtype"], max_token=most, max_reside=n, max_step_tokens=step, prefill_chunk=step, device=DEVICE))
    del weights
    state = {"case": case, "runner": runner, "tokens": _tokens(case, seed).tolist(), "lengths": lengths,
             "ids": ["r%d" % i for i in range(case["batch"])], "room": _room(case)}
    if case["use"] in ("decode", "mixed"):
        _seat(state)
        _decode(state, 1)                # the first token behind the prompt: the engine is running
    return state


# ------------------------------------------------------------------------------------------- one pass
def _prompts(state):
    """All prompts in one step; the logits behind each one's last token."""
    from return_amd.engine import StepEntry
    runner = state["runner"]
    for rid in state["ids"]:
        runner.add_request(rid)
    entries = [StepEntry(rid, state["tokens"][i][:n], [n - 1])
               for i, (rid, n) in enumerate(zip(state["ids"], state["lengths"]))]
    return runner.step(entries)


def _seat(state):
    _prompts(state)
    state["held"] = list(state["lengths"])


def _end(state):
    for rid in state["ids"]:
        state["runner"].free_request(rid)


def _decode(state, steps):
    """Single-token steps of all requests, each launched before the one before it is collected. The tokens are
    given; the sampler runs as in generation (nucleus sampling) and what it picks is not used."""
    runner, ids, held = state["runner"], state["ids"], state["held"]
    n = len(ids)
    rows, ticket = [], None
    for s in range(steps):
        ahead = runner.decode_launch(ids, [state["tokens"][i][held[i]] for i in range(n)], [0.7] * n, [0] * n, [0.9] * n,
                                     [(0.37 + 0.11 * i + 0.23 * s) % 1.0 for i in range(n)])
        rows.append(ahead[2].clone())
        if ticket is not None:
            runner.decode_collect(ticket)
        ticket = ahead
        for i in range(n):
            held[i] += 1
    runner.decode_collect(ticket)
    return torch.stack(rows)


def _mixed(state):
    """A newcomer's prompt in portions, each in one step with a token of every other request."""
    from return_amd.engine import StepEntry
    case, runner, ids, held = state["case"], state["runner"], state["ids"], state["held"]
    n, p = len(ids), case["portion"]
    runner.add_request("new")
    rows, ticket = [], None
    for s in range(case["steps"]):
        last = s == case["steps"] - 1
        entries = [StepEntry(rid, [state["tokens"][i][held[i]]], [0]) for i, rid in enumerate(ids)]
        entries.append(StepEntry("new", state["tokens"][n][s * p:(s + 1) * p], [p - 1] if last else []))
        m = n + int(last)
        ahead = runner.step_launch(entries, [0.7] * m, [0] * m, [0.9] * m, [(0.37 + 0.11 * i) % 1.0 for i in range(m)])
        rows.append(ahead[2].clone())
        if ticket is not None:
            runner.decode_collect(ticket)
        ticket = ahead
        for i in range(n):
            held[i] += 1
    runner.decode_collect(ticket)
    runner.free_request("new")
    return rows


def run(state):
    case = state["case"]
    if case["use"] == "prompt":
        out = _prompts(state)
        _end(state)
        return out
    if case["use"] == "job":
        first = _prompts(state)
        state["held"] = list(state["lengths"])
        out = [first, _decode(state, case["steps"])]
        _end(state)
        return out
    if max(state["held"]) + case["steps"] > state["room"]:    # a conversation that is full ends, the next one begins
        _end(state)
        _seat(state)
        _decode(state, 1)
    return _decode(state, case["steps"]) if case["use"] == "decode" else _mixed(state)


# ------------------------------------------------------------------------------------------- what a pass needs
def work(case):
    """Bytes: every matrix once a step (of the experts those that the step's tokens choose, when they choose evenly),
    the keys and values read and written, recurrent states read and written once a step, the logits. Operations: two
    per matrix element and token, and the attention's."""
    import return_amd.models  # noqa: F401
    from return_amd.config import lookup_architecture
    raw = _config(case)
    cls, build_spec = lookup_architecture((raw.get("architectures") or [raw.get("architecture")])[0])
    spec = build_spec(cls.from_dict(raw))
    size = 2 if case["dtype"] == "bfloat16" else 4
    runs, vocab = _runs(raw), _vocab(raw)
    width = raw.get("hidden_size") or raw["width"]
    times = {}
    for i in runs:
        times[i] = times.get(i, 0) + 1
    dense = routed = 0
    for name, (shape, _) in spec.expected_tensors().items():
        at = re.match(r"(?:model\.layers\.|l)(\d+)\.", name)
        if at is None or len(shape) < 2:
            continue
        count = math.prod(shape) * times.get(int(at.group(1)), 0)
        if re.search(r"\.mlp\.e\d+\.", name):
            routed += count
        else:
            dense += count
    head = vocab * width
    lengths = _lengths(case)
    kv, states, attention = _kept(raw, runs, size)

    def step(tokens, seqs, before):
        """tokens in all, requests, keys that their queries read before these tokens (a number per request)"""
        share = 1.0 - (1.0 - 4 / 32) ** tokens
        data = (dense + routed * share + head) * size + states * 2 * seqs + (sum(before) + tokens) * kv
        data += seqs * vocab * 4 + tokens * width * size
        flops = 2.0 * tokens * (dense + routed * 4 / 32) + 2.0 * seqs * head
        return data, flops

    steps = []
    if case["use"] in ("prompt", "job"):
        data, flops = step(sum(lengths), len(lengths), [0])
        steps.append((data, flops + attention * sum(n * (n + 1) / 2 for n in lengths)))
    for s in range(case["steps"] if case["use"] != "prompt" else 0):
        held = [n + s + (2 if case["use"] in ("decode", "mixed") else 1) for n in lengths]
        tokens = len(held) + case["portion"]
        data, flops = step(tokens, len(held), held)
        p = case["portion"]
        data += s * p * kv if p else 0
        flops += attention * (sum(held) + (s * p * p + p * (p + 1) / 2 if p else 0))
        steps.append((data, flops))
    return {"bytes": sum(d for d, _ in steps), "flops": sum(f for _, f in steps)}


def _kept(raw, runs, size):
    """(bytes of keys and values per token over all layers, bytes of recurrent state per request, operations per
    query and key over all layers)."""
    if "num_hidden_layers" in raw:
        d, n = raw["head_dim"], len(runs)
        return 2 * raw["num_key_value_heads"] * d * size * n, 0, 4.0 * raw["num_attention_heads"] * d * n
    kv = states = ops = 0
    for i in runs:
        layer = raw["layers"][i]
        m = layer["mixer"]
        kind = layer["type"]
        if kind == "parallel":
            states += m["right"]["width"] * 4
            m, kind = m["left"], "attention"
        if kind == "latent_attention":
            kv += (m["kv_rank"] + m.get("rot_dim", 0)) * size
            ops += 2.0 * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"])
        elif kind == "attention":
            maps = 2 if "diff" in m else 1
            kv += m["kv_heads"] * (maps * m["dim"] + m["vdim"]) * size
            ops += 2.0 * m["heads"] * maps * (m["dim"] + m["vdim"])
        elif kind == "mamba2":
            states += m["heads"] * m["vdim"] * m["state"] * 4
        else:
            states += m["heads"] * m["dim"] * m["vdim"] * 4
    return kv, states, ops


def tolerance(case):
    """Measured against exact(): 0.5 to 5 millionths in 32 bits, 0.2 % (few layers) to 1.3 % (36 layers) in bfloat16."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5}
    return {"rel": 0.02}


# ------------------------------------------------------------------------------------------- the same in 64 bits
# Prompts lie in one padded block [requests, longest, ...]; everything is causal, so what stands behind a shorter
# request's end reaches nothing before it.
def _rms(x, eps, weight=None):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if weight is None else y * weight


def _layer_norm(x, eps, weight, bias=None):
    x = x - x.mean(-1, keepdim=True)
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * weight
    return y if bias is None else y + bias


def _silu(x):
    return x * torch.sigmoid(x)


def _turn(x, rot, pairs=False):
    """x [B, T, heads, D]: the first rot.dims elements of every head turn by their position; element i with
    i + dims/2, or neighbours with ``pairs``."""
    if not rot:
        return x
    dims, base, s = int(rot["dims"]), float(rot["base"]), rot.get("scaling")
    i = torch.arange(dims // 2, dtype=F64, device=x.device)
    f, gain = base ** (-2.0 * i / dims), 1.0
    if s and "original" in s:
        def place(turns):
            return dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(place(s["fast"])), 0), min(math.ceil(place(s["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, gain = f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1.0
    elif s:
        f = f / s["factor"]
    a = torch.arange(x.shape[1], dtype=F64, device=x.device)[:, None] * f
    cos, sin = (a.cos() * gain)[None, :, None], (a.sin() * gain)[None, :, None]
    out = x.clone()
    at = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    u, v = x[..., at[0]], x[..., at[1]]
    out[..., at[0]], out[..., at[1]] = u * cos - v * sin, v * cos + u * sin
    return out


def _attend(q, k, v, scale, temperature=None, cap=None, window=None, keep=0, chunk=None, sink=None):
    """q [B, T, H, D], k [B, T, G, D], v [B, T, G, V] -> [B, T, H, V]; sink: per head, a further term of the
    denominator as a logarithm."""
    B, T, H, _ = q.shape
    G, V = k.shape[2], v.shape[3]
    out = torch.empty(B, T, H, V, dtype=F64, device=q.device)
    per = max(1, min(T, int(2e8 / (H * T))))
    j = torch.arange(T, device=q.device)[None, :]
    for b in range(B):
        kk, vv = k[b].transpose(0, 1).contiguous(), v[b].transpose(0, 1).contiguous()      # [G, T, .]
        for a in range(0, T, per):
            qq = q[b, a:a + per]
            t = qq.shape[0]
            s = torch.matmul(qq.view(t, G, H // G, -1).permute(1, 2, 0, 3).reshape(G, H // G * t, -1),
                             kk.transpose(1, 2).contiguous()).view(H, t, T) * scale
            if temperature is not None:
                s = s * temperature[:, None, None]
            if cap:
                s = cap * torch.tanh(s / cap)
            i = torch.arange(a, a + t, device=q.device)[:, None]
            see = j <= i
            if window:
                see = see & ((i - j < window) | (j < keep))
            if chunk:
                see = see & (i // chunk == j // chunk)
            s = s.masked_fill(~see, -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[:, None, None])
            p = torch.exp(s - top)
            total = p.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[:, None, None] - top)
            o = torch.matmul((p / total).view(G, H // G * t, T), vv)
            out[b, a:a + t] = o.view(H, t, V).transpose(0, 1)
    return out


def _filter(x, taps, bias=None):
    """Causal filter on every channel: x [B, T, C], taps [C, K], the last tap on the row itself."""
    K = taps.shape[1]
    y = x * taps[:, K - 1]
    for j in range(1, K):
        y[:, j:] += x[:, :-j] * taps[:, K - 1 - j]
    return y if bias is None else y + bias


def _recur(q, k, v, decay, beta=None):
    """S_t = decay S_(t-1) + k (x) u, o_t = S_t^T q, with u = v, or beta (v - S^T k) for the delta rule.
    q, k [B, T, H, D], v [B, T, H, V], decay [B, T, H, D or 1], beta [B, T, H]."""
    B, T, H, D = q.shape
    S = torch.zeros(B, H, D, v.shape[3], dtype=F64, device=q.device)
    out = torch.empty_like(v)
    for t in range(T):
        S = S * decay[:, t, :, :, None]
        u = v[:, t]
        if beta is not None:
            u = beta[:, t, :, None] * (u - (k[:, t, :, None] @ S)[:, :, 0])
        S.addcmul_(k[:, t, :, :, None], u[:, :, None])
        out[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
    return out


class _Layer:
    """The tensors of one layer in 64 bits, by the rest of their names."""

    def __init__(self, weights, prefix):
        self.weights, self.prefix = weights, prefix

    def __getitem__(self, name):
        return self.weights[self.prefix + name].to(F64)

    def mul(self, x, name):
        return x @ self[name].T

    def under(self, prefix):
        return _Layer(self.weights, self.prefix + prefix)


def _heads(x, n):
    return x.view(*x.shape[:2], n, -1)


def _repeat(x, times):
    return x.repeat_interleave(times, dim=2)


def _softplus(x):
    return torch.logaddexp(x, torch.zeros((), dtype=F64, device=x.device))


def _clamped(w, x, limit, p=""):
    g = w.mul(x, p + "gate").clamp(max=limit)
    u = w.mul(x, p + "up").clamp(-limit, limit)
    return w.mul(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down")


def _gated(w, x, p=""):
    return w.mul(_silu(w.mul(x, p + "gate")) * w.mul(x, p + "up"), p + "down")


def _experts(w, x, ids, weights, expert):
    """Sum over a token's chosen experts of weight * expert(x, factor is in the weights)."""
    flat, out = x.reshape(-1, x.shape[-1]), torch.zeros(x.shape, dtype=F64, device=x.device).view(-1, x.shape[-1])
    for e in range(32):
        hit = (ids == e).nonzero()
        if hit.numel():
            out.index_add_(0, hit[:, 0], expert(flat[hit[:, 0]], weights[hit[:, 0], hit[:, 1], None], "e%d." % e))
    return out.view(x.shape)


def _grouped(choice, groups, per_group):
    """Choice scores with those outside the best groups taken out; a group scores its best ``per_group`` members."""
    g = choice.view(choice.shape[0], groups["count"], -1)
    best = g.topk(per_group, -1).values.sum(-1).topk(groups["keep"], -1).indices
    allowed = torch.zeros(g.shape[:2], dtype=torch.bool, device=choice.device).scatter_(1, best, True)
    return g.masked_fill(~allowed[..., None], -math.inf).reshape(choice.shape)


def _moe(model, w, x, mlp):
    top = mlp["router"]["top"]
    z = w.mul(x.reshape(-1, x.shape[-1]), "router")
    if model == "rupezen":
        s = torch.sigmoid(z)
        ids = _grouped(s + w["correction"], mlp["router"]["groups"], 2).topk(top, -1).indices
        p = s.gather(1, ids)
        return _experts(w, x, ids, p / (p.sum(-1, keepdim=True) + 1e-20), lambda h, a, e: a * _gated(w, h, e))
    if model == "safilorn":
        val, ids = (z + w["router.b"]).topk(top, -1)
        return _experts(w, x, ids, val.softmax(-1), lambda h, a, e: a * _clamped(w, h, mlp["expert"]["limit"], e))
    if model == "fefulorn":
        s = z.softmax(-1)
        ids = _grouped(s, mlp["router"]["groups"], 1).topk(top, -1).indices
        y = _experts(w, x, ids, s.gather(1, ids), lambda h, a, e: a * _clamped(w, h, mlp["expert"]["limit"], e))
        return y + _clamped(w, x, mlp["shared"]["limit"], "shared.") * torch.sigmoid(w.mul(x, "shared.sg"))
    s = torch.sigmoid(z)
    ids = s.topk(top, -1).indices
    y = _experts(w, x, ids, s.gather(1, ids), lambda h, a, e: _gated(w, a * h, e))
    return y + _gated(w, x, "shared.") * torch.sigmoid(w.mul(x, "shared.sg"))


def _latent(w, h, m, eps, pairs, window=None):
    H, C, R = m["heads"], m["kv_rank"], m.get("rot_dim", 0)
    q = _heads(w.mul(_rms(w.mul(h, "dq"), eps, w["dq.norm"]), "uq") if m.get("q_rank") else w.mul(h, "q"), H)
    z = w.mul(h, "dkv")
    c = _rms(z[..., :C], eps, w["dkv.norm"])
    k, v = _heads(w.mul(c, "uk"), H), _heads(w.mul(c, "uv"), H)
    if R:
        D = m["dim"]
        q = torch.cat([q[..., :D], _turn(q[..., D:], m["rot"], pairs)], -1)
        k = torch.cat([k, _turn(z[..., None, C:], m["rot"], pairs).expand(-1, -1, H, -1)], -1)
    return _attend(q, k, v, m["scale"], window=window, sink=w["sink"] if R else None)


def _kofipel_mixer(w, h, layer, eps):
    m = layer["mixer"]
    H, G = m["heads"], m["kv_heads"]
    if layer["type"] == "attention":
        q, k = _heads(w.mul(h, "q") + w["q.b"], H), _heads(w.mul(h, "k") + w["k.b"], G)
        o = _attend(_turn(q, m["rot"]), _turn(k, m["rot"]), k, m["scale"], w["temp"], m["softcap"], m["mask"]["size"],
                    m["mask"]["keep_first"], sink=torch.zeros(H, dtype=F64, device=h.device))
        return w.mul(o.flatten(2), "o") + w["o.b"]
    q, k, v = (_silu(_filter(w.mul(h, n), w[n + ".conv"])) for n in "qkv")
    q, k = (_heads(x, G) * torch.rsqrt((_heads(x, G) ** 2).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    decay = torch.exp(-torch.exp(w["A_log"])[:, None] * _heads(_softplus(w.mul(w.mul(h, "a1"), "a2") + w["dt_bias"]), H))
    o = _recur(_repeat(q, H // G) * m["dim"] ** -0.5, _repeat(k, H // G), _heads(v, H), decay, torch.sigmoid(w.mul(h, "b")))
    return w.mul((_rms(o, eps, w["norm"]) * torch.sigmoid(_heads(w.mul(w.mul(h, "g1"), "g2"), H))).flatten(2), "o")


def _mepolix_mixer(w, h, layer, eps):
    m = layer["mixer"]
    if layer["type"] == "delta":
        H, G = m["heads"], m["kv_heads"]
        q, k, v = (_silu(_filter(w.mul(h, n), w[n + ".conv"])) for n in "qkv")
        q, k = (_heads(x, G) * torch.rsqrt((_heads(x, G) ** 2).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        decay = torch.exp(-torch.exp(w["A_log"]) * _softplus(w.mul(h, "a") + w["dt_bias"]))[..., None]
        o = _recur(_repeat(q, H // G) * m["dim"] ** -0.5, _repeat(k, H // G), _heads(v, H), decay, torch.sigmoid(w.mul(h, "b")))
        return w.mul((_rms(o, eps, w["norm"]) * _heads(_silu(w.mul(h, "g")), H)).flatten(2), "o")
    a, c, l, r = m["left"], m["right"], w.under("left."), w.under("right.")
    q = _turn(_rms(_heads(l.mul(h, "q"), a["heads"]), eps, l["q.norm"]), a["rot"])
    k = _turn(_rms(_heads(l.mul(h, "k"), a["kv_heads"]), eps, l["k.norm"]), a["rot"])
    left = l.mul(_attend(q, k, _heads(l.mul(h, "v"), a["kv_heads"]), a["scale"], sink=l["sink"]).flatten(2), "o")
    y = torch.nn.functional.gelu(r.mul(h, "y") + r["y.b"], approximate="tanh")
    u = _filter(r.mul(h, "x") + r["x.b"], r["conv"], r["conv.b"])
    gates = [torch.sigmoid((torch.einsum("btnc,ndc->btnd", _heads(u, c["blocks"]), r[n]) + r[n + ".b"]).flatten(2)) for n in ("ra", "ri")]
    log_a = -8.0 * gates[0] * _softplus(r["lam"])
    decay, x = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * gates[1] * u
    S, out = torch.zeros_like(u[:, 0]), torch.empty_like(u)
    for t in range(u.shape[1]):
        S = decay[:, t] * S + x[:, t]
        out[:, t] = S
    return m["left_scale"] * left + m["right_scale"] * r.mul(out * y, "o")


def _mamba(w, h, m, eps):
    B, T, _ = h.shape
    H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    inner = H * P
    z, xbc, dt = w.mul(h, "in").split([inner, inner + 2 * G * N, H], -1)
    xbc = _silu(_filter(xbc, w["conv"], w["conv.b"]))
    x, Bm, C = xbc.split([inner, G * N, G * N], -1)
    x, dt = _heads(x, H), _softplus(dt + w["dt_bias"])
    y = _recur(_repeat(_heads(C, G), H // G), _repeat(_heads(Bm, G), H // G) * dt[..., None], x,
               torch.exp(-torch.exp(w["A_log"]) * dt)[..., None])
    y = (y + w["D"][:, None] * x).flatten(2) * _silu(z)
    return w.mul(_rms(_heads(y, m["norm_groups"]), eps).flatten(2) * w["norm"], "o")


def _stream(case, raw, weights, tokens):
    """The stream after the last layer, [B, T, width]; tokens [B, T]."""
    model = case["model"]
    if model in _QWEN:
        eps, d, rot = raw["rms_norm_eps"], raw["head_dim"], {"dims": raw["head_dim"], "base": raw["rope_theta"]}
        x = weights["model.embed_tokens.weight"].to(F64)[tokens]
        for i in range(raw["num_hidden_layers"]):
            w = _Layer(weights, "model.layers.%d." % i)
            h, a = _rms(x, eps, w["input_layernorm.weight"]), w.under("self_attn.")
            q = _turn(_rms(_heads(a.mul(h, "q_proj.weight"), raw["num_attention_heads"]), eps, a["q_norm.weight"]), rot)
            k = _turn(_rms(_heads(a.mul(h, "k_proj.weight"), raw["num_key_value_heads"]), eps, a["k_norm.weight"]), rot)
            v = _heads(a.mul(h, "v_proj.weight"), raw["num_key_value_heads"])
            x = x + a.mul(_attend(q, k, v, d ** -0.5).flatten(2), "o_proj.weight")
            h, f = _rms(x, eps, w["post_attention_layernorm.weight"]), w.under("mlp.")
            x = x + f.mul(_silu(f.mul(h, "gate_proj.weight")) * f.mul(h, "up_proj.weight"), "down_proj.weight")
        return _rms(x, eps, weights["model.norm.weight"].to(F64))
    eps = raw["norm"]["eps"]
    x = weights["embed"].to(F64)[tokens] * (raw.get("embedding") or {}).get("scale", 1.0)
    first, results, passes = x, [x], 0
    for i in _runs(raw):
        layer, w = raw["layers"][i], _Layer(weights, "l%d." % i)
        m, mlp, mix, ff = layer["mixer"], layer["mlp"], w.under("mix."), w.under("mlp.")
        if model == "kofipel":
            h = _rms(x, eps, w["norm1"])
            x = x + _kofipel_mixer(mix, h + _filter(h, w["canon1"]), layer, eps)
            h = _rms(x, eps, w["norm2"])
            h = h + _filter(h, w["canon2"])
            x = x + ff.mul(torch.relu(ff.mul(h, "up")) ** 2, "down")
            n = raw["token_side"]["dim"]
            side = weights["side.embed"].to(F64)[tokens][..., i * n:(i + 1) * n]
            y = w.mul(torch.nn.functional.gelu(w.mul(x, "side.gate"), approximate="tanh") * side, "side.proj")
            x = x + _rms(y, eps, w["side.norm"])
        elif model == "mepolix":
            x = x + _layer_norm(_mepolix_mixer(mix, x, layer, eps), eps, w["norm1"])
            x = x + _layer_norm(_gated(ff, x), eps, w["norm2"])
        elif model == "rupezen":
            loop = raw["loop"]
            if i == loop["start"]:
                x = torch.cat([x, first], -1) @ weights["loop.in"].to(F64).T + weights["loop.step"].to(F64)[passes]
                passes += 1
            h = _rms(x, eps, w["norm1"])
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            q, k = (_turn(_heads(mix.mul(h, n), 2 * c), m["rot"], True).unflatten(2, (c, 2)) for n, c in (("q", H), ("k", G)))
            v, c = _heads(mix.mul(h, "v"), G), m["mask"]["size"]
            one, two = (_attend(q[:, :, :, j].contiguous(), k[:, :, :, j], v, m["scale"], chunk=c) for j in (0, 1))
            lam = torch.exp((mix["lq1"] * mix["lk1"]).sum()) - torch.exp((mix["lq2"] * mix["lk2"]).sum()) + m["diff"]
            x = x + raw["residual_mult"] * mix.mul((_rms(one - lam * two, eps) * (1 - m["diff"])).flatten(2), "o")
            x = x + raw["residual_mult"] * _moe(model, ff, _rms(x, eps, w["norm2"]), mlp)
        elif model == "safilorn":
            h = _rms(x, eps, 1 + w["norm1"])
            if layer["type"] == "latent_attention":
                y = mix.mul((_latent(mix, h, m, eps, False) * torch.sigmoid(mix.mul(h, "g"))[..., None]).flatten(2), "o")
            else:
                H = m["heads"]
                q, k, v = (_heads(mix.mul(h, n), H) for n in "qkv")
                decay = torch.sigmoid(_heads(mix.mul(mix.mul(h, "a1"), "a2") + mix["a2.b"], H)) ** (1 / m["tau"])
                o = _rms(_recur(q * m["dim"] ** -0.5, k, v, decay), eps, mix["norm"])
                y = mix.mul(o.flatten(2) * _silu(mix.mul(h, "g")), "o")
            x = x + _rms(y, eps, 1 + w["norm1b"])
            h = _rms(x, eps, 1 + w["norm2"])
            if mlp["kind"] == "dense":
                y = ff.mul(_silu(ff.mul(h, "gate") + ff["gate.b"]) * (ff.mul(h, "up") + ff["up.b"]), "down") + ff["down.b"]
            else:
                y = _moe(model, ff, h, mlp)
            results.append(x + _rms(y, eps, 1 + w["norm2b"]))
            x = sum(a * r for a, r in zip(w["dwa"], results))
        elif model == "fefulorn":
            h = _rms(x, eps, w["norm1"])
            if layer["type"] == "mamba2":
                y = _mamba(mix, h, m, eps)
            elif layer["type"] == "latent_attention":
                y = mix.mul(_latent(mix, h, m, eps, False, m["mask"]["size"]).flatten(2), "o")
            else:      # (at most one such layer in these shapes: its values are the first, nothing is blended in)
                q, k, v = (_heads(mix.mul(h, n) + mix[n + ".b"], m["heads" if n == "q" else "kv_heads"]) for n in "qkv")
                y = mix.mul(_attend(_turn(q, m["rot"]), _turn(k, m["rot"]), v, m["scale"], window=m["mask"]["size"]).flatten(2), "o")
            x = x + y + _moe(model, ff, _rms(x, eps, w["norm2"]), mlp)
        else:
            h = _layer_norm(x, eps, w["norm1"], w["norm1.b"])
            if layer["type"] == "latent_attention":
                y = _latent(mix, h, m, eps, True)
            else:
                q = _turn(_heads(_rms(mix.mul(h, "q"), eps, mix["q.norm"]), m["heads"]), m["rot"])
                k = _turn(_heads(_rms(mix.mul(h, "k"), eps, mix["k.norm"]), m["kv_heads"]), m["rot"])
                y = _attend(q, k, _heads(mix.mul(h, "v"), m["kv_heads"]), m["scale"], sink=torch.zeros(m["heads"], dtype=F64, device=h.device))
                y = y * _heads(torch.sigmoid(mix.mul(h, "g")), m["heads"])
            x = x + mix.mul(y.flatten(2), "o") + (_clamped(ff, h, mlp["limit"]) if mlp["kind"] == "dense" else _moe(model, ff, h, mlp))
    if model == "mapalorn":
        return _layer_norm(x, eps, weights["final.norm"].to(F64), weights["final.norm.b"].to(F64))
    if model == "mepolix":
        return _layer_norm(x, eps, weights["final.norm"].to(F64))
    return _rms(x, eps, weights["final.norm"].to(F64) + (1.0 if model == "safilorn" else 0.0))


def _head(raw, weights, x):
    name = ("lm_head.weight", "model.embed_tokens.weight") if "hidden_size" in raw else ("head", "embed")
    w = weights[name[0]] if name[0] in weights and not raw.get("tie_word_embeddings") else weights[name[1]]
    z = x @ w.to(F64).T
    cap = raw.get("logit_softcap")
    return cap * torch.tanh(z / cap) if cap else z


@torch.no_grad()
def exact(case, seed):
    """What run() returns on a new state, in 64 bits."""
    raw, (_, weights) = _config(case), _weights(case, seed)
    lengths, tokens, steps = _lengths(case), _tokens(case, seed).to(DEVICE), case["steps"]
    B, extra = case["batch"], {"prompt": 0, "job": steps, "decode": steps + 1, "mixed": steps + 1}[case["use"]]
    longest, first = max(lengths) + extra, 1 if case["use"] in ("decode", "mixed") else 0
    part = max(1, int(6e8 // (longest * 4 * (raw.get("hidden_size") or raw["width"]))))       # requests at a time
    rows = [_stream(case, raw, weights, tokens[b:min(b + part, B), :longest]) for b in range(0, B, part)]
    rows = torch.cat([r[torch.arange(r.shape[0], device=r.device)[:, None], at]
                      for r, at in zip(rows, _places(lengths, extra, first, case["use"], part))])      # [B, places, width]
    if case["use"] == "prompt":
        return _head(raw, weights, rows[:, 0])
    if case["use"] == "job":
        return [_head(raw, weights, rows[:, 0]), torch.stack([_head(raw, weights, rows[:, 1 + s]) for s in range(steps)])]
    out = [_head(raw, weights, rows[:, s]) for s in range(steps)]
    if case["use"] == "decode":
        return torch.stack(out)
    new = _stream(case, raw, weights, tokens[B:, :steps * case["portion"]])[:, -1]
    out[-1] = torch.cat([out[-1], _head(raw, weights, new)])
    return out


def _places(lengths, extra, first, use, part):
    """Per block of requests, the places whose logits run() returns, [requests, places]."""
    at = torch.tensor([[n + first + s if use in ("decode", "mixed") else n - 1 + s
                        for s in range(extra - first if use in ("decode", "mixed") else extra + 1)] for n in lengths], device=DEVICE)
    return [at[b:b + part] for b in range(0, len(lengths), part)]
