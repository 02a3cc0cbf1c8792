"""The work this engine is timed by: steps of its decoders as a program that serves or replays
them runs them, through `Engine.step` and `Engine.generate`.

    listed()             the cases, by name
    draw(rng)            one more case of the ranges the listed ones stand for
    prepare(case, seed)  an engine with its weights, and requests with what their caches hold
    run(state)           one pass: the logits (and sampled tokens) it returns
    work(case)           the bytes and operations a pass cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    the same outputs in 64 bits, in plain tensor operations

A case is one of three kinds.  "step": one `Engine.step` in which `decodes` requests bring a token
each, over caches of `context_from` to `context_to` tokens, and `prompts` requests bring a portion of
`prompt_from` to `prompt_to` tokens, from position `start` (their caches hold what lies before it).
"replay": `prompts` requests opened, run through their prompts in one step and then `tokens` times
with a given next token each, closed: what the trace replay does, and the only repeatable form of
decoding for decoders with a recurrent state.  "generate": `Engine.generate` over `prompts` prompts,
`tokens` new tokens each, sampled, and the logits of the last prompt's every place (a score of it).

Shapes are the engine's own: the tiny shape of its tests, the Llama-3.2-1B, Llama-3.1-8B and
Llama-3.1-70B shapes (the last in fewer layers, to fit beside others in memory) and the decoders that
are measured beside Llama at the 1B widths.  Weights are random, as no checkpoint is needed for timing.
Routed experts appear in 32-bit only: in bfloat16 two correct implementations choose different experts
for tokens whose scores nearly tie, and logits could not be compared."""
import math
import zlib

import torch

PAGE = 16
STEP_TOKENS = 2048          # the engine's default budget of a step


def _llama(layers, hidden, heads, kv_heads, head_dim, inter, factor, tied):
    return dict(architectures=["LlamaForCausalLM"], num_hidden_layers=layers, hidden_size=hidden, num_attention_heads=heads,
                num_key_value_heads=kv_heads, head_dim=head_dim, intermediate_size=inter, vocab_size=128256, rope_theta=500000.0,
                rope_scaling=dict(rope_type="llama3", factor=factor, low_freq_factor=1.0, high_freq_factor=4.0,
                                  original_max_position_embeddings=8192),
                max_position_embeddings=8192, rms_norm_eps=1e-5, tie_word_embeddings=tied, hidden_act="silu")


_TINY = dict(_llama(3, 96, 3, 1, 32, 320, 8.0, False), vocab_size=384, max_position_embeddings=512, rms_norm_eps=1e-6)
_TINY["rope_scaling"] = dict(_TINY["rope_scaling"], original_max_position_embeddings=64)

_LLAMAS = {"llama_tiny": _TINY,
           "llama_1b": _llama(16, 2048, 32, 8, 64, 8192, 32.0, True),
           "llama_8b": _llama(32, 4096, 32, 8, 128, 14336, 8.0, False),
           "llama_70b": _llama(80, 8192, 64, 8, 128, 28672, 8.0, False)}


def _tuvodra(repeats):
    """Layers in threes at the 1B widths: a minGRU, a selective scan, windowed attention with a feed-forward."""
    three = [{"type": "mingru", "mixer": {"width": 2048}, "mlp": None},
             {"type": "mamba1", "mixer": {"inner": 4096, "state": 16, "conv": 4, "dt_rank": 128}, "mlp": None},
             {"type": "attention", "mixer": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 1024}},
              "mlp": {"kind": "dense", "ff": 8192}}]
    return {"architecture": "Tuvodra", "vocab": 128256, "width": 2048, "streams": 4, "embedding": {"scale": 1.0},
            "norm": {"eps": 1e-6, "groups": 4}, "layers": [dict(layer) for _ in range(repeats) for layer in three]}


def _tevovik(repeats):
    """Layers in threes at the 1B widths, the second on the first's keys and values: differential attention and 16 experts in
    four groups, two groups kept and four experts chosen."""
    mix = lambda kv_from: {"heads": 16, "kv_heads": 4, "dim": 64, "vdim": 128, "scale": 0.125, "diff": 0.4, "mask": {"size": 4096},
                           **({} if kv_from is None else {"kv_from": kv_from})}
    mlp = lambda: {"kind": "moe", "expert": {"ff": 2048}, "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}}}
    return {"architecture": "Tevovik", "vocab": 128256, "width": 2048, "embedding": {"scale": 50.0}, "norm": {"eps": 1e-6},
            "layers": [{"type": "attention", "mixer": mix(3 * r if i == 1 else None), "mlp": mlp()} for r in range(repeats) for i in range(3)]}


def _shape(case):
    model, layers = case["model"], case["layers"]
    if model == "tuvodra":
        return _tuvodra(layers // 3)
    if model == "tevovik":
        return _tevovik(layers // 3)
    return dict(_LLAMAS[model], num_hidden_layers=layers)


# ---- the cases ------------------------------------------------------------------------------------------------------

def _step(model, layers, dtype="bfloat16", decodes=0, context=(0, 0), prompts=0, prompt=(0, 0), start=0):
    return {"kind": "step", "model": model, "layers": layers, "dtype": dtype, "decodes": decodes, "context_from": context[0],
            "context_to": context[1], "prompts": prompts, "prompt_from": prompt[0], "prompt_to": prompt[1], "start": start}


def _replay(model, layers, dtype, prompts, prompt, tokens):
    return {"kind": "replay", "model": model, "layers": layers, "dtype": dtype, "prompts": prompts, "prompt_from": prompt[0],
            "prompt_to": prompt[1], "tokens": tokens}


def _generate(prompts, prompt, tokens):
    return {"kind": "generate", "model": "llama_tiny", "layers": 3, "dtype": "float32", "prompts": prompts, "prompt_from": prompt[0],
            "prompt_to": prompt[1], "tokens": tokens}


def listed():
    named = lambda name, case: dict(case, name=name)
    return [
        # The smallest model, through the scheduler and the sampler: launches and host work are what it costs.
        named("generate_tiny_f32", _generate(5, (1, 300), 24)),
        # One user talking to a small model: the case that the reference quotes a bandwidth for.
        named("decode_1b_1", _step("llama_1b", 16, decodes=1, context=(2047, 2047))),
        # The headline: eight requests over 2,048 tokens each, the 8B shape.
        named("decode_8b_8", _step("llama_8b", 32, decodes=8, context=(2047, 2047))),
        # A busy server's decode step: 64 requests of all lengths.
        named("decode_8b_64", _step("llama_8b", 32, decodes=64, context=(509, 3585))),
        # The true 32-bit path decoding, for those who check numbers with it.
        named("decode_1b_f32_8", _step("llama_1b", 16, "float32", decodes=8, context=(200, 1800))),
        # A full step's worth of one prompt: the headline's other half.
        named("prompt_8b_2048", _step("llama_8b", 32, prompts=1, prompt=(2048, 2048))),
        # Several short prompts of uneven lengths that arrive together.
        named("prompts_1b_ragged", _step("llama_1b", 16, prompts=6, prompt=(17, 661))),
        # The 32-bit path over a prompt.
        named("prompt_1b_f32", _step("llama_1b", 16, "float32", prompts=1, prompt=(1023, 1023))),
        # Continuous batching on the 1B shape: many requests decode beside prompt portions, a step's budget full.
        named("serve_1b", _step("llama_1b", 16, decodes=160, context=(128, 4096), prompts=3, prompt=(331, 927))),
        # The 70B shape's mixed step (eight of its layers): 16 requests decode at 4,096 beside a prompt's second portion.
        named("mixed_70b", _step("llama_70b", 8, decodes=16, context=(4095, 4095), prompts=1, prompt=(2048, 2048), start=2048)),
        # A recurrent decoder: prompts, then single tokens.
        named("tuvodra_replay", _replay("tuvodra", 6, "bfloat16", 4, (389, 635), 12)),
        # A decoder with routed experts and differential attention, decoding.
        named("decode_tevovik_f32_8", _step("tevovik", 6, "float32", decodes=8, context=(200, 1000))),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    what = rng.choice(["decode_1b", "decode_8b", "decode_f32", "prompt_1b", "prompt_8b", "prompt_f32", "serve_1b", "mixed_70b", "tuvodra",
                       "tevovik", "generate"])
    between = lambda low, high: (lambda top: (max(low, int(top * rng.uniform(0.1, 1.0))), top))(_log(rng, low, high))
    if what in ("decode_1b", "decode_8b"):
        n = _log(rng, 1, 160 if what == "decode_1b" else 64)
        return _step("llama_" + what[-2:], 16 if what == "decode_1b" else 32, decodes=n, context=between(30, min(8000, 200000 // n)))
    if what == "decode_f32":
        return _step("llama_1b", 16, "float32", decodes=_log(rng, 1, 32), context=between(30, 2000))
    if what in ("prompt_1b", "prompt_8b"):
        n = rng.randint(1, 8)
        return _step("llama_" + what[-2:], 16 if what == "prompt_1b" else 32, prompts=n, prompt=between(9, 2048 // n))
    if what == "prompt_f32":
        n = rng.randint(1, 3)
        return _step("llama_1b", 16, "float32", prompts=n, prompt=between(9, 1023 // n))
    if what == "serve_1b":
        n = rng.randint(1, 4)
        return _step("llama_1b", 16, decodes=_log(rng, 4, 160), context=between(60, 4096), prompts=n, prompt=between(30, 1850 // n),
                     start=rng.choice([0, 0, rng.randint(1, 3000)]))
    if what == "mixed_70b":
        return _step("llama_70b", rng.choice([2, 4, 8]), decodes=_log(rng, 1, 16), context=between(60, 4000), prompts=1, prompt=between(100, 2048),
                     start=rng.choice([0, 2048, rng.randint(1, 3000)]))
    if what == "tuvodra":
        n = rng.randint(1, 6)
        return _replay("tuvodra", rng.choice([3, 6]), "bfloat16", n, between(9, 2048 // n), rng.randint(4, 16))
    if what == "tevovik":
        if rng.random() < 0.5:
            return _step("tevovik", rng.choice([3, 6]), "float32", decodes=_log(rng, 1, 16), context=between(30, 1000))
        return _step("tevovik", rng.choice([3, 6]), "float32", prompts=1, prompt=between(9, 400))
    return _generate(rng.randint(1, 8), between(1, 400), rng.randint(8, 48))


def _spread(n, low, high):
    """`n` lengths from `low` to `high`, long and short ones in turns."""
    even = [high if n == 1 else low + (high - low) * i // (n - 1) for i in range(n)]
    return even[0::2] + even[1::2][::-1]


def _lengths(case):
    """(tokens in the cache of each decoding request, tokens of each prompt)."""
    return (_spread(case["decodes"], case["context_from"], case["context_to"]) if case["kind"] == "step" else [],
            _spread(case["prompts"], case["prompt_from"], case["prompt_to"]))


# ---- weights and tokens, from the seed alone ----------------------------------------------------------------------------

# (mean, standard deviation) of what a tensor's name ends with; matrices and everything else: N(0, 0.02)
# (Llama's matrices that write into the stream are smaller by the square root of how often the deepest shape writes, and its table's
# rows large beside what a layer adds, as in models that train: with 0.02 everywhere a stack of 32 layers enlarges a rounding until
# logits of two correct implementations differ by 6 %.)
_NORMALS = {"llama": {"norm.weight": (1.0, 0.1), "layernorm.weight": (1.0, 0.1), "o_proj.weight": (0.0, 0.0016), "down_proj.weight": (0.0, 0.0016),
                      "embed_tokens.weight": (0.0, 0.5)},
            "tuvodra": {"norm1": (1.0, 0.1), "norm2": (1.0, 0.1), "final.norm": (1.0, 0.1), ".in": (0.3, 0.1), ".out": (1.0, 0.1),
                        "hc1.mix": (0.25, 0.1), "hc2.mix": (0.25, 0.1), "conv": (0.0, 0.3), "mix.dt": (0.0, 0.1), "dt.b": (-2.0, 0.5),
                        "A_log": (0.0, 0.5), "mix.D": (1.0, 0.1), "r1": (0.5, 0.2), "r2": (0.5, 0.05), "mix.in": (0.0, 0.02)},
            "tevovik": {"norm1": (0.0, 0.1), "norm2": (0.0, 0.1), "final.norm": (0.0, 0.1), "q.norm": (1.0, 0.1), "k.norm": (1.0, 0.1),
                        "lq1": (0.0, 0.1), "lk1": (0.0, 0.1), "lq2": (0.0, 0.1), "lk2": (0.0, 0.1), "router": (0.0, 0.1)}}


def _weight(model, seed, name, shape):
    """A tensor as a file would hold it (bfloat16), made on the GPU."""
    mean, std = 0.0, 0.02
    matched = 0
    for end, normal in _NORMALS[model.split("_")[0]].items():
        if name.endswith(end) and len(end) > matched:
            (mean, std), matched = normal, len(end)
    generator = torch.Generator(device="cuda").manual_seed(zlib.crc32(f"{seed}:{name}".encode()) + (seed << 32))
    return torch.empty(tuple(shape), dtype=torch.bfloat16, device="cuda").normal_(mean, std, generator=generator)


class _Weights:
    """The tensors of a model by name, each made when it is asked for."""

    def __init__(self, model, config, seed):
        from llm_rs_amd import Model
        self._model, self._seed = model, seed
        self._shapes = {name: tuple(spec.shape) for name, spec in Model(config.model_spec(), torch.bfloat16, "cpu").tensors().items()}

    def shapes(self):
        return dict(self._shapes)

    def __getitem__(self, name):
        return _weight(self._model, self._seed, name, self._shapes[name])

    def __iter__(self):
        return iter(self._shapes)

    def __len__(self):
        return len(self._shapes)


def _vocab(case):
    shape = _shape(case)
    return shape.get("vocab_size") or shape["vocab"]


def _sequences(case, seed):
    """Every token of the case: a list for each decoding request (its cache's tokens and the one it brings) and one for each
    prompt (what lies before the portion, the portion, and the tokens of a replay)."""
    contexts, prompts = _lengths(case)
    start = case.get("start", 0)
    more = case["tokens"] if case["kind"] == "replay" else 0
    lengths = [n + 1 for n in contexts] + [start + n + more for n in prompts]
    generator = torch.Generator().manual_seed(seed)
    flat = torch.randint(0, _vocab(case), (sum(lengths),), generator=generator).tolist()
    out, at = [], 0
    for n in lengths:
        out.append(flat[at:at + n])
        at += n
    return out[:len(contexts)], out[len(contexts):]


def prepare(case, seed):
    from llm_rs_amd import Engine, StepEntry, config_from_dict
    config = config_from_dict(_shape(case))
    contexts, prompts = _lengths(case)
    decoding, prompting = _sequences(case, seed)
    more = case.get("tokens", 0)
    pages = sum(-(-(len(s) + more + 1) // PAGE) for s in decoding + prompting) + 8
    if case["kind"] == "generate":
        pages += -(-case["prompt_to"] // PAGE)
    engine = Engine(config, _Weights(case["model"], config, seed), dtype=case["dtype"], device="cuda", page_size=PAGE, num_pages=pages,
                    max_requests=max(8, len(decoding) + len(prompting)), max_batch_tokens=STEP_TOKENS,
                    max_chunk=32 if case["kind"] == "generate" else 0)
    state = {"kind": case["kind"], "engine": engine, "seed": seed}
    if case["kind"] == "generate":
        state.update(prompts=prompting, tokens=case["tokens"], seeds=[seed + i for i in range(len(prompting))])
        return state
    if case["kind"] == "replay":
        n = case["tokens"]
        state.update(prompts=[s[:-n] for s in prompting], following=[[s[len(s) - n + j] for s in prompting] for j in range(n)])
        return state

    def fill(slot, tokens):
        for at in range(0, len(tokens), STEP_TOKENS):
            engine.step([StepEntry(slot, at, tokens[at:at + STEP_TOKENS], [])])

    entries = []
    for tokens in decoding:
        slot = engine.open_request()
        fill(slot, tokens[:-1])
        entries.append(StepEntry(slot, len(tokens) - 1, tokens[-1:], [0]))
    start = case["start"]
    for tokens in prompting:
        slot = engine.open_request()
        fill(slot, tokens[:start])
        entries.append(StepEntry(slot, start, tokens[start:], [len(tokens) - start - 1]))
    state["entries"] = entries
    return state


def run(state):
    engine = state["engine"]
    if state["kind"] == "step":
        return engine.step(state["entries"])
    from llm_rs_amd import StepEntry
    if state["kind"] == "generate":
        tokens = engine.generate(state["prompts"], max_new_tokens=state["tokens"], temperature=0.8, top_k=40, top_p=0.9, seed=state["seeds"])
        slot, prompt = engine.open_request(), state["prompts"][-1]
        logits = engine.step([StepEntry(slot, 0, prompt, list(range(len(prompt))))])
        engine.close_request(slot)
        return {"tokens": torch.tensor(tokens), "logits": logits}
    slots = [engine.open_request() for _ in state["prompts"]]
    places = [len(p) for p in state["prompts"]]
    out = [engine.step([StepEntry(s, 0, p, [len(p) - 1]) for s, p in zip(slots, state["prompts"])]).clone()]
    for j, tokens in enumerate(state["following"]):
        out.append(engine.step([StepEntry(s, n + j, [t], [0]) for s, n, t in zip(slots, places, tokens)]).clone())
    for slot in slots:
        engine.close_request(slot)
    return out


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------

def _layer_weights(case):
    """(matrix elements of one layer that every token passes, elements of one expert, experts, experts a token uses), averaged over
    the layers."""
    if case["model"] == "tuvodra":
        mingru = 4 * 2048 * 2048
        mamba = 2048 * 8192 + 4096 * 160 + 4096 * 128 + 4096 * 2048
        attention = 2048 * (2048 + 512 + 512) + 2048 * 2048 + 3 * 2048 * 8192
        return (mingru + mamba + attention) / 3, 0, 0, 0
    if case["model"] == "tevovik":
        # (a layer of three has no k and v matrices of its own)
        return 2048 * 2048 * 2 + 2048 * (512 + 512) * 2 / 3 + 2048 * 32, 3 * 2048 * 2048, 16, 4
    d = _shape(case)
    q, kv = d["num_attention_heads"] * d["head_dim"], d["num_key_value_heads"] * d["head_dim"]
    return d["hidden_size"] * (2 * q + 2 * kv + 3 * d["intermediate_size"]), 0, 0, 0


def _attention_widths(case):
    """(attention layers, query width, numbers a token leaves in the cache of one layer that has one, layers with a cache, window)."""
    if case["model"] == "tuvodra":
        return case["layers"] // 3, 2048, 1024, case["layers"] // 3, 1024
    if case["model"] == "tevovik":
        return case["layers"], 2048, 1024, case["layers"] * 2 // 3, 4096
    d = _shape(case)
    return (case["layers"], d["num_attention_heads"] * d["head_dim"], 2 * d["num_key_value_heads"] * d["head_dim"], case["layers"], 1 << 30)


def _step_work(case, entries, wanted):
    """One step of `entries` = (start, tokens) with `wanted` rows of logits."""
    size = 2 if case["dtype"] == "bfloat16" else 4
    d = _shape(case)
    hidden = d.get("hidden_size") or d["width"]
    dense, expert, experts, top = _layer_weights(case)
    T = sum(n for _, n in entries)
    touched = experts * (1.0 - (1.0 - top / experts) ** T) if experts else 0.0
    weights = case["layers"] * (dense + touched * expert) + _vocab(case) * hidden
    layers, q_width, cached, with_cache, window = _attention_widths(case)
    pairs = sum(sum(min(s + i + 1, window) for i in range(n)) for s, n in entries)          # (query, key) pairs of a layer
    read = sum(min(s, window) for s, _ in entries)
    bytes_ = size * (weights + T * hidden + with_cache * cached * (read + T)) + 4 * wanted * _vocab(case)
    flops = 2 * T * case["layers"] * (dense + top * expert) + 4 * layers * q_width * pairs + 2 * wanted * hidden * _vocab(case)
    return bytes_, flops


def work(case):
    contexts, prompts = _lengths(case)
    if case["kind"] == "step":
        steps = [([(n, 1) for n in contexts] + [(case["start"], n) for n in prompts], len(contexts) + len(prompts))]
    else:       # prompts together, then a token each at a time
        steps = [([(0, n) for n in prompts], len(prompts))]
        steps += [([(n + j, 1) for n in prompts], len(prompts)) for j in range(case["tokens"] - (case["kind"] == "generate"))]
        if case["kind"] == "generate":
            steps.append(([(0, prompts[-1])], prompts[-1]))
    each = [_step_work(case, entries, wanted) for entries, wanted in steps]
    return {"bytes": float(sum(b for b, _ in each)), "flops": float(sum(f for _, f in each))}


def tolerance(case):
    # 32-bit: sums of thousands of products in another order, through the layers: up to 1.2e-5 off the 64-bit result.
    # bfloat16: every activation that passes through memory rounded to 8 bits, through up to 32 layers: up to 0.7 % off.
    if case["dtype"] == "float32":
        return {"rel": 5e-5, "differ": 0.01}
    return {"rel": 0.025}


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------------

EXACT_MAX_FLOPS = 3.0e14        # some seconds of 64-bit products


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softmax_heads(q, k, v, scale, bias):
    """q [T, heads, d], k [T, kv_heads, d], v [T, kv_heads, dv]; `bias(head)` is added to the scores [T, T] of a head."""
    T, heads, _ = q.shape
    out = torch.empty(T, heads, v.shape[2], dtype=q.dtype, device=q.device)
    for a in range(heads):
        g = a // (heads // k.shape[1])
        scores = (q[:, a].contiguous() @ k[:, g].contiguous().T) * scale + bias(a)
        out[:, a] = torch.softmax(scores, dim=-1) @ v[:, g].contiguous()
    return out


def _mask(T, size, chunked):
    """0 where a position sees another, -inf elsewhere: the last `size` positions, or those of its own stretch of `size`."""
    i = torch.arange(T, device="cuda")
    seen = i[None, :] <= i[:, None]
    seen &= (i[None, :] // size == i[:, None] // size) if chunked else (i[:, None] - i[None, :] < size)
    return torch.where(seen, 0.0, -math.inf).double()


def _llama_exact(case, get, sequences, wants):
    d = _shape(case)
    D, H, KV, hd, F = d["hidden_size"], d["num_attention_heads"], d["num_key_value_heads"], d["head_dim"], d["intermediate_size"]
    eps, s = d["rms_norm_eps"], d["rope_scaling"]
    # the angles are a table of the model: frequencies in 32 bits, times the position in 32 bits
    freq = d["rope_theta"] ** (-torch.arange(hd // 2, dtype=torch.float64) * 2.0 / hd)
    wave, L = 2.0 * math.pi / freq, s["original_max_position_embeddings"]
    blend = (L / wave - s["low_freq_factor"]) / (s["high_freq_factor"] - s["low_freq_factor"])
    freq = torch.where(wave < L / s["high_freq_factor"], freq,
                       torch.where(wave > L / s["low_freq_factor"], freq / s["factor"], (1.0 - blend) * freq / s["factor"] + blend * freq))
    longest = max(len(t) for t in sequences)
    angle = (torch.arange(longest, dtype=torch.float32)[:, None] * freq.float()[None, :]).double().cuda()
    cos, sin = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]

    def rotate(x):
        a, b, c, n = x[..., :hd // 2], x[..., hd // 2:], cos[:len(x)], sin[:len(x)]
        return torch.cat([a * c - b * n, b * c + a * n], dim=-1)

    table = get("model.embed_tokens.weight", (d["vocab_size"], D))
    xs = [table[torch.tensor(t, device="cuda")].double() for t in sequences]
    for i in range(case["layers"]):
        at = lambda leaf, *shape: get(f"model.layers.{i}.{leaf}.weight", shape).double()
        n1, n2 = at("input_layernorm", D), at("post_attention_layernorm", D)
        wq, wk, wv, wo = at("self_attn.q_proj", H * hd, D), at("self_attn.k_proj", KV * hd, D), at("self_attn.v_proj", KV * hd, D), at("self_attn.o_proj", D, H * hd)
        gate, up, down = at("mlp.gate_proj", F, D), at("mlp.up_proj", F, D), at("mlp.down_proj", D, F)
        for j, x in enumerate(xs):
            T, h = len(x), _rms(x, eps) * n1
            mask = _mask(T, T, False)
            o = _softmax_heads(rotate((h @ wq.T).view(T, H, hd)), rotate((h @ wk.T).view(T, KV, hd)), (h @ wv.T).view(T, KV, hd), hd ** -0.5, lambda a: mask)
            x = x + o.reshape(T, H * hd) @ wo.T
            h = _rms(x, eps) * n2
            xs[j] = x + (_silu(h @ gate.T) * (h @ up.T)) @ down.T
        del wq, wk, wv, wo, gate, up, down
    head = table if d["tie_word_embeddings"] else get("lm_head.weight", (d["vocab_size"], D))
    norm, head = get("model.norm.weight", (D,)).double(), head.double()
    return [(_rms(x[w], eps) * norm) @ head.T for x, w in zip(xs, wants)]


def _tuvodra_exact(case, get, sequences, wants):
    d = _shape(case)
    D, S, eps, groups = d["width"], d["streams"], d["norm"]["eps"], d["norm"]["groups"]
    normed = lambda x, w: _rms(x.reshape(len(x), groups, D // groups), eps).reshape(len(x), D) * w
    table = get("embed", (d["vocab"], D)).double()
    xs = [table[torch.tensor(t, device="cuda")][None].repeat(S, 1, 1) for t in sequences]

    def mingru(h, at):
        z, u = torch.sigmoid(h @ at("z", D, D).T + at("z.b", D)), h @ at("x", D, D).T + at("x.b", D)
        cand, keep = z * torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), 1.0 - z
        s, rows = torch.zeros(D, dtype=h.dtype, device=h.device), torch.empty_like(z)
        for t in range(len(h)):
            s = keep[t] * s + cand[t]
            rows[t] = s
        return (rows * _silu(h @ at("g", D, D).T)) @ at("o", D, D).T

    def mamba(h, at, m):
        C, N, K, R = m["inner"], m["state"], m["conv"], m["dt_rank"]
        T = len(h)
        x, g = (h @ at("in", 2 * C, D).T).split(C, dim=1)
        taps = at("conv", C, K)
        padded = torch.cat([torch.zeros(K - 1, C, dtype=h.dtype, device=h.device), x])
        x = _silu(sum(padded[j:j + T] * taps[:, j] for j in range(K)) + at("conv.b", C))
        delta, B, Cs = (x @ at("x", R + 2 * N, C).T).split([R, N, N], dim=1)
        step = torch.nn.functional.softplus(delta @ at("dt", C, R).T + at("dt.b", C))
        A, taken = -torch.exp(at("A_log", C, N)), step * x
        state, rows = torch.zeros(C, N, dtype=h.dtype, device=h.device), torch.empty_like(x)
        for t in range(T):
            state = torch.exp(step[t][:, None] * A) * state + taken[t][:, None] * B[t]
            rows[t] = state @ Cs[t]
        return ((rows + at("D", C) * x) * _silu(g)) @ at("o", D, C).T

    def attention(h, at, m):
        T, H, G, dim = len(h), m["heads"], m["kv_heads"], m["dim"]
        q = _rms((h @ at("q", H * dim, D).T + at("q.b", H * dim)).view(T, H, dim), eps)
        k = _rms((h @ at("k", G * dim, D).T + at("k.b", G * dim)).view(T, G, dim), eps)
        v = (h @ at("v", G * dim, D).T + at("v.b", G * dim)).view(T, G, dim)
        r1, r2, i = at("r1", H), at("r2", H), torch.arange(T, device="cuda")
        mask, far = _mask(T, m["mask"]["size"], False), (i[:, None] - i[None, :]).clamp(min=0).double()
        o = _softmax_heads(q, k, v, m["scale"], lambda a: mask - r1[a] * torch.log1p(r2[a] * far))
        return o.reshape(T, H * dim) @ at("o", D, H * dim).T

    def feed_forward(h, at, m):
        return (_silu(h @ at("gate", m["ff"], D).T) * (h @ at("up", m["ff"], D).T)) @ at("down", D, m["ff"]).T

    for i, layer in enumerate(d["layers"]):
        mixer = {"mingru": lambda h, at, m: mingru(h, at), "mamba1": mamba, "attention": attention}[layer["type"]]
        halves = [("mix", "hc1", "norm1", mixer, layer["mixer"])] + ([("mlp", "hc2", "norm2", feed_forward, layer["mlp"])] if layer["mlp"] else [])
        for part, link, norm, sublayer, sizes in halves:
            at = lambda leaf, *shape: get(f"l{i}.{part}.{leaf}", shape).double()
            w_in, w_out, mix = (get(f"l{i}.{link}.{n}", shape).double() for n, shape in (("in", (S,)), ("out", (S,)), ("mix", (S, S))))
            weight = get(f"l{i}.{norm}", (D,)).double()
            for j, x in enumerate(xs):
                y = sublayer(normed((w_in[:, None, None] * x).sum(0), weight), at, sizes)
                xs[j] = (mix.T @ x.reshape(S, -1)).view_as(x) + w_out[:, None, None] * y
    final = get("final.norm", (D,)).double()
    return [normed(x.sum(0)[w], final) @ table.T for x, w in zip(xs, wants)]


def _tevovik_exact(case, get, sequences, wants):
    d = _shape(case)
    D, eps = d["width"], d["norm"]["eps"]
    table = get("embed", (d["vocab"], D)).double()
    rate = 10000.0 ** (-2.0 * torch.arange(D // 2, dtype=torch.float64, device="cuda") / D)
    xs = []
    for t in sequences:
        angle = torch.arange(len(t), dtype=torch.float64, device="cuda")[:, None] * rate
        xs.append(table[torch.tensor(t, device="cuda")] * d["embedding"]["scale"] + torch.stack([torch.sin(angle), torch.cos(angle)], dim=-1).view(len(t), D))
    kept = {}
    for i, layer in enumerate(d["layers"]):
        m, f = layer["mixer"], layer["mlp"]
        H, G, dim, dv, F = m["heads"], m["kv_heads"], m["dim"], m["vdim"], f["expert"]["ff"]
        router, E, top = f["router"], f["router"]["experts"], f["router"]["top"]
        at = lambda leaf, *shape: get(f"l{i}.mix.{leaf}", shape).double()
        lam = torch.exp((at("lq1", dim) * at("lk1", dim)).sum()) - torch.exp((at("lq2", dim) * at("lk2", dim)).sum()) + m["diff"]
        norm1, norm2 = 1.0 + get(f"l{i}.norm1", (D,)).double(), 1.0 + get(f"l{i}.norm2", (D,)).double()
        w_route = get(f"l{i}.mlp.router", (E, D)).double()
        experts = [tuple(get(f"l{i}.mlp.e{e}.{n}", (D, F) if n == "down" else (F, D)).double() for n in ("gate", "up", "down")) for e in range(E)]
        for j, x in enumerate(xs):
            T = len(x)
            q = _rms((x @ at("q", 2 * H * dim, D).T).view(T, 2 * H, dim), eps) * at("q.norm", dim)
            if m.get("kv_from") is None:
                kept[i, j] = (_rms((x @ at("k", 2 * G * dim, D).T).view(T, 2 * G, dim), eps) * at("k.norm", dim), (x @ at("v", G * dv, D).T).view(T, G, dv))
            k, v = kept[m.get("kv_from", i), j]
            mask = _mask(T, m["mask"]["size"], True)
            maps = [_softmax_heads(q[:, half::2], k[:, half::2], v, m["scale"], lambda a: mask) for half in range(2)]
            o = _rms(maps[0] - lam * maps[1], eps) * (1.0 - m["diff"]) * torch.sigmoid(x @ at("g", H, D).T)[:, :, None]
            x = x + _rms(o.reshape(T, H * dv) @ at("o", D, H * dv).T, eps) * norm1
            scores = torch.softmax(x @ w_route.T, dim=-1)
            count, keep = router["groups"]["count"], router["groups"]["keep"]
            best = scores.view(T, count, E // count).amax(dim=2).topk(keep, dim=1).indices
            open_to = torch.zeros(T, count, device="cuda").scatter_(1, best, 1.0).repeat_interleave(E // count, dim=1)
            chosen = scores.masked_fill(open_to == 0, -1.0).topk(top, dim=1).indices
            y = torch.zeros_like(x)
            for e, (gate, up, down) in enumerate(experts):
                rows = (chosen == e).any(dim=1).nonzero()[:, 0]
                if len(rows):
                    y[rows] += (_silu(x[rows] @ gate.T) * (x[rows] @ up.T) * scores[rows, e:e + 1]) @ down.T
            xs[j] = x + _rms(y, eps) * norm2
    final, head = 1.0 + get("final.norm", (D,)).double(), get("head", (d["vocab"], D)).double()
    return [(_rms(x[w], eps) * final) @ head.T for x, w in zip(xs, wants)]


def exact(case, seed):
    decoding, prompting = _sequences(case, seed)
    sequences = decoding + prompting
    whole = _step_work(case, [(0, len(t)) for t in sequences], 1)[1]
    if whole > EXACT_MAX_FLOPS:
        return None
    get = lambda name, shape: _weight(case["model"], seed, name, shape)
    of = {"tuvodra": _tuvodra_exact, "tevovik": _tevovik_exact}.get(case["model"], _llama_exact)
    if case["kind"] == "generate":      # (which tokens are drawn is no computed number)
        return {"tokens": None, "logits": of(case, get, prompting[-1:], [list(range(len(prompting[-1])))])[0]}
    if case["kind"] == "replay":
        n = case["tokens"]
        rows = of(case, get, sequences, [list(range(len(t) - n - 1, len(t))) for t in sequences])
        return [torch.stack([r[j] for r in rows]) for j in range(n + 1)]
    return torch.cat(of(case, get, sequences, [[-1] for _ in sequences]))
