"""The Tuvodra decoder in the engine against the plain decoder (plain_tuvodra.py): every mechanism alone, the replay
regimes (whole prompts, decoding through the cache and the state, portions, mixed batches under a pool and slots that
are used again), inputs made so that a window's edge, a far key or a long-held state shows in the logits, long
decoding, and greedy generation through the scheduler."""
from __future__ import annotations

import pytest
import torch

from llm_rs_amd import Engine, StepEntry
from llm_rs_amd.engine.trace import TraceReplayer
from plain_tuvodra import plain_group_rmsnorm, plain_tuvodra_logits
from replay_cases import collect, live_token_need, mixed, portions, random_tokens, tail_decoded, whole
from tuvodra_cases import (CONFIGS, PAGE_SIZE, allowed_error, attention, check_rows, config, make_model, mamba1, mingru,
                           one_layer, reference)

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]


def replay(engine, steps):
    replayer = TraceReplayer.for_engine(engine)
    outputs = []
    for step in steps:
        out = replayer.step(step)
        outputs.append(None if out is None else torch.from_numpy(out.copy()))
    return collect(steps, outputs)


def engine_for(typed, tensors, dtype, page_size, tokens, max_requests=4):
    return Engine(typed, tensors, dtype=dtype, page_size=page_size, num_pages=max(-(-tokens // page_size), 1), max_requests=max_requests)


def run_regimes(cfg, typed, tensors, dtype, page_size, requests, regimes):
    exact = reference(cfg, tensors, requests)
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    for name, steps in regimes.items():
        eng = engine_for(typed, tensors, dtype, page_size, live_token_need(steps, 64))
        check_rows(replay(eng, steps), exact, requests, allowed, name)


# ---- each mechanism alone -----------------------------------------------------------------------------------------

ALONE = {
    "mingru": mingru(28),
    "mingru+ff": mingru(44, ff=72),
    "mamba1": mamba1(36, 6, 3, 4),
    "mamba1 one tap": mamba1(20, 9, 1, 2, ff=24),
    "mamba1 many states": mamba1(12, 130, 2, 5),
    "mamba1 many taps": mamba1(20, 3, 9, 2),
    "mamba1 six taps": mamba1(28, 2, 6, 1, ff=16),
    "attention": attention(4, 2, 12, 12, 0.4, 7),
    "attention wide values": attention(3, 3, 8, 24, 1.3, 50, ff=32),
    "attention narrow values, one kv head": attention(5, 1, 20, 4, 0.05, 3),
    "attention window of one": attention(2, 2, 16, 16, 0.25, 1),
    "attention, heads of 32 in fours": attention(4, 1, 32, 32, 0.2, 21),
    "attention, heads of 128": attention(6, 2, 128, 128, 0.09, 70, ff=48),
    "attention, heads of 64, window of a page": attention(8, 4, 64, 64, 0.11, 16),
    "attention, heads of 64 in threes": attention(6, 2, 64, 64, 0.13, 29),
    "attention, heads of 32, fourteen to a key head": attention(14, 1, 32, 32, 0.3, 40),
    "attention, heads of 96": attention(4, 2, 96, 96, 0.1, 23),
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("which", list(ALONE))
def test_one_layer_of_each_kind(which, dtype):
    for streams, groups in ((1, 1), (2, 4), (5, 2)):
        cfg = one_layer(ALONE[which], streams=streams, groups=groups)
        typed, tensors = make_model(cfg, seed=streams)
        requests = {"a": random_tokens(cfg["vocab"], 45, 1), "b": random_tokens(cfg["vocab"], 3, 2)}
        run_regimes(cfg, typed, tensors, dtype, 4, requests,
                    {"whole": whole(requests), "decoded": tail_decoded(requests, tail=20), "portions": portions(requests, (2, 5, 2, 9, 3))})


# ---- whole models in every regime -----------------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("which", list(CONFIGS))
def test_replay_regimes(which, dtype):
    cfg = CONFIGS[which]
    typed, tensors = make_model(cfg, seed=3)
    lengths = [1, 2, 23, 70, 131, 40, 17]          # more requests than slots: slots and pages are used again
    requests = {f"r{i}": random_tokens(cfg["vocab"], n, 10 + i) for i, n in enumerate(lengths)}
    run_regimes(cfg, typed, tensors, dtype, PAGE_SIZE[which], requests,
                {"whole": whole(requests), "decoded": tail_decoded(requests, tail=32), "portions": portions(requests),
                 "portions of two and three": portions(requests, (2, 3)), "mixed": mixed(requests, live=4),
                 "mixed, two live": mixed(requests, live=2, prefill_sizes=(2, 31, 4))})


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_batch_of_unequal_requests_equals_each_alone(dtype):
    cfg = CONFIGS["odd"]
    typed, tensors = make_model(cfg, seed=5)
    requests = {"long": random_tokens(cfg["vocab"], 90, 1), "short": random_tokens(cfg["vocab"], 2, 2),
                "one": random_tokens(cfg["vocab"], 1, 3), "mid": random_tokens(cfg["vocab"], 33, 4)}
    eng = engine_for(typed, tensors, dtype, 4, 4 * 128)
    together = [{"step": 0, "entries": [{"id": r, "tokens": t, "want": list(range(len(t)))} for r, t in requests.items()], "end": list(requests)}]
    rows_together = replay(eng, together)
    rows_alone = replay(eng, whole(requests))        # the same engine: the slots and pages of the batch, used again
    exact = reference(cfg, tensors, requests)
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    check_rows(rows_together, exact, requests, allowed, "together")
    check_rows(rows_alone, exact, requests, allowed, "alone")
    for rid, toks in requests.items():            # and beyond rounding, being in a batch changes nothing
        for p in range(len(toks)):
            d = float((rows_together[rid][p] - rows_alone[rid][p]).abs().max()) / float(exact[rid].abs().max())
            assert d <= allowed, (rid, p, d)


# ---- inputs under which an edge shows ------------------------------------------------------------------------------

def marked_attention_model(window, dim=16, vdim=12, heads=2, kv_heads=1, scale=2.0, width=32, vocab=50, mark=7):
    """One attention layer in which the key of token `mark` stands out for every query: q's bias points where that
    key points, so the marked key scores scale * dim and any other key about scale * sqrt(dim) * N(0, 1); with the
    marked token inside the window the output is its value, outside it a mix of the others."""
    cfg = config(width, vocab, 2, 2, 4.0, [attention(heads, kv_heads, dim, vdim, scale, window)])

    def change(t):
        x = t["embed"].double()[mark] * 4.0 * float(t["l0.hc1.in"].double().sum())
        h = plain_group_rmsnorm(x, t["l0.norm1"].double(), 1e-5, 2)
        key = (t["l0.mix.k"].double() @ h + t["l0.mix.k.b"].double()).reshape(kv_heads, dim)
        t["l0.mix.q.b"] = (50.0 * key.repeat_interleave(heads // kv_heads, dim=0).reshape(-1)).to(torch.bfloat16)
        t["l0.mix.v"] = (t["l0.mix.v"].double() * 20.0).to(torch.bfloat16)      # values that tell tokens apart in the logits
        t["l0.mix.o"] = (t["l0.mix.o"].double() * 20.0).to(torch.bfloat16)
    typed, tensors = make_model(cfg, seed=11, change=change)
    return cfg, typed, tensors


def sequence_with_mark(vocab, n, at, mark, seed):
    toks = [t if t != mark else (t + 1) % vocab for t in random_tokens(vocab, n, seed)]
    toks[at] = mark
    return toks


# head shapes: values narrower than keys (the kernel for any sizes) and heads the matrix-core kernels take
HEAD_SHAPES = {"any sizes": dict(dim=16, vdim=12, heads=2, kv_heads=1, width=32), "matrix cores": dict(dim=64, vdim=64, heads=4, kv_heads=2, width=64)}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", list(HEAD_SHAPES))
@pytest.mark.parametrize("window,at", [(9, 3), (16, 0), (17, 15), (33, 16), (40, 31), (64, 1), (65, 30)])
def test_a_key_just_inside_and_just_outside_the_window(window, at, shape, dtype):
    cfg, typed, tensors = marked_attention_model(window, **HEAD_SHAPES[shape])
    toks = sequence_with_mark(cfg["vocab"], at + window + 6, at, 7, seed=window)
    requests = {"m": toks}
    exact = reference(cfg, tensors, requests)
    inside, outside = at + window - 1, at + window
    # the plain decoder itself: the marked key's leaving the window moves the logits by much more than any bound below
    gap = float((exact["m"][inside] - exact["m"][outside]).abs().max()) / float(exact["m"].abs().max())
    unmarked = {"m": [t if i != at else (t + 2) % cfg["vocab"] for i, t in enumerate(toks)]}
    moved = float((reference(cfg, tensors, unmarked)["m"][inside] - exact["m"][inside]).abs().max()) / float(exact["m"].abs().max())
    assert gap > 0.05 and moved > 0.05, (gap, moved)
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    assert allowed < min(gap, moved) / 2, (allowed, gap, moved)
    regimes = {"whole": whole(requests), "decoded over the edge": tail_decoded(requests, tail=8),
               "portions of two": portions(requests, (2,)), "a portion that ends inside": portions(requests, (inside + 1, 1, 2)),
               "a portion that starts outside": portions(requests, (outside, 3))}
    for name, steps in regimes.items():
        eng = engine_for(typed, tensors, dtype, 16, 256)
        check_rows(replay(eng, steps), exact, requests, allowed, name)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", list(HEAD_SHAPES))
def test_a_far_key_among_hundreds_across_pages(shape, dtype):
    cfg, typed, tensors = marked_attention_model(window=1000, **HEAD_SHAPES[shape])
    for at in (0, 15, 16, 250):
        toks = sequence_with_mark(cfg["vocab"], 600, at, 7, seed=at)
        requests = {"m": toks}
        exact = reference(cfg, tensors, requests)
        unmarked = {"m": [t if i != at else (t + 2) % cfg["vocab"] for i, t in enumerate(toks)]}
        moved = float((reference(cfg, tensors, unmarked)["m"][599] - exact["m"][599]).abs().max()) / float(exact["m"].abs().max())
        assert moved > 0.05, moved
        allowed = allowed_error(dtype, cfg, tensors, requests, exact)
        for name, steps in {"whole": whole(requests), "decoded": tail_decoded(requests, tail=40),
                            "portions": portions(requests, (64, 3, 130, 2))}.items():
            eng = engine_for(typed, tensors, dtype, 16, 640)
            check_rows(replay(eng, steps), exact, requests, allowed, f"mark at {at}, {name}")


def held_state(t, dt_rank=2):
    """Two marked tokens (the last two ids) carry features that no other token has: feature 0 opens the recurrence
    for them (a gate near 1, an input many times the others'), feature 1 tells them apart; every other token leaves
    the state nearly as it was (gates near 0, slow decay), and what reads the state is made large enough to show."""
    e = t["embed"].double()
    e[:, 0:2] = 0.0
    e[-2, 0], e[-2, 1], e[-1, 0], e[-1, 1] = 1.0, 1.0, 1.0, -1.0
    t["embed"] = e.to(torch.bfloat16)
    g = torch.Generator().manual_seed(0)
    signs = lambda n: torch.sign(torch.randn(n, generator=g, dtype=torch.float64))
    for name in list(t):
        w = t[name].double()
        if name.endswith(".mix.z.b"): w = torch.full_like(w, -12.0)
        elif name.endswith(".mix.z"): w[:, 0] = 8.0
        elif name.endswith(".mix.x") and w.shape[1] == e.shape[1]: w[:, 1] = signs(w.shape[0]) * 3.0      # minGRU's candidate
        elif name.endswith(".mix.x"): w[dt_rank:] *= 20                                                   # the scan's B and C
        elif name.endswith((".mix.g", ".mix.o")): w = w * 20
        elif name.endswith(".mix.in"):
            C = w.shape[0] // 2
            w[C:] *= 20
            w[:C, 0] = 5.0
            w[:C, 1] = signs(C) * 2.0
        elif name.endswith(".mix.conv"): w = w.abs()
        elif name.endswith(".mix.dt.b"): w = torch.full_like(w, -3.0)
        elif name.endswith(".mix.A_log"): w = torch.full_like(w, -5.0)
        else: continue
        t[name] = w.to(torch.bfloat16)


def long_memory(t):
    """Gates and step sizes so small that a state holds what it saw long ago."""
    for name in t:
        if name.endswith(".mix.z.b"):
            t[name] = torch.full_like(t[name], -5.0)
        if name.endswith(".mix.dt.b"):
            t[name] = torch.full_like(t[name], -6.0)
        if name.endswith(".mix.A_log"):
            t[name] = torch.full_like(t[name], -3.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("layer", ["mingru", "mamba1"])
def test_the_first_token_is_still_in_the_state_after_hundreds(layer, dtype):
    cfg = one_layer(mingru(24) if layer == "mingru" else mamba1(24, 4, 3, 2), width=32, vocab=40)
    typed, tensors = make_model(cfg, seed=2, change=held_state)
    toks = [38] + [t % 38 for t in random_tokens(40, 299, 9)]
    other = [39] + toks[1:]
    requests = {"a": toks, "b": other}
    exact = reference(cfg, tensors, requests)
    moved = float((exact["a"][299] - exact["b"][299]).abs().max()) / float(exact["a"].abs().max())
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    assert moved > 0.05 and allowed < moved / 2, (moved, allowed)          # what the first token was still shows at the end
    for name, steps in {"whole": whole(requests), "decoded": tail_decoded(requests, tail=64), "portions": portions(requests, (2, 97, 3, 50)),
                        "both at once": mixed(requests, live=2, prefill_sizes=(40, 2, 7))}.items():
        eng = engine_for(typed, tensors, dtype, 16, 1024)
        check_rows(replay(eng, steps), exact, requests, allowed, name)


@pytest.fixture
def chunk_length(request):
    from llm_rs_amd.kernels import kernels
    kernels().scan_set_chunk(request.param)
    yield request.param
    kernels().scan_set_chunk(0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chunk_length", [32, 64], indirect=True)
@pytest.mark.parametrize("layer", ["mingru", "mamba1", "mamba1 many states"])
def test_portions_longer_than_a_chunk_of_the_recurrences(layer, chunk_length, dtype):
    """Entries of 64 tokens and more run their recurrences in chunks side by side: lengths at the chunks' edges, side
    by side with short entries in one step, portions that start in the middle of a sequence, and a state (slow gates,
    slow decay) in which everything before still counts."""
    mixer = {"mingru": mingru(70), "mamba1": mamba1(72, 5, 4, 3), "mamba1 many states": mamba1(10, 70, 2, 2)}[layer]
    cfg = one_layer(mixer, width=32, vocab=40)
    typed, tensors = make_model(cfg, seed=8, change=long_memory)
    lengths = {"a": 64, "b": 65, "c": 128, "d": 129, "e": 200, "f": 1, "g": 3, "h": 321}
    requests = {r: random_tokens(40, n, 20 + i) for i, (r, n) in enumerate(lengths.items())}
    exact = reference(cfg, tensors, requests)
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    together = [{"step": 0, "entries": [{"id": r, "tokens": t, "want": list(range(len(t)))} for r, t in requests.items()], "end": list(requests)}]
    eng = engine_for(typed, tensors, dtype, 16, sum(-(-n // 16) * 16 for n in lengths.values()), max_requests=8)
    check_rows(replay(eng, together), exact, requests, allowed, "together")
    for name, steps in {"whole": whole(requests), "portions": portions(requests, (3, 66, 2, 127, 64, 65)),
                        "mixed": mixed(requests, live=3, prefill_sizes=(70, 2, 130))}.items():
        eng = engine_for(typed, tensors, dtype, 16, live_token_need(steps, 64))
        check_rows(replay(eng, steps), exact, requests, allowed, name)


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_slot_used_again_starts_from_nothing(dtype):
    cfg = CONFIGS["plain"]
    typed, tensors = make_model(cfg, seed=4, change=long_memory)
    first, second = random_tokens(cfg["vocab"], 50, 1), random_tokens(cfg["vocab"], 30, 2)
    eng = Engine(typed, tensors, dtype=dtype, page_size=16, num_pages=8, max_requests=1)      # one slot, pages for one request
    exact = reference(cfg, tensors, {"first": first, "second": second})
    allowed = allowed_error(dtype, cfg, tensors, {"first": first, "second": second}, exact)
    for rid, toks in (("first", first), ("second", second), ("first", first)):
        slot = eng.open_request()
        assert slot == 0
        head = eng.step([StepEntry(slot, 0, toks[:20], list(range(20)))]).cpu().clone()
        tail = eng.step([StepEntry(slot, 20, toks[20:], list(range(len(toks) - 20)))]).cpu()
        eng.close_request(slot)
        got = torch.cat([head, tail]).double()
        err = float((got - exact[rid]).abs().max()) / float(exact[rid].abs().max())
        assert err <= allowed, (rid, err, allowed)


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding_with_recorded_steps(dtype):
    cfg = CONFIGS["odd"]
    typed, tensors = make_model(cfg, seed=6)
    requests = {"a": random_tokens(cfg["vocab"], 330, 1), "b": random_tokens(cfg["vocab"], 321, 2)}
    exact = reference(cfg, tensors, requests)
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    steps = [{"step": 0, "entries": [{"id": r, "tokens": t[:9], "want": list(range(9))} for r, t in requests.items()], "end": []}]
    for i in range(9, 330):
        live = [r for r, t in requests.items() if i < len(t)]
        steps.append({"step": len(steps), "entries": [{"id": r, "tokens": [requests[r][i]], "want": [0]} for r in live],
                      "end": [r for r in live if i == len(requests[r]) - 1]})
    eng = engine_for(typed, tensors, dtype, 4, 704)
    check_rows(replay(eng, steps), exact, requests, allowed, "decoding")
    assert eng.runner.graph_replays > 100           # the single-token steps were recorded and replayed


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("streams,width,groups", [(5, 42, 3), (2, 40, 2), (4, 36, 1), (1, 44, 2)])
def test_steps_of_many_rows_mix_the_streams_inside_the_next_norm(streams, width, groups, dtype):
    """From 128 rows on, a sublayer's mix of the streams runs in the launch of the norm that reads them next: rows of
    a length that is and is not a multiple of four, few and many streams, steps just below and above that bound."""
    cfg = config(width, 53, streams, groups, 1.5, [mingru(24, ff=32), attention(2, 1, 8, 8, 0.5, 11), mamba1(16, 3, 2, 2, ff=20)])
    typed, tensors = make_model(cfg, seed=streams)
    requests = {"a": random_tokens(53, 127, 1), "b": random_tokens(53, 128, 2), "c": random_tokens(53, 300, 3)}
    run_regimes(cfg, typed, tensors, dtype, 16, requests,
                {"whole": whole(requests), "portions": portions(requests, (128, 2, 129, 41))})


@pytest.mark.parametrize("rows,streams,width,groups", [(1, 4, 2048, 4), (5, 1, 256, 1), (3, 2, 768, 3), (130, 3, 3072, 2), (4, 4, 8192, 8), (2, 4, 2304, 9)])
def test_rows_held_in_registers_are_mixed_and_normed_in_one_launch(rows, streams, width, groups):
    """Up to four streams and groups of whole 256 features: mix and norm in one launch against the mix by itself (bit for bit) and
    the norm in 64 bits; rows of fewer pieces than a block has threads, and of more."""
    from llm_rs_amd import kernels
    k, g = kernels(), torch.Generator(device="cuda").manual_seed(rows + width)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    x, y, mix, w_in, w_out, weight = rnd(streams, rows, width), rnd(rows, width), rnd(streams, streams), rnd(streams), rnd(streams), rnd(width)
    mixed = x.clone()
    k.streams_mix(mixed, mix, w_out, y)
    u = (mixed.double() * w_in.double()[:, None, None]).sum(0)
    want = plain_group_rmsnorm(u, weight.double(), 1e-5, groups)
    size = u.abs().amax(-1, keepdim=True) / want.abs().amax(-1, keepdim=True)          # what a rounding of u is in the result
    for dtype in (torch.float32, torch.bfloat16):
        streams_now, room = x.clone(), y.clone()
        out, combined = torch.empty((rows, width), dtype=dtype, device="cuda"), torch.empty((rows, width), device="cuda")
        k.group_rmsnorm(out, streams_now, weight, 1e-5, groups, w_in=w_in, zero=room, combined=combined, mix=(mix, w_out, room))
        assert torch.equal(streams_now, mixed) and not room.any()
        # (a sum of S products in 32 bits: S roundings of its largest term; the norm's own few more)
        assert ((combined.double() - u).abs() <= 2 ** -23 * (streams + 1) * (mixed.abs().double() * w_in.abs().double()[:, None, None]).sum(0)).all()
        assert ((out.double() - want).abs() <= want.abs() * (2 ** -8 if dtype == torch.bfloat16 else 2 ** -20) + 2 ** -20 * u.abs().amax() / size).all()
        last = torch.tensor([rows - 1], dtype=torch.int32, device="cuda")
        one = torch.empty((1, width), dtype=dtype, device="cuda")
        k.group_rmsnorm(one, mixed, weight, 1e-5, groups, last, w_in=w_in)
        assert torch.equal(one[0], out[-1])


@pytest.mark.parametrize("rows,streams,width,groups", [(1, 4, 2048, 4), (5, 1, 256, 1), (3, 2, 768, 3), (130, 3, 3072, 2), (4, 4, 8192, 8), (3, 4, 8192, 32),
                                                       (2, 4, 2304, 9), (2, 2, 2304, 1), (7, 4, 2048, 1), (3, 3, 4096, 2)])
def test_rows_held_in_registers_get_the_bits_of_the_general_norm(rows, streams, width, groups):
    """A group's squares are added in one order whether or not a block holds its row in registers (a weight whose rows do not begin
    on 16 bytes is the general kernel's), with and without a mix: groups shorter and longer than a block, whole and cut."""
    from llm_rs_amd import kernels
    k, g = kernels(), torch.Generator(device="cuda").manual_seed(rows + width)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    x, y, mix, w_in, w_out = rnd(streams, rows, width), rnd(rows, width), rnd(streams, streams), rnd(streams), rnd(streams)
    room = rnd(width + 1)
    weights = room[1:], room[1:].clone()
    assert weights[0].data_ptr() % 16 and weights[1].data_ptr() % 16 == 0
    for dtype in (torch.float32, torch.bfloat16):
        for with_mix in (False, True):
            got = []
            for weight in weights:
                streams_now, out = x.clone(), torch.empty((rows, width), dtype=dtype, device="cuda")
                k.group_rmsnorm(out, streams_now, weight, 1e-5, groups, w_in=w_in, mix=(mix, w_out, y) if with_mix else None)
                got.append((out, streams_now))
            assert all(torch.equal(a, b) for a, b in zip(*got)), (dtype, with_mix)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("entries,channels,states", [(1, 64, 16), (4, 4096, 16), (3, 70, 5), (2, 100, 1), (5, 130, 9)])
def test_single_tokens_through_the_scan_equal_the_walk(entries, channels, states, dtype):
    """Where the caller says that every entry brings one token the scan and the convolution run in kernels of their own: the
    same bits as the walk, the states too."""
    from llm_rs_amd import kernels
    k, g = kernels(), torch.Generator(device="cuda").manual_seed(channels)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    x, bc, dt, gate = rnd(entries, channels).to(dtype), rnd(entries, 2 * states + 3).to(dtype), rnd(entries, channels), rnd(entries, channels)
    A, D, bias, taps = -torch.exp(rnd(states, channels)), rnd(channels), rnd(channels), rnd(channels, 4)
    slots = torch.randperm(entries + 2, generator=torch.Generator().manual_seed(1))[:entries].int().cuda()
    starts, entry = torch.arange(entries + 1, dtype=torch.int32, device="cuda"), torch.arange(entries, dtype=torch.int32, device="cuda")
    before = rnd(entries + 2, channels * (states + 3))
    got = []
    for longest in (0, 1):
        state, out, conv = before.clone(), torch.zeros((entries, channels), dtype=dtype, device="cuda"), torch.zeros((entries, channels), dtype=dtype, device="cuda")
        k.causal_conv(gate, taps, bias, state[:, channels * states:], starts, slots, entry, channels, conv, silu=True, longest=longest)
        k.selective_scan(x, bc, 3, 3 + states, dt, bias, A, D, gate, state, starts, slots, out, longest=longest)
        got.append((state, out, conv))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and not torch.equal(got[0][0], before)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("streams,tokens,width", [(1, 3, 8), (4, 1, 2048), (3, 17, 97), (16, 5, 1000)])
def test_embeddings_into_every_stream(streams, tokens, width, dtype):
    """The rows times the scale in 32-bit, the same bits in every stream."""
    from llm_rs_amd.kernels import kernels
    g = torch.Generator().manual_seed(width)
    table, ids = torch.randn(50, width, generator=g).to(dtype), torch.randint(0, 50, (tokens,), generator=g).int()
    out = torch.full((streams, tokens, width), float("nan"), device="cuda")
    kernels().embed_streams(out, table.cuda(), ids.cuda(), 3.5)
    assert torch.equal(out.cpu(), (table[ids.long()].float() * 3.5).expand(streams, tokens, width))


@pytest.mark.parametrize("entries", [1, 4, 8, 9, 16])
@pytest.mark.parametrize("channels,hidden,rank", [(16, 8, 8), (48, 72, 24), (512, 2048, 40), (4096, 2048, 128), (2576, 1032, 16), (4112, 2048, 16), (8208, 64, 72), (16384, 72, 16)])
def test_products_that_step_their_mixers_equal_the_kernels_behind_plain_ones(channels, hidden, rank, entries):
    """One token a request: the products with the convolution, minGRU's state and the scan's against the product and the mixer's own
    kernel.  Both read the same bfloat16 numbers; the products' 32-bit sums may be added in another order (K 2^-24 of the terms' sizes,
    under 1e-4 of states near 1), and outputs round once more (2^-8 of them)."""
    from llm_rs_amd.kernels import EPI_STORE_F32, kernels
    k, g = kernels(), torch.Generator(device="cuda").manual_seed(channels + entries)
    rnd = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    b16 = lambda *shape: rnd(*shape).bfloat16()
    C, slots = channels, torch.randperm(entries + 2, generator=torch.Generator().manual_seed(entries))[:entries].int().cuda()
    starts, entry = torch.arange(entries + 1, dtype=torch.int32, device="cuda"), torch.arange(entries, dtype=torch.int32, device="cuda")
    before = rnd(entries + 2, C * 19 + 4)

    def compare(named, got, want):
        for name, a, b in zip(named, got, want):
            tol = dict(rtol=2.0 ** -7, atol=2e-3) if a.dtype == torch.bfloat16 else dict(rtol=1e-4, atol=1e-4)
            torch.testing.assert_close(a, b, msg=lambda m: f"{name}: {m}", **tol)

    x, w, taps, bias = b16(entries, hidden), (rnd(2 * C + 4, hidden) / hidden ** 0.5).bfloat16(), rnd(C, 4), rnd(C)
    plain, fused = torch.empty(entries, 2 * C + 4, device="cuda"), torch.empty(entries, 2 * C + 4, device="cuda")
    states, outs = [before.clone(), before.clone()], [torch.empty(entries, C, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    k.gemm(x, w, plain, EPI_STORE_F32)
    k.causal_conv(plain, taps, bias, states[0][:, 16 * C:], starts, slots, entry, C, outs[0], silu=True, longest=1)
    k.conv_product_step(x, w, fused, taps, bias, states[1][:, 16 * C:], slots, C, outs[1])
    compare(("convolved", "its state", "the gate's sums"), (outs[1], states[1], fused[:, C:]), (outs[0], states[0], plain[:, C:]))

    x, w, bz, bc = b16(entries, hidden), (rnd(3 * C, hidden) / hidden ** 0.5).bfloat16(), rnd(C), rnd(C)
    sums = torch.empty(entries, 3 * C, device="cuda")
    states, outs = [before.clone(), before.clone()], [torch.empty(entries, C, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    k.gemm(x, w, sums, EPI_STORE_F32)
    k.mingru_scan(sums, bz, bc, states[0], starts, slots, C, outs[0], 1)
    k.mingru_product_step(x, w, bz, bc, states[1], slots, C, outs[1])
    compare(("minGRU", "its state"), (outs[1], states[1]), (outs[0], states[0]))

    u, dbc, w, gate = b16(entries, C), b16(entries, rank + 32), (rnd(C, rank) / rank ** 0.5).bfloat16(), rnd(entries, C)
    A, D, bias = -torch.exp(rnd(16, C)), rnd(C), rnd(C) - 2.0
    dt = torch.empty(entries, C, device="cuda")
    states, outs = [before.clone(), before.clone()], [torch.empty(entries, C, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    k.gemm(dbc[:, :rank], w, dt, EPI_STORE_F32)
    k.selective_scan(u, dbc, rank, rank + 16, dt, bias, A, D, gate, states[0], starts, slots, outs[0], longest=1)
    k.scan_product_step(dbc, rank, w, u, bias, A, D, gate, states[1], slots, outs[1])
    compare(("scan", "its state"), (outs[1], states[1]), (outs[0], states[0]))


def test_a_scan_of_many_states_is_left_to_its_own_kernel(monkeypatch):
    """Asked by the measured cases; and a step whose products convolve but leave the scan to its kernel against one whose products do both (a
    bfloat16 rounding, 2^-8, of the results of either and of what they make of the next product, in two layers)."""
    from llm_rs_amd.kernels import kernels
    k = kernels()
    assert all(k.product_steps_scan(*at) for at in ((1, 16384), (9, 12288), (14, 8192), (16, 4096)))
    assert not any(k.product_steps_scan(*at) for at in ((16, 8192), (12, 12288), (16, 16384)))
    cfg = config(64, 40, 2, 2, 2.0, [mamba1(96, 16, 4, 8), mamba1(32, 16, 4, 16)])
    typed, tensors = make_model(cfg, seed=21)
    rows = []
    for in_product in (True, False):
        asked = []
        monkeypatch.setattr(type(k), "product_steps_scan", lambda self, *at: asked.append(at) or in_product)
        eng = engine_for(typed, tensors, "bfloat16", 16, 256)
        slots = [eng.open_request() for _ in range(3)]
        eng.step([StepEntry(s, 0, random_tokens(40, 5 + s, s), []) for s in slots])
        rows.append([eng.step([StepEntry(s, 5 + s + j, [7 * j + s], [0]) for s in slots]).clone() for j in range(4)])
        assert (3, 96) in asked and (3, 32) in asked
    for one, other in zip(*rows):
        torch.testing.assert_close(one, other, rtol=2.0 ** -6, atol=2.0 ** -6 * float(other.abs().max()))


@pytest.mark.parametrize("dtype", DTYPES)
def test_a_step_of_more_than_a_thousand_tokens(dtype):
    """Steps this long take the convolution several tokens a block: a long portion beside a short one, both continued
    in the next step, over narrow and wide channels and several tap counts."""
    cfg = config(32, 40, 2, 2, 2.0, [mamba1(72, 5, 4, 3), mamba1(320, 4, 3, 2), mingru(40), mamba1(24, 20, 2, 2, ff=48)])
    typed, tensors = make_model(cfg, seed=12)
    requests = {"a": random_tokens(40, 1100, 1), "b": random_tokens(40, 40, 2)}
    exact = reference(cfg, tensors, requests)
    allowed = allowed_error(dtype, cfg, tensors, requests, exact)
    cuts = {"a": 1031, "b": 5}
    steps = [{"step": 0, "entries": [{"id": r, "tokens": t[:cuts[r]], "want": list(range(cuts[r]))} for r, t in requests.items()], "end": []},
             {"step": 1, "entries": [{"id": r, "tokens": t[cuts[r]:], "want": list(range(len(t) - cuts[r]))} for r, t in requests.items()], "end": list(requests)}]
    eng = engine_for(typed, tensors, dtype, 16, 1280)
    check_rows(replay(eng, steps), exact, requests, allowed, "two steps")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("which", ["even", "odd"])
def test_sizes_that_are_no_multiples_of_four(which, dtype):
    """No vector load fits these rows: every kernel's narrow path, also in steps long enough for chunks and fused norms."""
    cfg = {"even": config(46, 51, 3, 2, 1.0, [mingru(30), mamba1(26, 3, 3, 3, ff=22), attention(3, 1, 10, 6, 0.3, 9, ff=14)]),
           "odd": config(45, 37, 2, 3, 2.5, [attention(2, 2, 7, 5, 0.4, 6), mingru(17, ff=9), mamba1(15, 5, 2, 1)])}[which]
    typed, tensors = make_model(cfg, seed=13)
    requests = {"a": random_tokens(cfg["vocab"], 140, 1), "b": random_tokens(cfg["vocab"], 21, 2), "c": random_tokens(cfg["vocab"], 2, 3)}
    run_regimes(cfg, typed, tensors, dtype, 16, requests,
                {"whole": whole(requests), "decoded": tail_decoded(requests, tail=20), "portions": portions(requests, (3, 131, 2)),
                 "mixed": mixed(requests, live=3)})


# ---- configurations drawn at random -----------------------------------------------------------------------------------

def random_configuration(seed):
    import random
    r = random.Random(seed)
    width = r.choice([24, 40, 64, 96, 136])
    groups = r.choice([g for g in (1, 2, 3, 4, 8) if width % g == 0])
    layers = []
    for _ in range(r.randint(2, 5)):
        ff = r.choice([None, None, 8 * r.randint(2, 12)])
        kind = r.choice(["mingru", "mamba1", "attention"])
        if kind == "mingru":
            layers.append(mingru(4 * r.randint(3, 30), ff=ff))
        elif kind == "mamba1":
            layers.append(mamba1(4 * r.randint(3, 30), r.choice([1, 4, 16, 24, 33, 70]), r.randint(1, 5), r.randint(1, 9), ff=ff))
        else:
            kv = r.choice([1, 2, 3])
            dim = r.choice([8, 20, 32, 64, 128])
            vdim = r.choice([dim, dim, 4 * r.randint(1, 10)])
            layers.append(attention(kv * r.choice([1, 2, 4]), kv, dim, vdim, r.uniform(0.05, 0.5), r.choice([1, 5, 16, 17, 31, 32, 48, 100, 500]), ff=ff))
    return config(width, r.randint(30, 200), r.randint(1, 6), groups, r.uniform(0.5, 10.0), layers, eps=r.choice([1e-5, 1e-6, 1e-3]))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("seed", range(8))
def test_configurations_drawn_at_random(seed, dtype):
    cfg = random_configuration(seed)
    typed, tensors = make_model(cfg, seed=seed)
    requests = {f"r{i}": random_tokens(cfg["vocab"], n, 70 + i) for i, n in enumerate([150, 3, 66, 1, 35])}
    run_regimes(cfg, typed, tensors, dtype, 16, requests,
                {"whole": whole(requests), "decoded": tail_decoded(requests, tail=36), "portions": portions(requests, (2, 70, 3, 33)),
                 "mixed": mixed(requests, live=3)})


# ---- generation through the scheduler --------------------------------------------------------------------------------

def plain_greedy(cfg, tensors, prompt, n):
    toks, margins = list(prompt), []
    for _ in range(n):
        row = plain_tuvodra_logits(cfg, tensors, toks)[-1]
        top = torch.topk(row, 2).values
        margins.append(float(top[0] - top[1]) / float(row.abs().max()))
        toks.append(int(torch.argmax(row)))
    return toks[len(prompt):], margins


@pytest.mark.parametrize("which", ["odd", "plain"])
def test_greedy_generation_through_the_scheduler(which):
    cfg = CONFIGS[which]
    typed, tensors = make_model(cfg, seed=8)
    prompts = [random_tokens(cfg["vocab"], n, 20 + n) for n in (1, 5, 19, 40, 3, 27)]
    eng = Engine(typed, tensors, dtype="float32", page_size=PAGE_SIZE[which], num_pages=64, max_requests=3, max_batch_tokens=24)
    outs = eng.generate(prompts, max_new_tokens=12)
    for prompt, out in zip(prompts, outs):
        want, margins = plain_greedy(cfg, tensors, prompt, 12)
        out = list(out.tokens if hasattr(out, "tokens") else out)
        for i, (a, b) in enumerate(zip(out, want)):
            if a != b:
                assert margins[i] < 1e-4, (prompt, i, out, want)       # a tie within rounding may fall either way
                break


# ---- the programs, on a model folder ----------------------------------------------------------------------------------

def test_the_programs_on_a_model_folder(tmp_path):
    """A folder with config.json and model.safetensors through `bin/trace_run` (a mixed trace under a small pool, both
    dtypes) and through `bin/llm-rs complete` (greedy): the architecture is chosen by the file."""
    import json
    import os
    import subprocess
    import sys

    import numpy as np
    from tuvodra_cases import make_folder
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    cfg = CONFIGS["plain"]
    folder = make_folder(tmp_path, cfg, seed=11)
    typed, tensors = make_model(cfg, seed=11)
    requests = {f"r{i}": random_tokens(cfg["vocab"], n, 50 + i) for i, n in enumerate([33, 2, 90, 47, 18])}
    exact = reference(cfg, tensors, requests)
    steps = mixed(requests, live=3)
    text = "".join(json.dumps(s) + "\n" for s in steps)
    for dtype in DTYPES:
        out = tmp_path / f"out_{dtype}"
        p = subprocess.run([sys.executable, os.path.join(root, "bin", "trace_run"), "--model", folder, "--dtype", dtype, "--out", str(out),
                            "--max-tokens", str(live_token_need(steps, 64))], input=text, capture_output=True, text=True, timeout=600)
        assert p.returncode == 0, p.stderr[-2000:]
        assert [l for l in p.stdout.split("\n") if l.startswith("done")] == [f"done {s['step']}" for s in steps]
        outputs = []
        for s in steps:
            n = sum(len(e["want"]) for e in s["entries"])
            outputs.append(torch.from_numpy(np.fromfile(out / f"{s['step']}.f32", dtype="<f4").reshape(n, cfg["vocab"]).copy()) if n else None)
        check_rows(collect(steps, outputs), exact, requests, allowed_error(dtype, cfg, tensors, requests, exact), f"trace_run {dtype}")
    prompt = requests["r3"]
    p = subprocess.run([sys.executable, os.path.join(root, "bin", "llm-rs"), "-m", folder, "--dtype", "float32", "--num-pages", "64", "complete",
                        "--prompt-ids", " ".join(map(str, prompt)), "-n", "10", "--temperature", "0"], capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stderr[-2000:]
    got = [int(t) for t in p.stdout.split()]
    want, margins = plain_greedy(cfg, tensors, prompt, 10)
    for i, (a, b) in enumerate(zip(got, want)):
        if a != b:
            assert margins[i] < 1e-4, (i, got, want)
            break
    assert len(got) == 10
