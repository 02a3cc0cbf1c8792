"""The rules by which single tokens of a mixed step wait for its tiles or run beside them, and by which the tiles' keys are shared out, asked of the
kernel library as its launcher asks them."""
import ctypes

import pytest

from llm_rs_amd.csrc import build as native
from llm_rs_amd.engine.step import StepContext

# (heads, kv heads, width, portions as (start, tokens), single tokens, their keys together, in turn): the time in turn is 0.87, 0.93, 0.89
# and 0.84 of the time side by side, and then 1.12, 1.03, 1.12, 1.09, 1.04, 1.14, 1.42 and 1.33 of it
MEASURED = [(64, 8, 128, [(2048, 2048)], 16, 65536, True), (64, 8, 128, [(1000, 2940)], 14, 18283, True), (32, 8, 128, [(2048, 4096)], 37, 56901, True),
            (32, 4, 128, [(2048, 2048)] * 2, 9, 40709, True),
            (64, 8, 128, [(0, 1800)], 16, 32000, False), (64, 8, 128, [(0, 1800)], 16, 4800, False),
            (64, 8, 128, [(0, 1800)], 8, 32000, False), (64, 8, 128, [(0, 1800)], 100, 30000, False),
            (64, 8, 128, [(2048, 1600)], 250, 500000, False), (32, 8, 128, [(0, 1365)] * 3, 100, 220327, False),
            (32, 8, 64, [(500, 4096)], 231, 369050, False), (16, 16, 64, [(0, 1365)] * 3, 236, 60193, False)]


@pytest.mark.parametrize("heads,kv,width,portions,singles,keys,in_turn", MEASURED)
def test_single_tokens_wait_where_that_is_faster(heads, kv, width, portions, singles, keys, in_turn):
    seen = sum(count * start + count * (count + 1) // 2 for start, count in portions)
    ask = native.load_hip().llmrs_attention_in_turn
    ask.argtypes, ask.restype = [ctypes.c_int] * 3 + [ctypes.c_long] * 2 + [ctypes.c_int] * 5, ctypes.c_int
    tokens, entries = sum(count for _, count in portions) + singles, len(portions) + singles
    assert bool(ask(tokens, entries, singles, keys, seen, heads, kv, width, width, 1)) == in_turn
    for unknown in ((-1, keys, seen), (singles, 0, seen), (0, 0, seen)):
        assert not ask(tokens, entries, *unknown, heads, kv, width, width, 1)


# (heads, kv heads, width, entries as (start, tokens), window, in shares): the time in shares is 0.54, 0.67, 0.55, 0.72, 0.64, 0.49, 0.68 and 0.44 of the
# time without, and then, where they are not taken, 1.36, 1.05, 1.05, 1.32, 1.05, 1.06 and 1.09 of it
SHARES = [(32, 8, 128, [(8000, 512)], 0, True), (32, 8, 64, [(0, 1024)], 0, True), (32, 8, 128, [(3000, 400)], 768, True), (32, 8, 128, [(3000, 1000)], 768, True),
          (32, 8, 128, [(100, 1800)], 0, True), (64, 8, 128, [(2048, 200)] + [(299, 1)] * 4, 0, True), (64, 8, 128, [(2048, 100)] + [(3999, 1)] * 16, 0, True),
          (32, 8, 64, [(3000, 427)] + [(3500, 1)] * 11, 0, True),
          (32, 8, 128, [(0, 600)] * 12, 0, False), (64, 8, 128, [(2048, 2048)], 0, False), (32, 8, 128, [(300, 109)] * 2 + [(3220, 1)] * 10, 0, False),
          (32, 8, 128, [(0, 2048)], 300, False), (32, 8, 64, [(0, 92)] + [(2900, 1)] * 14, 0, False), (64, 8, 128, [(300, 94)] + [(2620, 1)] * 25, 0, False),
          (32, 8, 64, [(300, 506)] + [(1900, 1)] * 15, 0, False)]


@pytest.mark.parametrize("heads,kv,width,entries,window,shares", SHARES)
def test_keys_are_shared_out_where_that_is_faster(heads, kv, width, entries, window, shares):
    sees = lambda p: min(p + 1, window or p + 1)
    singles = [start + 1 for start, count in entries if count == 1]
    seen = sum(sees(start + i) for start, count in entries if count > 1 for i in range(count)) if singles else 0
    ask = native.load_hip().llmrs_attention_in_shares
    ask.argtypes, ask.restype = [ctypes.c_int] * 3 + [ctypes.c_long] * 2 + [ctypes.c_int] * 5, ctypes.c_int
    tokens, longest = sum(count for _, count in entries), max(start + count for start, count in entries)
    assert bool(ask(tokens, len(entries), len(singles), sum(singles), seen, heads, kv, width, window, longest)) == shares
    assert not ask(255, 1, 0, 0, 0, heads, kv, width, window, 255) and not ask(4, 4, 4, 4000, 0, heads, kv, width, window, 1000)


@pytest.mark.parametrize("window,chunk", [(0, 0), (1, 0), (7, 0), (40, 0), (0, 1000)])
def test_keys_that_portions_see(window, chunk):
    """Counted one token at a time."""
    class Runner:
        device = "cpu"
    ctx = StepContext(Runner())
    ctx.entries, ctx.max_seq_len = [(0, 0, 5), (1, 3, 1), (2, 6, 30), (3, 50, 2), (4, 90, 1)], 91
    reach = window or chunk or 1000
    assert ctx.portion_keys(window, chunk) == sum(min(start + i + 1, reach) for _, start, count in ctx.entries if count > 1 for i in range(count))
