"""The arrays that a step's context hands out: views of the step's words, made when they are asked for."""
import types

import pytest
import torch

from llm_rs_amd.engine.step import StepContext


class Runner:
    device = torch.device("cpu")


def test_arrays_are_those_of_the_step_that_is_bound():
    runner = Runner()
    ctx = StepContext(runner)
    assert ctx.tokens is None and ctx.slot_maps == [] and ctx.block_tables == []
    for T, R, n, widths in ((5, 2, 1, [3]), (1, 1, 1, [64, 2]), (7, 3, 0, [])):
        at, where = 4, {}
        for name, size in (("tokens", T), ("positions", T), ("token_entry", T), ("q_starts", R + 1), ("seq_lens", R), ("slots", R), ("want_rows", n), ("sampling", 4 * n)):
            where[name], at = (at, size), at + size
        slot_maps = [at + i * T for i in range(len(widths))]
        at += len(widths) * T
        tables = []
        for w in widths:
            tables.append(at)
            at += R * w
        dev = torch.arange(at, dtype=torch.int32)
        ctx.n_tokens, ctx.n_entries, ctx.n_want = T, R, n
        ctx.lay_out(dev, types.SimpleNamespace(slot_maps=slot_maps, tables=tables, widths=widths, **{k: v[0] for k, v in where.items()}))
        for name, (first, size) in where.items():
            got = getattr(ctx, name)
            assert got is getattr(ctx, name) and got.flatten().tolist() == list(range(first, first + size)), name
        assert tuple(ctx.sampling.shape) == (n, 4)
        assert [m.tolist() for m in ctx.slot_maps] == [list(range(o, o + T)) for o in slot_maps]
        assert [tuple(t.shape) for t in ctx.block_tables] == [(R, w) for w in widths] and [int(t[0, 0]) for t in ctx.block_tables] == tables
    with pytest.raises(AttributeError):
        ctx.no_such_array
