"""Views of the workspace that the step function keeps from step to step: whoever holds a step's result, and whatever mode a step ran in, the next one
gets its room as it was asked for."""
import pytest
import torch

from emulated_kernels import EmulatedKernels
from llm_rs_amd import Engine, LlamaConfig, StepEntry, random_model_tensors, use_kernels
from tiny_configs import TINY_A


@pytest.fixture
def engine():
    cfg = LlamaConfig.from_dict(TINY_A)
    with use_kernels(EmulatedKernels()):
        yield Engine(cfg, random_model_tensors(cfg, 3), dtype="float32", device="cpu", page_size=4, num_pages=64, max_requests=4)


def test_steps_inside_and_outside_of_inference_mode(engine):
    """A step's room made inside is written by torch's own operations outside, and the other way round."""
    slot = engine.open_request()
    entries = lambda at: [StepEntry(slot, at, [3, 4], [0, 1])]
    want = engine.step([StepEntry(slot, 0, [5, 6, 7], [2])]).clone()
    with torch.inference_mode():
        inside = engine.step(entries(3)).clone()
    logits = engine.step(entries(3))
    assert torch.equal(logits, inside)
    logits.add_(1.0)
    with torch.inference_mode():
        room = engine.runner.workspace("new", (3, 2), torch.float32)
        room.zero_()
    engine.runner.workspace("new", (3, 2), torch.float32).add_(1.0)
    engine.runner.workspace("new", (2, 2), torch.float32).add_(1.0)
    assert torch.equal(engine.step([StepEntry(slot, 0, [5, 6, 7], [2])]), want)


@pytest.mark.parametrize("planned", [False, True])
def test_a_callers_logits_may_be_reshaped_in_place(engine, planned):
    core, runner = engine.cache.core, engine.runner
    slot = core.add_request([5, 6, 7], 8)
    assert slot >= 0
    for step in range(3):
        if planned:
            logits, n, plan = runner.run_planned()
            assert n == 1 and len(plan) == 1
        else:
            logits = engine.step([StepEntry(slot, 0, [5, 6, 7], [0, 1])])
        assert tuple(logits.shape) == (1 if planned else 2, runner.model.spec.vocab_size)
        if planned:
            core.commit([int(logits[0].argmax())])
        logits.t_()
