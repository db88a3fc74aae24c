"""Engines whose token budget is small replay graphs for steps with prompt portions too: the logits are those of launched
steps, whichever entries want some, and stay as they are when later steps run."""

import pytest
import torch

from atom_amd import LLMEngine
from atom_amd.engine.core import StepEntry
from helpers import gpu_ops, random_ids, tiny_folder
from tiny import PAGE

pytestmark = pytest.mark.gpu


def engine(which, **kw):
    return LLMEngine(tiny_folder(which), dtype="fp32", ops=gpu_ops(), kv_cache_block_size=PAGE[which], num_kvcache_blocks=64,
                     max_num_seqs=4, cudagraph_capture_sizes=[1, 2, 4], **kw)


def test_portions_of_a_small_budget_are_replayed():
    ids = [random_ids("B", n, 7 + n) for n in (40, 21, 60)]
    steps = [[StepEntry(0, ids[0][:16])], [StepEntry(0, ids[0][16:32]), StepEntry(1, ids[1][:5], [4])],
             [StepEntry(0, ids[0][32:39], [6]), StepEntry(1, ids[1][5:20], [])],
             [StepEntry(0, ids[0][39:], [0]), StepEntry(1, ids[1][20:], []), StepEntry(2, ids[2][:33], [32])],
             [StepEntry(2, ids[2][33:], [26])]]
    outs, replays = [], []
    for kw in ({"max_num_batched_tokens": 64}, {"max_num_batched_tokens": 64, "enforce_eager": True}):
        core = engine("B", **kw).core
        outs.append([core.step(step) for step in steps])
        replays.append(core.graphs.mixed_replays if core.graphs is not None else 0)
    assert replays == [5, 0]
    for a, b in zip(*outs):
        assert (a is None) == (b is None)
        if a is not None:   # in 32 bits a row does not depend on what else is in the step, padding included
            assert a.shape == b.shape and float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


def test_large_budgets_launch_their_portions():
    core = engine("B", max_num_batched_tokens=256).core
    core.step([StepEntry(0, random_ids("B", 9, 3))])
    assert core.graphs.prefill_sizes == [] and core.graphs.mixed_replays == 0
