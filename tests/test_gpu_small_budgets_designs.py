"""Portions under a small token budget, replayed and launched, in the other designs: convolutions, recurrences, token shifts, chunked
and latent caches all take a portion beside single tokens and padding, and the requests' memory goes on from it."""

import importlib

import pytest

from atom_amd import LLMEngine
from atom_amd.engine.core import StepEntry
from helpers import gpu_ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("number", [0, 1])
@pytest.mark.parametrize("design", ["lotorax", "ralitar", "leduvik", "savidra", "benolix", "domasun"])
def test_portions_are_replayed_as_they_are_launched(design, number):
    tiny = importlib.import_module(f"{design}_tiny")
    which = list(tiny.CONFIGS)[number]
    a, b, c = (tiny.ids(which, n, 7 + n) for n in (40, 21, 60))
    steps = [[StepEntry(0, a[:16], [])], [StepEntry(0, a[16:31], [14]), StepEntry(1, b[:5], [4])],
             [StepEntry(0, a[31:32], [0]), StepEntry(1, b[5:19], [])],
             [StepEntry(0, a[32:33], [0]), StepEntry(1, b[19:20], [0]), StepEntry(2, c[:33], [32])],
             [StepEntry(0, a[33:34], [0]), StepEntry(2, c[33:], [26])],
             [StepEntry(0, a[34:35], [0]), StepEntry(1, b[20:21], [0])]]
    outs, replays = [], []
    for sizes in (None, []):
        core = LLMEngine(tiny.folder(which), dtype="fp32", ops=gpu_ops(), kv_cache_block_size=16, num_kvcache_blocks=64, max_num_seqs=4,
                         max_num_batched_tokens=64, max_model_len=128, cudagraph_capture_sizes=[1, 2, 4],
                         cudagraph_prefill_sizes=sizes).core
        outs.append([core.step(step) for step in steps])
        replays.append((core.graphs.usable, core.graphs.mixed_replays))
    usable = replays[0][0]
    assert replays == [(usable, 5 if usable else 0), (usable, 0)]
    for got, want in zip(*outs):
        assert (got is None) == (want is None)
        if got is not None:   # in 32 bits a row does not depend on what else is in the step, padding included
            assert got.shape == want.shape and float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())
