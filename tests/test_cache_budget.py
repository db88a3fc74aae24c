"""What the cache's budget leaves free: memory a step takes in its parts beside the activations."""

from types import SimpleNamespace

import torch

from atom_amd.engine.llm_engine import LLMEngine
from atom_amd.kernels.hip import HipKernels
from atom_amd.parts.delta import GatedDeltaRule
from atom_amd.parts.mlp import GatedMLP


def _ops():
    lib = SimpleNamespace(atom_delta_chunks_supports=lambda dim, vdim: dim in (64, 128),
                          atom_delta_chunks_floats=lambda heads, dim, vdim: heads * (64 * (3 * dim + 64 + vdim) + dim))
    ops = SimpleNamespace(lib=lib, use_delta_chunks=True, DELTA_CHUNKS_FROM=HipKernels.DELTA_CHUNKS_FROM,
                          DELTA_SCRATCH_BYTES=HipKernels.DELTA_SCRATCH_BYTES)
    ops.delta_scratch = lambda *a: HipKernels.delta_scratch(ops, *a)
    return ops


def _budget(blocks, tokens, monkeypatch):
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda dev: (250 << 30, 288 << 30))
    config = SimpleNamespace(device="cuda:0", enforce_eager=True, gpu_memory_utilization=0.99, max_num_batched_tokens=tokens,
                             max_num_seqs=8)
    return LLMEngine._cache_budget(SimpleNamespace(config=config, model=SimpleNamespace(blocks=blocks), ops=_ops()))


def test_the_delta_rules_chunks_are_left_their_scratch_memory(monkeypatch):
    def rule(heads, dim, decay="head"):
        return GatedDeltaRule(512, heads, heads // 2, dim, dim, 4, 1e-6, decay=decay)

    plain = _budget([GatedMLP(512, 1024)], 4096, monkeypatch)
    place = 4 * 32 * (64 * (3 * 128 + 64 + 128) + 128)
    assert _budget([rule(32, 128), rule(8, 128)], 4096, monkeypatch) == plain - (64 + 8) * place
    assert _budget([rule(32, 128)], 16384, monkeypatch) == plain - (1 << 30) // place * place     # 264 places are beyond the bound
    assert _budget([rule(32, 32)], 16384, monkeypatch) == plain                                   # walked whatever their length
    assert _budget([rule(32, 128)], 127, monkeypatch) == _budget([rule(32, 128, "channel")], 255, monkeypatch) == plain
