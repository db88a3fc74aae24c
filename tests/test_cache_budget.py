"""What the cache's budget leaves free: memory a step takes in its parts beside the activations."""

import ctypes
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


def _f32_mlp(hidden, inter, dtype=torch.float32):
    part = GatedMLP(hidden, inter)
    part.params = {name: torch.empty(spec.shape, dtype=dtype, device="meta") for name, spec in part.param_specs().items()}
    return part


def test_float32_products_are_left_their_scratch_memory(monkeypatch):
    ops = _ops()
    ops.F32_SPLIT_ROWS = HipKernels.F32_SPLIT_ROWS
    ops.product_scratch = lambda *a: HipKernels.product_scratch(ops, *a)
    monkeypatch.setattr("test_cache_budget._ops", lambda: ops)
    plain = _budget([_f32_mlp(1024, 4096, torch.bfloat16)], 4096, monkeypatch)
    assert _budget([_f32_mlp(512, 1024), _f32_mlp(1024, 4096)], 4096, monkeypatch) == plain - 6 * 2048 * 4096
    assert _budget([_f32_mlp(1024, 4096)], 300, monkeypatch) == plain - 6 * 300 * 4096
    assert _budget([_f32_mlp(1024, 4096)], 64, monkeypatch) == _budget([_f32_mlp(1000, 4100)], 4096, monkeypatch) == plain
    rule = GatedDeltaRule(512, 8, 4, 128, 128, 4, 1e-6)
    rule.params = {"o.weight": torch.empty(512, 65536, device="meta")}
    assert _budget([rule], 256, monkeypatch) == plain - 6 * 256 * 65536


def test_decode_graphs_are_left_the_scratch_memory_of_their_products():
    ops = SimpleNamespace(product_scratch=lambda rows, k: 6 * rows * k)
    config = SimpleNamespace(cudagraph_capture_sizes=[1, 128], max_num_seqs=128, cudagraph_prefill_sizes=[], cudagraph_prefill_slots=2,
                             max_num_batched_tokens=4096, max_model_len=4096)

    def estimate(dtype):
        engine = LLMEngine.__new__(LLMEngine)
        engine.config, engine.ops = config, ops
        block = SimpleNamespace(walk=lambda: [_f32_mlp(1024, 4096, dtype)])
        engine.model = SimpleNamespace(blocks=[block], spec=SimpleNamespace(hidden_size=1024, vocab_size=100))
        return engine._graph_estimate()

    assert estimate(torch.float32) == estimate(torch.bfloat16) + 6 * 128 * 4096


def test_bfloat16_products_of_many_rows_are_left_what_their_plans_take(monkeypatch):
    from atom_amd.kernels.build import build

    ops = _ops()
    ops.lib = ctypes.CDLL(build())
    ops.lib.atom_gemm_many_scratch.restype = ops.lib.atom_gemm_many_scratch_most.restype = ctypes.c_long
    ops.use_many_gemm, ops.many_rows, ops.num_cus, ops._many_most = True, 257, 256, {}
    ops.product_scratch = lambda rows, k: 0
    ops.many_scratch = lambda *a: HipKernels.many_scratch(ops, *a)
    monkeypatch.setattr("test_cache_budget._ops", lambda: ops)

    def taken(rows, n, k, gate, apart):
        plan = (ctypes.c_int * 4)()
        if ops.lib.atom_gemm_many_plan(rows, n, k, gate, apart, 256, plan) != 0:
            return 0
        tile, whole, slices, as_slices = plan
        return 4 * slices * rows * n if as_slices else ops.lib.atom_gemm_many_scratch(rows, n, gate, tile, whole, slices)

    def most(part, tokens):
        return max(taken(m, n // 2 if gate else n, k, gate, apart) for n, k in (tuple(p.shape) for p in part.params.values() if p.dim() == 2)
                   for m in range(257, tokens + 1) for gate, apart in ((0, 0), (0, 1), (1, 0)))

    plain = _budget([GatedMLP(512, 1024)], 4096, monkeypatch)
    for hidden, inter, tokens in ((512, 1024, 4096), (1024, 2048, 700), (2560, 9728, 2000), (576, 1096, 300)):
        part = _f32_mlp(hidden, inter, torch.bfloat16)
        assert _budget([part], tokens, monkeypatch) == plain - most(part, tokens)
        assert most(part, tokens) <= 128 << 20 and (most(part, tokens) > 0 or tokens == 300)
    assert _budget([_f32_mlp(1024, 4096, torch.bfloat16)], 256, monkeypatch) == plain
    assert _budget([_f32_mlp(100, 300, torch.bfloat16)], 4096, monkeypatch) == plain     # no size the kernel takes
    small = _f32_mlp(1024, 2816, torch.bfloat16)
    assert most(small, 2048) < 100 << 20                                                 # not the bound of all plans
