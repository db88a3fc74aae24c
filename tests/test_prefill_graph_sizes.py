"""Which sizes of prompt portions graphs are captured for: what the caller says, an empty list too; the engine's choice otherwise."""

from types import SimpleNamespace

import torch

from atom_amd.config.engine_config import Config
from atom_amd.engine.arg_utils import EngineArgs, FlexibleArgumentParser
from atom_amd.engine.llm_engine import LLMEngine


def sizes(configured, batched=64, max_len=4096, layer_bytes=1 << 20, dtype=torch.bfloat16):
    engine = LLMEngine.__new__(LLMEngine)
    engine.dtype = dtype
    part = SimpleNamespace(params={"weight": torch.empty(layer_bytes // dtype.itemsize, dtype=dtype, device="meta")})
    engine.config = SimpleNamespace(cudagraph_prefill_sizes=configured, max_num_batched_tokens=batched, max_model_len=max_len)
    engine.model = SimpleNamespace(blocks=[SimpleNamespace(walk=lambda: [part])])
    return engine._prefill_graph_sizes()


def test_what_the_caller_says_holds():
    assert sizes([]) == [] and sizes([24]) == [24] and sizes([256, 512], batched=16384) == [256, 512]


def test_the_engine_chooses_where_nothing_is_said():
    assert Config.__dataclass_fields__["cudagraph_prefill_sizes"].default is None
    assert sizes(None) == [16, 64] and sizes(None, batched=16384) == [] and sizes(None, layer_bytes=1 << 30) == []


def test_float32_layers_are_padded_dearly():
    for layer, half, single in ((1 << 20, [16, 64], [16, 64]), (100 << 20, [16, 64], []), (250 << 20, [], [])):
        assert sizes(None, layer_bytes=layer) == half and sizes(None, layer_bytes=layer, dtype=torch.float32) == single


def test_the_command_line_says_none_some_or_leaves_it_to_the_engine():
    parser = FlexibleArgumentParser()
    EngineArgs.add_cli_args(parser)

    def said(*args):
        return EngineArgs.from_cli_args(parser.parse_args(["--model", "m", *args]))._get_engine_kwargs()["cudagraph_prefill_sizes"]

    assert said() == said("--cudagraph-prefill-sizes", "[]") == [] and said("--cudagraph-prefill-sizes", "[32]") == [32]
    assert said("--cudagraph-prefill-sizes", "auto") is None
