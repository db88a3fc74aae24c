"""A sandwich block whose norms are of another kind, or have another eps, than those of the block before it: the norm left pending
is formed on its own."""

from types import SimpleNamespace

import pytest
import torch

from atom_amd.parts.base import NORMS, Norm, PartChoice, PendingPost
from atom_amd.parts.block import SandwichBlock
from atom_amd.parts.norm import LayerNorm
from plain_kernels import PlainKernels

WIDTH = 16


class Scaled(Norm):
    """Nothing but a weight: no eps, no bias, no ``forward_post``."""

    accepts_deferred = False

    def __init__(self, size, prefix=""):
        super().__init__(prefix)
        self.size = size

    def forward(self, ctx, x, out_dtype=None):
        return (x * self.params["weight"]).to(out_dtype or ctx.dtype)

    def forward_residual(self, ctx, x, residual):
        residual += x
        return self.forward(ctx, residual), residual


class Half:
    accepts_deferred = True

    def forward(self, ctx, x, cache=None):
        return 0.5 * x


def block(kind, monkeypatch, **kw):
    monkeypatch.setitem(NORMS._items, "scaled", Scaled)
    b = SandwichBlock.__new__(SandwichBlock)
    g = torch.Generator().manual_seed(7)
    for name in ("mixer_pre", "mixer_post", "ffn_pre", "ffn_post"):
        norm = PartChoice(kind, dict(size=WIDTH, **kw)).build(NORMS, prefix=name)
        norm.params["weight"] = 1 + 0.1 * torch.randn(WIDTH, generator=g)
        if kind == "layernorm":
            norm.params["bias"] = 0.1 * torch.randn(WIDTH, generator=g)
        setattr(b, name, norm)
    b._mixer, b.ffn = Half(), Half()
    return b


@pytest.mark.parametrize("kind,kw", [("scaled", {}), ("layernorm", {"eps": 0.5}), ("layernorm", {"eps": 1e-5})])
def test_what_follows_a_layer_norms_block(kind, kw, monkeypatch):
    ctx = SimpleNamespace(ops=PlainKernels(), dtype=torch.float32)
    first, second = block("layernorm", monkeypatch, eps=1e-5), block(kind, monkeypatch, **kw)
    x = torch.randn(3, WIDTH, generator=torch.Generator().manual_seed(1))

    hidden, stream = first.forward(ctx, x, None, None)
    assert isinstance(hidden, PendingPost) and isinstance(first.ffn_post, LayerNorm)
    copy = stream.clone()
    apart, want_stream = second.forward(ctx, hidden.resolve(ctx), copy, None)
    got, got_stream = second.forward(ctx, hidden, stream, None)
    if isinstance(got, PendingPost):
        got, apart = got.resolve(ctx), apart.resolve(ctx)
    assert torch.allclose(got_stream, want_stream, atol=1e-6) and torch.allclose(got, apart, atol=1e-6)
