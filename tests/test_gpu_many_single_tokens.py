"""The single-token kernels of a decode step with many requests: every request's result has the bits that it has alone (which
``test_gpu_single_token_steps.py`` compares with float64), requests that are padding write zeros, other slots stay as they are."""

import pytest
import torch

from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
COUNTS = [33, 64]


def rnd(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(DEV)


def i32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def alone_and_together(launch, rows, state, width, dtype, count):
    """``launch(rows, state, cu, slots, out)`` for all requests (each a row of every tensor of ``rows``), and for some of them."""
    slots = torch.randperm(count + 3, generator=torch.Generator().manual_seed(5))[:count].tolist()
    slots[7] = -1
    together, out = state.clone(), torch.full((count, width), 7.0, dtype=dtype, device=DEV)
    assert launch(rows, together, i32(range(count + 1)), i32(slots), out) is out
    assert float(out[7].abs().max()) == 0 and bool(out.isfinite().all())
    unused = sorted(set(range(count + 3)) - set(slots))
    assert torch.equal(together[unused], state[unused])
    for r in (0, 8, count // 2, count - 1):
        single, row = state.clone(), torch.empty((1, width), dtype=dtype, device=DEV)
        assert launch([t[r:r + 1].contiguous() for t in rows], single, i32([0, 1]), i32([slots[r]]), row) is row
        assert torch.equal(row[0], out[r]) and torch.equal(single[slots[r]], together[slots[r]])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("heads,kv_heads,dim,per_channel,rank", [(16, 8, 128, True, 64), (4, 4, 64, False, 0)])
def test_delta_step(heads, kv_heads, dim, per_channel, rank, count, dtype):
    ops = gpu_ops()
    C, decays, v = (2 * kv_heads + heads) * dim, heads * (dim if per_channel else 1), heads * dim
    a_off, g_off = C + heads, C + heads + (rank or decays)
    decay2, gate2 = (rnd((n, rank), s, 0.2).to(dtype) if rank else None for n, s in ((decays, 3), (v, 4)))
    rows, state = [rnd((count, g_off + (rank or v)), 1)], rnd((count + 3, 3 * C + v * dim), 8, 0.3)
    taps, rest = rnd((C, 4), 2, 0.5).to(dtype), (rnd((heads,), 5, 0.5), rnd((decays,), 6) - 1, 1 + rnd((dim,), 7, 0.2))

    def launch(rows, state, cu, slots, out):
        return ops.delta_step(rows[0], taps, state, 3 * C, cu, slots, C, a_off, decay2, g_off, gate2, *rest, 1e-5, out, heads,
                              kv_heads, dim, dim, per_channel, "silu")

    alone_and_together(launch, rows, state, v, dtype, count)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("count", COUNTS)
@pytest.mark.parametrize("heads,groups,dim", [(64, 1, 128), (6, 2, 64)])
def test_space_step(heads, groups, dim, count, dtype):
    ops = gpu_ops()
    inner = heads * 64
    C = inner + 2 * groups * dim
    rows = [rnd((count, inner + C + (heads + 3) // 4 * 4), 1)]
    taps, bias, norm = rnd((C, 4), 2, 0.5).to(dtype), rnd((C,), 3, 0.3), 1 + rnd((inner,), 7, 0.2)
    head, state = (rnd((heads,), 4) - 1, rnd((heads,), 5, 0.5), rnd((heads,), 6)), rnd((count + 3, 3 * C + inner * dim), 8, 0.3)

    def launch(rows, state, cu, slots, out):
        return ops.space_step(rows[0], inner, taps, bias, state, 3 * C, cu, slots, *head, norm, 1e-5, out, heads, groups, dim, 64, 1)

    alone_and_together(launch, rows, state, inner, dtype, count)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("count", COUNTS)
def test_mix_step(count, dtype, heads=32, rank=64):
    ops = gpu_ops()
    c = heads * 64
    rows = [rnd((count, c), s) for s in (1, 2, 3, 4)] + [torch.tanh(rnd((count, rank), 5))]
    decay2, state = rnd((c, rank), 6, 0.2).to(dtype), rnd((count + 3, 8 + c * 64), 10, 0.3)
    rest = rnd((c,), 7) - 2, rnd((heads, 64), 8, 0.3), 1 + rnd((c,), 9, 0.2)

    def launch(rows, state, cu, slots, out):
        return ops.mix_step(*rows, decay2, *rest, state, 8, cu, slots, out, heads, 64, 1e-5)

    alone_and_together(launch, rows, state, c, dtype, count)
