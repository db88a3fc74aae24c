"""The delta rule in chunks of 64 tokens against float64, token by token, at the edges of chunks and tiles."""

import pytest
import torch

import plain_savidra as ps
from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


def tables(lens, slots):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu, *(torch.tensor(v, dtype=torch.int32, device=DEV) for v in (cu, slots))


def chunked(ops, monkeypatch, per_channel, H, G, D, V, lens, slots, qkv, gates, decay, a_log, dt_bias, before):
    """Outputs and state of the chunk kernels, which are made to take every request and seen to run."""
    monkeypatch.setattr(ops, "DELTA_CHUNKS_FROM", {False: 1, True: 1})
    assert ops.lib.atom_delta_chunks_supports(D, V)
    ran, kernel = [], ops.lib.atom_delta_chunks
    monkeypatch.setattr(ops.lib, "atom_delta_chunks", lambda *a: ran.append(1) or kernel(*a))
    _, cu, slot = tables(lens, slots)
    state, out = before.to(DEV), torch.empty((sum(lens), H, V), device=DEV)
    ops.delta_rule(qkv.to(DEV), gates.to(DEV), 2, H, a_log.to(DEV), dt_bias.to(DEV), state, 7, cu, slot, out, H, G, D, V,
                   decay=decay.to(DEV), per_channel=per_channel)
    assert ran == [1]
    return out, state


def check(out, state, H, G, D, V, lens, slots, qkv, gates, decay, a_log, dt_bias, before, bound):
    cu, wide = tables(lens, slots)[0], dt_bias.numel()
    unit = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    for s, (n, slot) in enumerate(zip(lens, slots)):
        rows = slice(cu[s], cu[s + 1])
        if slot < 0:
            assert float(out[rows].abs().max()) == 0
            continue
        if n == 0:
            continue
        x = qkv[rows].double()
        q = unit(x[:, :G * D].view(n, G, D)).repeat_interleave(H // G, 1) * D ** -0.5
        k = unit(x[:, G * D:2 * G * D].view(n, G, D)).repeat_interleave(H // G, 1)
        step = torch.nn.functional.softplus(decay[rows, 2:2 + wide].double() + dt_bias.double(), threshold=40).view(n, H, -1)
        g = torch.exp(-torch.exp(a_log.double()).view(1, H, 1) * step).expand(n, H, D)
        want, S = ps.delta_rule(q, k, x[:, 2 * G * D:].view(n, H, V), torch.sigmoid(gates[rows, H:2 * H].double()), g,
                                before[slot, 7:].double().view(H, D, V))
        for got, exact in ((out[rows], want), (state[slot, 7:].view(H, D, V), S)):
            off = float((got.double().cpu() - exact).norm() / exact.norm())
            assert off <= bound, off
    idle = [s for s in range(5) if s not in slots]
    assert torch.equal(state.cpu()[idle], before[idle])


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("H,G,D,V,lens,slots", [
    (2, 1, 128, 128, [65, 1, 64, 200], [3, 0, 1, 4]), (4, 2, 64, 48, [129, 0, 63], [2, 3, 0]), (3, 3, 128, 16, [70], [1]),
    (2, 2, 64, 192, [5, 66], [-1, 2]), (1, 1, 128, 112, [400], [0])])
@pytest.mark.parametrize("pace", [-4.0, 0.0, 6.0])
def test_chunks_against_float64(per_channel, H, G, D, V, lens, slots, pace, monkeypatch):
    """``pace`` moves the decays: near one, about a half a token, and down to e^-60 a token.  A token's outputs are float32
    sums of at most D + 64 terms behind two triangular products."""
    T, wide = sum(lens), H * D if per_channel else H
    qkv, gates = rnd((T, 2 * G * D + H * V), 1), rnd((T, 2 * H + 1), 2)
    decay, a_log, dt_bias = rnd((T, wide + 3), 3) + pace, 2 * torch.rand((H,), generator=torch.Generator().manual_seed(4)), rnd((wide,), 5, 0.3)
    given = qkv, gates, decay, a_log, dt_bias, rnd((5, 7 + H * D * V), 6, 0.3)
    sizes = H, G, D, V, lens, slots
    check(*chunked(gpu_ops(), monkeypatch, per_channel, *sizes, *given), *sizes, *given, 1e-6)


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("forgets", [lambda t: t % 16 < 1, lambda t: t % 16 < 14, lambda t: t % 2 == 0, lambda t: t % 10 == 3])
def test_chunks_forget_then_hold(per_channel, D, forgets, monkeypatch):
    """Tokens that forget by e^-100 among tokens that keep nearly everything: the weights between those that keep are as
    exact as where nobody forgets, however large the sum of logarithms before them."""
    H, G, V, lens, slots = 2, 1, 32, [150, 90], [2, 0]
    T, wide = sum(lens), H * D if per_channel else H
    strong = torch.tensor([forgets(t) for n in lens for t in range(n)])
    decay = torch.where(strong[:, None], 12.5, -7.0) + rnd((T, wide + 3), 3, 0.3)
    a_log, dt_bias = torch.full((H,), 8.0).log(), rnd((wide,), 5, 0.1)
    given = rnd((T, 2 * G * D + H * V), 1), rnd((T, 2 * H + 1), 2), decay, a_log, dt_bias, rnd((5, 7 + H * D * V), 6, 0.3)
    sizes = H, G, D, V, lens, slots
    check(*chunked(gpu_ops(), monkeypatch, per_channel, *sizes, *given), *sizes, *given, 1e-6)


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("D,V", [(64, 48), (128, 32)])
@pytest.mark.parametrize("what", ["q", "k", "v", "beta", "decay", "state"])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("where", [5, 64 + 21, 79])
def test_what_is_not_finite_stays_behind_its_token(per_channel, D, V, what, value, where, monkeypatch):
    """A NaN or an infinity in a token's input reaches that token and those behind it and nothing else: the same outputs and
    entries of the state are finite as in the walk token by token, and those are close to it."""
    ops = gpu_ops()
    H, G, lens, slots = 2, 1, [150, 90], [2, 0]
    T, wide = sum(lens), H * D if per_channel else H
    qkv, gates, decay = rnd((T, 2 * G * D + H * V), 1), rnd((T, 2 * H + 1), 2), rnd((T, wide + 3), 3)
    before = rnd((5, 7 + H * D * V), 6, 0.3)
    {"q": qkv, "k": qkv, "v": qkv, "beta": gates, "decay": decay, "state": before}[what][
        2 if what == "state" else where, {"q": 3, "k": D + 9, "v": 2 * D + V + 17, "beta": H + 1, "decay": 2 + wide // 2, "state": 7 + 5}[what]] = value
    sizes, given = (H, G, D, V, lens, slots), (qkv, gates, decay, rnd((H,), 4, 0.3), rnd((wide,), 5, 0.3), before)
    got = chunked(ops, monkeypatch, per_channel, *sizes, *given)
    monkeypatch.setattr(ops, "use_delta_chunks", False)
    _, cu, slot = tables(lens, slots)
    state, out = before.to(DEV), torch.empty((T, H, V), device=DEV)
    ops.delta_rule(qkv.to(DEV), gates.to(DEV), 2, H, given[3].to(DEV), given[4].to(DEV), state, 7, cu, slot, out, H, G, D, V,
                   decay=decay.to(DEV), per_channel=per_channel)
    assert what == "state" or bool(out[:where].isfinite().all())
    for mine, walk in zip(got, (out, state)):
        held = walk.isfinite()
        assert torch.equal(mine.isfinite(), held)
        assert float((mine[held] - walk[held]).norm()) <= 1e-6 * float(walk[held].norm())


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("step", [0, -1, 1, 200])
@pytest.mark.parametrize("others", [[1] * 24, [500], [1, 127, 128, 255, 256, 3]])
def test_a_request_is_worked_alike_alone_and_beside_others(per_channel, D, step, others):
    """Walk or chunks is a matter of a request's own tokens: around the number where one gives way to the other, outputs
    and state have the same bits alone and in steps with single tokens, shorter and longer portions."""
    ops = gpu_ops()
    n = ops.DELTA_CHUNKS_FROM[per_channel] + step
    H, G, V = 2, 1, 32
    for lens in ([n] + others, others + [n]):
        at, place, T = sum(lens[:lens.index(n)]), lens.index(n), sum(lens)
        wide = H * D if per_channel else H
        qkv, gates, decay = rnd((T, 2 * G * D + H * V), 1), rnd((T, 2 * H + 1), 2), rnd((T, wide + 3), 3)
        a_log, dt_bias = rnd((H,), 4, 0.3).to(DEV), rnd((wide,), 5, 0.3).to(DEV)
        got = []
        for rows, some in ((slice(0, T), lens), (slice(at, at + n), [n])):
            _, cu, slots = tables(some, list(range(len(some))) if len(some) > 1 else [place])
            state = rnd((len(lens), 7 + H * D * V), 6, 0.3).to(DEV)
            out = torch.empty((sum(some), H, V), device=DEV)
            ops.delta_rule(qkv[rows].contiguous().to(DEV), gates[rows].contiguous().to(DEV), 2, H, a_log, dt_bias, state, 7, cu,
                           slots, out, H, G, D, V, decay=decay[rows].contiguous().to(DEV), per_channel=per_channel,
                           max_q_len=max(some), min_q_len=min(some))
            got.append((out if len(some) == 1 else out[at:at + n], state[place]))
        for whole, alone in zip(*got):
            assert torch.equal(whole, alone)


@pytest.mark.parametrize("per_channel", [False, True])
def test_chunks_begin_where_they_are_said_to(per_channel, monkeypatch):
    """Which kernels a step launches: by the longest and the shortest request, whatever the number of either."""
    ops = gpu_ops()
    least = ops.DELTA_CHUNKS_FROM[per_channel]
    H, G, D, V = 2, 1, 64, 16
    ran = []
    for name in ("atom_delta_chunks", "atom_delta_rule"):
        monkeypatch.setattr(ops.lib, name, lambda *a, name=name, kernel=getattr(ops.lib, name): ran.append(name) or kernel(*a))
    for lens, want in (([least], ["atom_delta_chunks"]), ([least - 1] * 3, ["atom_delta_rule"]), ([1] * 40, ["atom_delta_rule"]),
                       ([least, 2 * least], ["atom_delta_chunks"]), ([1] * 40 + [least], ["atom_delta_chunks", "atom_delta_rule"])):
        T, wide = sum(lens), H * D if per_channel else H
        _, cu, slots = tables(lens, list(range(len(lens))))
        state, out = torch.zeros((len(lens), H * D * V), device=DEV), torch.empty((T, H, V), device=DEV)
        ran.clear()
        ops.delta_rule(rnd((T, 2 * G * D + H * V), 1).to(DEV), rnd((T, H), 2).to(DEV), 0, 0, rnd((H,), 4).to(DEV),
                       rnd((wide,), 5).to(DEV), state, 0, cu, slots, out, H, G, D, V, decay=rnd((T, wide), 3).to(DEV),
                       per_channel=per_channel, max_q_len=max(lens), min_q_len=min(lens))
        assert ran == want
        assert bool(out.isfinite().all())


@pytest.mark.parametrize("per_channel", [False, True])
@pytest.mark.parametrize("room", [1, 2, 5, 9, 1000])
def test_bounded_scratch_memory(per_channel, room, monkeypatch):
    """Places beyond the scratch memory's bound are worked afterwards in the same memory, with the same bits, wherever the
    bound cuts a request."""
    ops = gpu_ops()
    H, G, D, V, lens, slots = 2, 1, 64, 48, [300, 0, 64, 65, 511, 1], [0, 4, 2, -1, 3, 1]
    T, wide = sum(lens), H * D if per_channel else H
    given = (rnd((T, 2 * G * D + H * V), 1), rnd((T, 2 * H + 1), 2), rnd((T, wide + 3), 3), rnd((H,), 4, 0.3), rnd((wide,), 5, 0.3),
             rnd((5, 7 + H * D * V), 6, 0.3))
    whole = chunked(ops, monkeypatch, per_channel, H, G, D, V, lens, slots, *given)
    monkeypatch.undo()
    place = 4 * ops.lib.atom_delta_chunks_floats(H, D, V)
    monkeypatch.setattr(ops, "DELTA_SCRATCH_BYTES", room * place + 4, raising=False)
    taken, empty = [], torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: taken.append(empty(*a, **k)) or taken[-1])
    cut = chunked(ops, monkeypatch, per_channel, H, G, D, V, lens, slots, *given)
    assert max(t.numel() * 4 for t in taken if t.shape[-1] * 4 == place) <= room * place
    for a, b in zip(whole, cut):
        assert torch.equal(a, b)
