"""Linear recurrences with one decay per head over runs of 64 tokens: the matrix-core kernels against float64 and against
the walk token by token (which takes the same rows where they do not begin at multiples of 16 bytes)."""

import pytest
import torch

import plain_leduvik as pl
from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


def scan(ops, H, G, K, V, lens, slots, raw, bias, a_log, skip, x, odd):
    """The outputs and the state after the step; ``odd``: the rows begin at odd places, so the walk takes them."""
    C = H * V + 2 * G * K
    rows = torch.zeros((sum(lens), C + (1 if odd else 4)))
    rows[:, :C] = x
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    state = rnd((5, 7 + H * K * V), 9, 0.5).to(DEV)
    out = torch.empty((sum(lens), H * V), device=DEV)
    d = rows.to(DEV)
    ops.linear_scan(d, H * V + G * K, G, d, H * V, G, d, 0, raw.to(DEV), 2, state, 7, i32(cu), i32(slots), out, H, K, V,
                    per_channel=False, skip=skip.to(DEV), max_q_len=max(lens), step_bias=bias.to(DEV), a_log=a_log.to(DEV))
    return out.double().cpu(), state.double().cpu()


@pytest.mark.parametrize("H,G,K,V,lens,slots", [
    (4, 1, 128, 64, [65, 1, 64, 300], [3, 0, 1, 4]), (8, 2, 64, 48, [129, 0, 63], [2, 3, 0]), (3, 3, 96, 16, [200], [1]),
    (16, 1, 80, 128, [70, 66], [-1, 2]), (2, 1, 64, 80, [1000], [0])])
@pytest.mark.parametrize("pace", [0.0, -4.0, 3.0])
def test_runs_against_float64_and_the_walk(H, G, K, V, lens, slots, pace):
    """``pace`` moves the step sizes: decays of about a half, near one, and down to e^-30 a token."""
    ops = gpu_ops()
    T = sum(lens)
    x = rnd((T, H * V + 2 * G * K), 1)
    raw, bias = rnd((T, H + 3), 2), rnd((H,), 3, 0.3) + pace
    a_log, skip = torch.log(1 + 7 * torch.rand((H,), generator=torch.Generator().manual_seed(4))), rnd((H,), 5)
    got, state = scan(ops, H, G, K, V, lens, slots, raw, bias, a_log, skip, x, odd=False)
    walked, walked_state = scan(ops, H, G, K, V, lens, slots, raw, bias, a_log, skip, x, odd=True)
    assert not torch.equal(got, walked)      # two kernels, two orders of sums
    before = rnd((5, 7 + H * K * V), 9, 0.5).double()
    at = 0
    for n, slot in zip(lens, slots):
        rows = slice(at, at + n)
        at += n
        if slot < 0 or n == 0:
            continue
        xx, kk, rr = x[rows].double().split([H * V, G * K, G * K], -1)
        dt = pl.softplus(raw[rows, 2:2 + H].double() + bias.double())
        want, S = pl.state_space_recurrence(xx.reshape(n, H, V), kk.reshape(n, G, K), rr.reshape(n, G, K), dt,
                                            torch.exp(a_log.double()), skip.double(), before[slot, 7:].reshape(H, K, V))
        for mine, walk, exact in ((got[rows], walked[rows], want.reshape(n, -1)),
                                  (state[slot, 7:], walked_state[slot, 7:], S.reshape(-1))):
            off, walk_off = (float((m - exact).norm() / exact.norm()) for m in (mine, walk))
            # float32 sums of up to K + 64 terms behind decays whose logarithms carry a rounding of the largest of them
            assert off <= 3e-6 and off <= 2 * walk_off + 2e-7, (off, walk_off)
    idle = [s for s in range(5) if s not in slots]
    assert torch.equal(state[idle], before.float().double()[idle])


@pytest.mark.parametrize("H,G,K,V", [(4, 2, 64, 48), (2, 1, 128, 64)])
@pytest.mark.parametrize("what", ["v", "k", "r", "step"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), 1e30])
@pytest.mark.parametrize("where", [5, 64 + 21, 79])
def test_what_is_not_finite_stays_behind_its_token(H, G, K, V, what, value, where):
    """A NaN, an infinity or a huge number in a token's input reaches that token and those behind it and nothing else: the
    same outputs and entries of the state are finite as in the walk token by token, and each token's are close to it."""
    ops = gpu_ops()
    lens, slots = [150, 90], [2, 0]
    T = sum(lens)
    x, raw, bias = rnd((T, H * V + 2 * G * K), 1), rnd((T, H + 3), 2), rnd((H,), 3, 0.3) - 2
    (raw if what == "step" else x)[where, {"v": V + 17, "k": H * V + 3, "r": H * V + G * K + 9, "step": 3}[what]] = value
    a_log, skip = torch.log(1 + 7 * torch.rand((H,), generator=torch.Generator().manual_seed(4))), rnd((H,), 5)
    mine, walk = (scan(ops, H, G, K, V, lens, slots, raw, bias, a_log, skip, x, odd=odd) for odd in (False, True))
    assert bool(walk[0][:where].isfinite().all())
    for got, want in zip(mine, walk):
        held = want.isfinite()
        assert torch.equal(got.isfinite(), held)
        got, want = (torch.where(held, z, 0.0) for z in (got, want))
        # a token's row (a slot's of the state): float32 sums of K + 64 terms of the size of its largest outputs; behind a huge
        # number a row is one product r . k scaled, whose own terms cancel by up to two digits
        bound = 1e-3 if value == 1e30 else 1e-5
        assert bool(((got - want).norm(dim=1) <= bound * want.norm(dim=1)).all())


@pytest.mark.parametrize("H,G,K,V", [(4, 2, 64, 48), (16, 1, 128, 64)])
@pytest.mark.parametrize("n", [1, 17, 64, 65, 200])
@pytest.mark.parametrize("others", [[1] * 24, [500], [3, 64, 65, 128]])
def test_a_request_is_worked_alike_alone_and_beside_others(H, G, K, V, n, others):
    """Walk or runs is a matter of a request's own tokens: outputs and state have the same bits alone and in steps with single
    tokens, shorter and longer portions, before it and behind it, a padded request among them."""
    ops = gpu_ops()
    for lens in ([n, 2] + others, others + [2, n]):
        place, pad, T = (0, 1, sum(lens)) if lens[0] == n else (len(lens) - 1, len(lens) - 2, sum(lens))
        at = sum(lens[:place])
        x, raw = rnd((T, H * V + 2 * G * K + 4), 1).to(DEV), rnd((T, H), 2).to(DEV)
        bias, a_log, skip = rnd((H,), 3, 0.3).to(DEV), rnd((H,), 4, 0.3).to(DEV), rnd((H,), 5).to(DEV)
        slots = [-1 if s == pad else s for s in range(len(lens))]
        got = []
        for rows, some, slot in ((slice(0, T), lens, slots), (slice(at, at + n), [n], [place])):
            i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
            state = rnd((len(lens), 7 + H * K * V), 6, 0.3).to(DEV)
            out = torch.full((sum(some), H * V), float("nan"), device=DEV)
            part = x[rows].contiguous()
            cu = [sum(some[:i]) for i in range(len(some) + 1)]
            ops.linear_scan(part, H * V + G * K, G, part, H * V, G, part, 0, raw[rows].contiguous(), 0, state, 7, i32(cu), i32(slot),
                            out, H, K, V, per_channel=False, skip=skip, max_q_len=max(some), step_bias=bias, a_log=a_log)
            assert bool(out.isfinite().all())
            got.append((out[at:at + n] if len(some) > 1 else out, state[place]))
        for beside, alone in zip(*got):
            assert torch.equal(beside, alone)
