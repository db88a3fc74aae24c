"""The states before the runs of a linear recurrence: blocks of 64 and of 32 value columns, several heads a block where the outputs
are read, against float64 and with the same bits whichever the launch takes."""

import pytest
import torch

import plain_leduvik as pl
from helpers import gpu_ops
from test_gpu_scan_runs import rnd, scan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,G,K,V", [(72, 3, 128, 64), (100, 2, 80, 48), (48, 1, 112, 80)])
def test_wide_and_narrow_blocks(H, G, K, V):
    """Together the requests' blocks of 64 columns are more than the CUs, alone they are fewer (and the blocks of 32): two
    channels' tiles at an odd end, runs of one, two and 63 tokens at the end of a request."""
    ops = gpu_ops()
    lens, slots = [193, 66, 129, 191], [3, 0, 4, 1]
    squares = -(-K // 64) * -(-V // 64)
    assert H * squares * len(lens) >= ops.num_cus > H * squares
    x, raw, bias = rnd((sum(lens), H * V + 2 * G * K), 1), rnd((sum(lens), H + 3), 2), rnd((H,), 3, 0.3) - 3
    a_log, skip = torch.log(1 + 7 * torch.rand((H,), generator=torch.Generator().manual_seed(4))), rnd((H,), 5)
    got, state = scan(ops, H, G, K, V, lens, slots, raw, bias, a_log, skip, x, odd=False)
    before, at = rnd((5, 7 + H * K * V), 9, 0.5).double(), 0
    for n, slot in zip(lens, slots):
        rows = slice(at, at + n)
        at += n
        alone, alone_state = scan(ops, H, G, K, V, [n], [slot], raw[rows], bias, a_log, skip, x[rows], odd=False)
        assert torch.equal(got[rows], alone) and torch.equal(state[slot], alone_state[slot])
        xx, kk, rr = x[rows].double().split([H * V, G * K, G * K], -1)
        dt = pl.softplus(raw[rows, 2:2 + H].double() + bias.double())
        want, S = pl.state_space_recurrence(xx.reshape(n, H, V), kk.reshape(n, G, K), rr.reshape(n, G, K), dt,
                                            torch.exp(a_log.double()), skip.double(), before[slot, 7:].reshape(H, K, V))
        for mine, exact in ((got[rows], want.reshape(n, -1)), (state[slot, 7:], S.reshape(-1))):
            # float32 sums of up to K + 64 terms behind decays whose logarithms carry a rounding of the largest of them
            assert float((mine - exact).norm() / exact.norm()) <= 3e-6
