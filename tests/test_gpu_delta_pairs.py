"""The delta rule's chunks with two tiles of value columns a block, which steps with more blocks of one tile than CUs take: the
bits of one tile a block, and float64's numbers."""

import pytest
import torch

from helpers import gpu_ops
from test_gpu_delta_chunks import check, chunked, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,V", [(64, 96), (128, 128), (128, 32)])
def test_two_tiles_a_block(D, V, monkeypatch):
    ops = gpu_ops()
    lens, slots, G = [130, 64, 1, 77], [3, 0, -1, 4], 2
    H = 2 * (ops.num_cus // (2 * (V // 16) * len(lens)) + 1)
    assert H * (V // 16) * len(lens) > ops.num_cus >= H * (V // 16)
    T = sum(lens)
    qkv, gates, decay = rnd((T, 2 * G * D + H * V), 1), rnd((T, 2 * H + 1), 2), rnd((T, H + 3), 3)
    a_log, dt_bias, before = rnd((H,), 4, 0.5), rnd((H,), 5, 0.3), rnd((5, 7 + H * D * V), 6, 0.3)
    qkv[140, 2 * G * D + 5] = float("nan")     # a value of the second request's eleventh token
    out, state = chunked(ops, monkeypatch, False, H, G, D, V, lens, slots, qkv, gates, decay, a_log, dt_bias, before)
    at = 0
    for n, slot in zip(lens, slots):
        if slot >= 0:
            rows = slice(at, at + n)
            alone = chunked(ops, monkeypatch, False, H, G, D, V, [n], [slot], qkv[rows], gates[rows], decay[rows], a_log, dt_bias,
                            before)
            assert torch.equal(out[rows].nan_to_num(7.0), alone[0].nan_to_num(7.0))
            assert torch.equal(state[slot].nan_to_num(7.0), alone[1][slot].nan_to_num(7.0))
        at += n
    qkv[140, 2 * G * D + 5] = 0.3
    given = qkv, gates, decay, a_log, dt_bias, before
    check(*chunked(ops, monkeypatch, False, H, G, D, V, lens, slots, *given), H, G, D, V, lens, slots, *given, 1e-6)
