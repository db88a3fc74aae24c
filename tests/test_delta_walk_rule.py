"""How many value columns a block of the delta rule's walk takes: by the requests that walk, not by those in the step."""

from types import SimpleNamespace

import pytest
import torch

from atom_amd.kernels.hip import HipKernels

FROM = HipKernels.DELTA_CHUNKS_FROM[False]


def chosen(lens, heads, vdim, told: bool) -> int:
    """The columns that ``delta_rule`` launches with for these requests; ``told``: their lengths are known on the host."""
    ops, seen = HipKernels.__new__(HipKernels), []
    ops._check = lambda name, t, *rest: t
    ops._stream = lambda: None
    ops.num_cus, ops.use_delta_chunks = 256, True

    def chunks(*args):
        seen.append(args[-2])
        return 0

    ops.lib = SimpleNamespace(atom_delta_chunks=chunks, atom_delta_rule=lambda *a: 0, atom_delta_chunks_supports=lambda d, v: 1,
                              atom_delta_chunks_floats=lambda h, d, v: 1)
    T, S = sum(lens), len(lens)
    f = lambda *shape: torch.empty(shape)  # noqa: E731
    known = {"max_q_len": max(lens), "walkers": ops.delta_walkers(lens, False)} if told else {}
    ops.delta_rule(f(T, 1), f(T, 2 * heads), 0, heads, f(heads), f(heads), f(9, 1), 0, torch.empty(S + 1, dtype=torch.int32),
                   torch.empty(S, dtype=torch.int32), f(T, heads, vdim), heads, heads, 128, vdim, **known)
    return seen[0]


@pytest.mark.parametrize("lens,columns", [([2048], 16), ([2048, 1, 1], 16), ([2048] + 31 * [1], 16), ([2048, FROM, FROM], 16),
                                          ([2048, FROM - 1, FROM - 1, FROM - 1], 16), ([1024, 1024], 16), ([1024] * 3, 32),
                                          ([2048, 1099, 1685, 736], 32), ([2048] + 8 * [1000], 32)])
def test_columns_by_the_requests_that_walk(lens, columns):
    assert chosen(lens, 16, 128, True) == columns
    assert chosen(lens, 16, 112, True) == 16      # no whole pairs of tiles


def test_columns_without_lengths_by_the_most_requests_that_may_walk():
    assert chosen([4 * FROM] + 60 * [1], 16, 128, False) == 32      # four may
    assert chosen([FROM, FROM], 16, 128, False) == 16
    assert chosen([2 * FROM] + 60 * [1], 16, 128, False) == 16
