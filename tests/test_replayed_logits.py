"""Whose the logits of a replayed step are: the graph's own output only for the first rows of a step of single tokens."""

from types import SimpleNamespace

import pytest
import torch

from atom_amd.engine.graphs import DecodeGraphs


class _Copied:
    def record(self):
        pass


def replayed(shape, rows, wants):
    """The logits of a step whose entries have these rows of the graph's output, after the next replay has written it anew."""
    graphs = DecodeGraphs.__new__(DecodeGraphs)
    graphs.replays = graphs.mixed_replays = 0
    first = torch.arange(24.0).view(8, 3)
    cap = SimpleNamespace(dev=torch.zeros(4), host=torch.zeros(4), copied=_Copied(), copy_pending=False, logits=first.clone(),
                          graph=SimpleNamespace(replay=lambda: None))
    graphs.shape_for, graphs.captured, graphs._fill = lambda e: shape, {shape: cap}, lambda *a: rows
    out = graphs.run([SimpleNamespace(want=[0] if w else []) for w in wants], [0] * len(rows))
    want = first[[r for r, w in zip(rows, wants) if w]]
    assert torch.equal(out, want)
    cap.logits.fill_(-1)
    return torch.equal(out, want)


@pytest.mark.parametrize("shape,rows,wants", [((0, 0, 8), [0, 1, 2, 3], [0, 0, 1, 1]), ((0, 0, 8), [0, 1, 2], [0, 1, 0]),
                                              ((0, 0, 8), [0, 1, 2, 3], [1, 0, 1, 1]), ((16, 2, 4), [0, 2, 3], [0, 1, 1]),
                                              ((16, 2, 4), [0, 1], [1, 1])])
def test_logits_that_stay_the_callers(shape, rows, wants):
    assert replayed(shape, rows, wants)


def test_logits_that_are_the_graphs():
    assert not replayed((0, 0, 8), [0, 1, 2], [1, 1, 0])
