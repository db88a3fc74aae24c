"""Scratch memory of a product belongs to it until its kernels are launched: the entry points let other threads run, which could be
handed the same memory and launch into it first."""

import weakref
from types import SimpleNamespace

import pytest
import torch

from atom_amd.kernels.hip import HipKernels


@pytest.mark.parametrize("entry", ["linear", "linear_silu"])
def test_the_pieces_of_a_float32_product_are_held_across_the_launch(entry):
    ops, seen = HipKernels.__new__(HipKernels), []
    ops._check = lambda name, t, *rest: t
    ops._stream = lambda: None
    ops._rows_takes = ops._skinny = lambda x, weight: False

    def scratch(x, weight, m, n, k):
        t = torch.empty(6 * m * k, dtype=torch.uint8)
        seen.append(weakref.ref(t))
        return t

    def launch(*args):
        assert seen[-1]() is not None, "given back before the launch"
        assert any(getattr(a, "value", None) == seen[-1]().data_ptr() for a in args)
        return 0

    ops._f32_scratch = scratch
    ops.lib = SimpleNamespace(atom_gemm_f32=launch, atom_gemm_f32_gate=launch)
    out = getattr(ops, entry)(torch.zeros(65, 32), torch.zeros(96, 32))
    assert len(seen) == 1 and out.shape == ((65, 96) if entry == "linear" else (65, 48))
    del out
    assert seen[-1]() is None
