"""Per-head products of many tokens, and the float32 product of any number, on the matrix cores (64 tokens by 128 columns a
block, K in stages of 64 through two buffers in LDS): one to five stages with whole and cut ends, edges of the tiles, gates and
strides, against float64 sums over the operands as they are multiplied (a float32 input rounded to bfloat16, or as it is)."""

import pytest
import torch

from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TYPES = [torch.float32, torch.bfloat16]


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


@pytest.mark.parametrize("k", [8, 64, 72, 128, 136, 192, 200, 256, 264])
@pytest.mark.parametrize("heads,m,n,gated", [(1, 96, 8, ""), (3, 129, 128, "head"), (8, 130, 136, "entry"), (2, 193, 250, "entry")])
@pytest.mark.parametrize("x_type,exact", [(torch.float32, False), (torch.bfloat16, False), (torch.float32, True)])
@pytest.mark.parametrize("y_type", TYPES)
def test_per_head_products_of_many_tokens(heads, m, n, gated, k, x_type, exact, y_type):
    ops = gpu_ops()
    m = m - 80 if exact else m      # 16 to 113: with the cut last block, and one that is nearly empty
    hsx, hsy = k + 8, n + (8 if n % 8 == 0 else 3)
    ldx, ldy = heads * hsx + 8, heads * hsy
    x = rnd((m, ldx), 1).to(x_type)
    w = rnd((heads, n, k), 2, k ** -0.5).to(torch.bfloat16)
    y = torch.full((m, ldy), 7.0, dtype=y_type, device=DEV)
    gate = {"": None, "head": rnd((m, heads), 3), "entry": rnd((m, heads * n), 3)}[gated]
    ops.heads_gemm(x.to(DEV), 8, ldx, hsx, w.to(DEV), y, 0, ldy, hsy, heads, m, n, k, alpha=0.7,
                   gate=None if gate is None else gate.to(DEV), ldg=0 if gate is None else gate.shape[1], gate_entries=gated == "entry", exact=exact)
    y = y.cpu().double()
    taken = x.double() if exact else x.to(torch.bfloat16).double()
    for h in range(heads):
        a, b = taken[:, 8 + h * hsx:8 + h * hsx + k], w[h].double()
        want, terms = 0.7 * a @ b.T, 0.7 * a.abs() @ b.abs().T
        if gated:
            g = torch.sigmoid(gate.double()[:, h * n:(h + 1) * n] if gated == "entry" else gate.double()[:, h:h + 1])
            want, terms = want * g, terms * g
        # k float32 additions (three pieces: 3 k) and a few more roundings (alpha, the gate) of the sum's terms; half a unit of a
        # bfloat16 result
        bound = ((3 * k if exact else k) + 8) * 2.0 ** -24 * terms + (2.0 ** -8 * want.abs() if y_type is torch.bfloat16 else 0.0) + 1e-30
        got = y[:, h * hsy:h * hsy + n]
        assert bool(((got - want).abs() <= bound).all()), f"head {h}: {float(((got - want).abs() / bound).max()):.2f} of the bound"
        assert bool((y[:, h * hsy + n:(h + 1) * hsy] == 7.0).all()), "columns between the heads' were written"


def test_more_columns_than_a_grids_first_dimension_holds_blocks():
    """2^31 columns of two heads and a few more: the heads in the grid's third dimension."""
    from atom_amd.kernels.hip import HipKernels

    if torch.cuda.mem_get_info(DEV)[0] < 48 << 30:
        pytest.skip("34 GB of weights")
    ops = HipKernels(DEV)
    ops.heads_split_from = 1
    heads, k, n = 2, 8, (1 << 30) + 64
    x = rnd((1, heads * k), 1).to(DEV)
    w = torch.empty((heads, n, k), dtype=torch.bfloat16, device=DEV).normal_()
    y = torch.empty((1, heads * n), dtype=torch.bfloat16, device=DEV)
    ops.heads_gemm(x, 0, heads * k, k, w, y, 0, heads * n, n, heads, 1, n, k, exact=True)
    for h in range(heads):
        for at in (0, n // 2 - 77, n - 300):
            want = w[h, at:at + 300].double() @ x[0, h * k:(h + 1) * k].double()
            got = y[0, h * n + at:h * n + at + 300].double()
            terms = w[h, at:at + 300].double().abs() @ x[0, h * k:(h + 1) * k].double().abs()
            assert bool(((got - want).abs() <= (3 * k + 8) * 2.0 ** -24 * terms + 2.0 ** -8 * want.abs()).all()), (h, at)
    del w, y
    torch.cuda.empty_cache()
