"""Float32 products as sums of bfloat16 pieces: the products through LDS and without agree to the bit, their error is that of
float32 sums, and operands whose pieces say nothing (infinities, NaN, numbers near the ends of the range) are summed again."""

import pytest
import torch

from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).to(DEV)


def through_lds(ops, x, w):
    return ops._f32_scratch(x, w, x.shape[0], w.shape[0], x.shape[1]) is not None


# K of one step, of a last slice that is short, of slices that are empty; rows and columns at the edges of both tiles; two portions
@pytest.mark.parametrize("m,n,k", [(449, 4099, 32), (449, 4096, 288), (512, 4100, 1056), (2112, 4096, 64), (465, 8192, 4096),
                                   (100, 30000, 32), (1000, 4160, 96), (129, 24580, 192), (1025, 8192, 4096)])
def test_wide_products_round_like_narrow_ones(m, n, k):
    ops = gpu_ops()
    x, w, b = rnd((m, k), 1), rnd((n, k), 2), rnd((n,), 3)
    assert through_lds(ops, x, w)
    y = ops.linear(x, w, b)
    want = x.double() @ w.double().T + b.double()
    assert float((y.double() - want).norm() / want.norm()) <= 2.0 ** -24 * (4 + (k / 128) ** 0.5)
    if k >= 1024:   # what is off is off independently row by row: the rows' mean is off by less (three deviations of it)
        off = y.double() - want
        assert float(off.mean(0).norm()) <= 3 * float(off.norm()) / m
    for rows in (slice(0, 1), slice(m - 1, m), slice(m // 2, m // 2 + 20)):
        assert torch.equal(ops.linear(x[rows].contiguous(), w, b), y[rows])
    gate = ops.linear_silu(x, w[:n // 2 * 2].contiguous())
    assert torch.equal(ops.linear_silu(x[:3].contiguous(), w[:n // 2 * 2].contiguous()), gate[:3])


@pytest.mark.parametrize("m,n,k", [(3, 70, 96), (449, 4096, 96)])
def test_values_that_pieces_cannot_hold(m, n, k):
    ops = gpu_ops()
    x, w = rnd((m, k), 1), rnd((n, k), 2)
    inf, nan = float("inf"), float("nan")
    x[0, 5], x[1, 7], x[2, 9] = inf, nan, 3.4e38          # hi of the last is infinite
    w[:, 9] *= 1e-6
    w[3, 5], w[4, 5], w[5, 11], w[6, 13] = 0.0, -1.0, -inf, nan
    y = ops.linear(x, w).cpu()
    terms = x.cpu().double()[:, None] * w.cpu().double()[None, :40]
    want = terms.sum(-1)
    assert torch.equal(y[:, :40].isnan(), want.isnan()) and torch.equal(y[:, :40].isinf(), want.isinf())
    held = want.isfinite()
    off = (y[:, :40].double() - want).abs()
    assert bool((off <= (32 + k / 32) * 2.0 ** -24 * terms.abs().sum(-1))[held].all())
    if m <= 40:
        assert int(held.sum()) > 10


@pytest.mark.parametrize("m,n,k", [(3, 70, 96), (449, 4096, 96)])
def test_numbers_below_the_range_of_pieces(m, n, k):
    ops = gpu_ops()
    x, w = rnd((m, k), 1, 2.0 ** -118), rnd((n, k), 2)
    x[1] = 0.0
    y = ops.linear(x, w).cpu()
    terms = x.cpu().double()[:, None] * w.cpu().double()[None, :40]
    assert float(y[1].abs().max()) == 0
    assert bool(((y[:, :40].double() - terms.sum(-1)).abs() <= (32 + k / 32) * 2.0 ** -24 * terms.abs().sum(-1) + 2.0 ** -149).all())


# results of ordinary size, one operand near an end of the range: x's entries about 2^x_exp, w's about 2^w_exp
@pytest.mark.parametrize("m,n,k", [(3, 70, 96), (449, 4096, 96), (20, 33, 1027)])
@pytest.mark.parametrize("x_exp,w_exp", [(-118, 63), (-122, 70), (-135, 50), (-140, 100), (63, -118), (90, -130), (112, -100), (-90, 118)])
def test_operands_near_the_ends_of_the_range(m, n, k, x_exp, w_exp):
    ops = gpu_ops()
    x, w = (torch.ldexp(rnd(s, seed).cpu().double(), torch.tensor(e)).float().to(DEV)
            for s, seed, e in (((m, k), 1, x_exp), ((n, k), 2, w_exp)))
    x[1] = 0.0
    y = ops.linear(x, w).cpu()
    terms = x.cpu().double()[:, None] * w.cpu().double()[None, :40]
    assert float(y[1].abs().max()) == 0
    assert bool(((y[:, :40].double() - terms.sum(-1)).abs() <= (32 + k / 32) * 2.0 ** -24 * terms.abs().sum(-1) + 2.0 ** -149).all())


@pytest.mark.parametrize("x_type,w_type", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("x_exp,w_exp", [(-122, 70), (70, -122), (110, -100), (-100, 110)])
def test_operands_of_two_types_near_the_ends_of_the_range(x_type, w_type, x_exp, w_exp):
    ops = gpu_ops()
    x, w = (torch.ldexp(rnd(s, seed).cpu().double(), torch.tensor(e)).to(t).to(DEV)
            for s, seed, e, t in (((5, 160), 1, x_exp, x_type), ((70, 160), 2, w_exp, w_type)))
    y = ops.linear(x, w, out_dtype=torch.float32).cpu()
    terms = x.cpu().double()[:, None] * w.cpu().double()[None]
    assert bool(((y.double() - terms.sum(-1)).abs() <= (32 + 160 / 32) * 2.0 ** -24 * terms.abs().sum(-1)).all())


# tiles of every kernel; K below four, ragged, of whole steps
@pytest.mark.parametrize("m,n,k", [(1, 70, 3), (3, 70, 1027), (9, 9000, 64), (30, 9000, 96), (40, 100, 130), (70, 5000, 100), (300, 3000, 96),
                                   (449, 4096, 64), (2100, 4100, 288)])
def test_results_that_are_not_finite_come_from_float32_sums(m, n, k):
    """Large operands whose results are ordinary numbers, beside infinities and NaN; a row's result is its own."""
    ops = gpu_ops()
    x, w = rnd((m, k), 1), rnd((n, k), 2, 2.0 ** -20)
    x[m // 2] *= 2.0 ** 122
    x[m - 1, k // 2], w[n // 2, k - 1] = float("inf"), float("nan")
    w[n - 1] *= 2.0 ** -70
    big, cols = m // 2, slice(max(0, n - 40), n)
    y = ops.linear(x, w)
    terms = x[big].cpu().double() * w[cols].cpu().double()
    if m > 1:
        off = (y[big, cols].cpu().double() - terms.sum(-1)).abs()
        held = terms.sum(-1).isfinite()
        assert bool((off <= (32 + k / 32) * 2.0 ** -24 * terms.abs().sum(-1))[held].all()) and int(held.sum()) >= 39
    assert not bool(y[m - 1].isfinite().any()) and bool(y[:, n // 2].isnan().all())
    for row in {0, big, m - 1}:
        assert torch.equal(ops.linear(x[row:row + 1].contiguous(), w)[0].nan_to_num(7.0), y[row].nan_to_num(7.0))
    w = w[:n // 2 * 2].contiguous()
    gate, want = ops.linear_silu(x, w), ops.linear(x, w)
    a, b = want[:, :n // 2], want[:, n // 2:]
    want = a / (1 + torch.exp(-a)) * b
    close = (gate - want).abs() <= 1e-5 * want.abs()
    assert bool((close | (gate == want) | (gate.isnan() & want.isnan())).all())


def test_results_that_are_not_finite_cost_little():
    ops = gpu_ops()

    def passes(x, w, n=3):
        events = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ops.linear(x, w)
        events[0].record()
        for _ in range(n):
            ops.linear(x, w)
        events[1].record()
        torch.cuda.synchronize()
        return events[0].elapsed_time(events[1])

    for m in (8, 465):
        x, w = rnd((m, 4096), 1), rnd((8192, 4096), 2)
        plain = passes(x, w)
        x[:, 7] = float("nan")
        assert passes(x, w) <= 15 * plain     # 5 to 6 times; summed one by one 30 and 130 times


def test_scratch_memory_is_within_what_the_cache_leaves_it():
    ops = gpu_ops()
    taken = 0
    for m in (65, 100, 465, 2048, 2049, 5000):
        for n, k in ((100, 32), (4096, 4096), (24576, 4096), (4096, 12288), (30000, 48)):
            size = ops.lib.atom_gemm_f32_scratch(None, 0, None, 0, m, n, k)
            assert size <= ops.product_scratch(m, k)
            taken += size == ops.product_scratch(m, k) > 0
    assert taken


# through linear (a float32 operand), and bfloat16 by bfloat16 where a caller asks for the float32 kernels
@pytest.mark.parametrize("x_type,w_type", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("m,n,k", [(1, 70, 1027), (9, 9000, 4096), (40, 300, 96), (300, 3000, 1040), (465, 4096, 4096)])
def test_products_of_other_types(m, n, k, x_type, w_type):
    """The error of float32 sums of a step's 32 terms, as float32 operands have it; a row does not depend on its batch."""
    ops = gpu_ops()
    x, w = rnd((m, k), 1).to(x_type), rnd((n, k), 2).to(w_type)
    y = ops._linear_f32(x, w, None, torch.float32, m, n, k)
    want = x.double() @ w.double().T
    off = float((y.double() - want).norm() / want.norm())
    print(f"{x_type} by {w_type}, {m} x {n} x {k}: {off:.3g}")
    assert off <= 2.0 ** -24 * (4 + (k / 128) ** 0.5)
    for row in {0, m // 2, m - 1}:
        assert torch.equal(ops._linear_f32(x[row:row + 1].contiguous(), w, None, torch.float32, 1, n, k)[0], y[row])
