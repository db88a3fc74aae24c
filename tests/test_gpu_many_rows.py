"""The bfloat16 product of many rows (``gemm_many.hip``): every tile, whole and cut along K, against the float64 product."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TILES = [(256, 256, 3), (192, 256, 3), (256, 192, 3), (256, 128, 3), (128, 256, 3), (128, 128, 4)]   # rows, columns, stages in LDS
# Float32 sums of k products, here at most 4,160, each sum off by 2^-24 of it: sqrt(k) 2^-24 = 3.9e-6 for random roundings; a
# result rounded to bfloat16 is off by up to 2^-8 of it.
SUMS, ROUNDED = 4e-6, 2.0 ** -8


def gpu_ops():
    from atom_amd.kernels.hip import HipKernels
    return HipKernels(DEV)


def operands(m, n, k, gate, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(m, k, generator=g, device=DEV, dtype=torch.bfloat16)
    w = torch.randn(n * (1 + gate), k, generator=g, device=DEV, dtype=torch.bfloat16) * k ** -0.5
    b = torch.randn(n * (1 + gate), generator=g, device=DEV)
    return x, w, b


def off(y, want):
    return float((y.double() - want).norm() / want.norm())


def activation(name):
    return {None: lambda v: v, "silu": torch.nn.functional.silu, "relu": torch.relu, "relu_squared": lambda v: torch.relu(v) ** 2,
            "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh")}[name]


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("m,n,k", [(1, 8, 512), (257, 264, 512), (300, 1000, 1024), (513, 776, 1088), (385, 520, 4160)])
def test_tiles(tile, m, n, k):
    ops, (bm, bn, stages) = gpu_ops(), TILES[tile]
    codes = {None: 0, "silu": 1, "relu": 2, "gelu_tanh": 3, "relu_squared": 4}
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None  # noqa: E731
    for gate, acts in ((0, (None, "relu_squared")), (1, ("silu", "relu", "gelu_tanh"))):
        x, w, b = operands(m, n, k, gate, tile)
        plain = x.double() @ w.double().T
        out = bn // 2 if gate else bn
        tiles = -(-m // bm) * -(-n // out)
        for whole, slices in {(tiles, 1), (0, 2), (tiles // 2, 3), (tiles - 1, 2)}:
            if (whole < tiles) != (slices > 1) or k // 64 // slices < stages:
                continue
            size = ops.lib.atom_gemm_many_scratch(m, n, gate, tile, whole, slices)
            for act in acts:
                for dtype, bias in ((torch.float32, b), (torch.bfloat16, None)):
                    parts = torch.full((max(size // 4, 4),), float("nan"), device=DEV)
                    y = torch.full((m + 1, n), 7.0, device=DEV, dtype=dtype)
                    status = ops.lib.atom_gemm_many(ptr(x), ptr(w), ptr(bias), ptr(y), ptr(parts), m, n, k, gate, codes[act],
                                                    int(dtype == torch.float32), tile, whole, slices, 0, stream)
                    assert status == 0
                    full = plain if bias is None else plain + bias.double()
                    want = activation(act)(full[:, :n]) * (full[:, n:] if gate else 1)
                    assert off(y[:m], want) < (SUMS if dtype == torch.float32 else ROUNDED), (gate, whole, slices, act, dtype)
                    assert bool((y[m] == 7).all()), "a row behind the last was written"
        if not gate and k // 64 // 2 >= stages:
            parts = torch.full((2, m, n), float("nan"), device=DEV)
            assert ops.lib.atom_gemm_many(ptr(x), ptr(w), None, None, ptr(parts), m, n, k, 0, 0, 0, tile, 0, 2, 1, stream) == 0
            assert off(parts.sum(0), plain) < SUMS


@pytest.mark.parametrize("m,n,k", [(257, 8192, 8192), (300, 2560, 9728), (1000, 4096, 5120), (2305, 1024, 8256), (536, 1544, 8192), (700, 3664, 2048)])
def test_products_of_the_engine(m, n, k):
    """As the parts call it: whole, as a sum of slices, with a bias, a gate and an activation, and replayed from a graph."""
    from atom_amd.kernels.hip import DeferredSum

    ops = gpu_ops()
    x, w, b = operands(m, n, k, 0, 5)
    assert ops._many(x, w) and ops._many_pays(m, n, k, None)
    plain = x.double() @ w.double().T
    limit = 2e-7 * k ** 0.5          # 2^-24 sqrt(k), three times that
    assert off(ops.linear(x, w, b), plain + b.double()) < ROUNDED
    y32 = ops.linear(x, w, b, out_dtype=torch.float32)
    assert off(y32, plain + b.double()) < limit
    lazy = ops.linear(x, w, b, defer=True)
    if n <= k:                       # a product that a reader adds: slices, by each of these plans
        assert isinstance(lazy, DeferredSum) and lazy.splits > 1 and lazy.bias is b
        assert off(lazy.partial.double().sum(0), plain) < limit
    else:
        assert isinstance(lazy, torch.Tensor) and off(lazy, plain + b.double()) < ROUNDED
    assert off(ops.linear_act(x, w, b, "relu_squared"), torch.relu(plain + b.double()) ** 2) < ROUNDED
    half = (plain + b.double()).split(n // 2, 1)
    # (gates of fewer than 321 rows, or of halves that are not eights, are the library's)
    gated = m >= 321 and n % 16 == 0
    assert ops._many_alone(x, w, b, torch.bfloat16, gate=True) == gated
    for name in ("silu", "relu", "gelu_tanh"):
        assert off(ops.linear_gated(x, w, b, name), activation(name)(half[0]) * half[1]) < ROUNDED
    assert off(ops.linear_silu(x, w, b), activation("silu")(half[0]) * half[1]) < ROUNDED
    free = plain.split(n // 2, 1)
    assert off(ops.linear_silu(x, w), activation("silu")(free[0]) * free[1]) < ROUNDED
    assert off(ops.linear_act(x, w, None, "relu"), torch.relu(plain)) < ROUNDED
    static, out = x.clone(), None
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.linear(static, w, b, out_dtype=torch.float32)
    for seed in (1, 2, 3):
        static.copy_(torch.randn(m, k, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV))
        graph.replay()
        assert torch.equal(out, ops.linear(static, w, b, out_dtype=torch.float32))


def test_plans():
    """Slices are whole stages, the parts stay within their bound, and every plan is one the kernel takes."""
    ops = gpu_ops()
    for m in (257, 536, 1048, 2305, 4111, 40000):
        for n, k in ((8, 512), (2560, 9728), (5120, 25600), (10240, 5120), (51200, 5120), (1000, 8192)):
            for gate in (0, 1):
                for apart in ((0,) if gate else (0, 1)):
                    plan = (ctypes.c_int * 4)()
                    assert ops.lib.atom_gemm_many_plan(m, n, k, gate, apart, 256, plan) == 0
                    tile, whole, slices, as_slices = plan
                    assert k // 64 // slices >= TILES[tile][2]
                    assert ops.lib.atom_gemm_many_scratch(m, n, gate, tile, whole, slices) <= ops.MANY_SCRATCH
                    assert not as_slices or (apart and whole == 0 and slices > 1)


def test_what_it_leaves_to_others():
    ops = gpu_ops()
    x, w, _ = operands(300, 1024, 8192, 0, 1)
    assert not ops._many(x[:256], w)                               # the tiles cut to the chip, or the library
    assert not ops._many(x, w[:1021])                              # columns in eights
    assert not ops._many(x[:, :8008], w[:, :8008])                 # whole stages
    odd = torch.empty(300 * 8192 + 1, device=DEV, dtype=torch.bfloat16)[1:].view(300, 8192)
    assert not ops._many(odd, w) and off(ops.linear(odd.copy_(x), w), x.double() @ w.double().T) < ROUNDED
    y = ops.linear(x, w)
    # results that are not finite stay in their rows and columns
    x[7, 100], w[9, 200] = float("inf"), float("nan")
    got = ops.linear(x, w)
    keep = torch.ones_like(got, dtype=torch.bool)
    keep[7], keep[:, 9] = False, False
    assert bool(got[:, 9].isnan().all()) and not bool(got[7].isfinite().any()) and torch.equal(got[keep], y[keep])


# Sizes whose plan hands slices on and sizes where it does not; (884, 3104, 4224) and (629, 6504, 11840) are such that the BLAS
# library's product would be cut in two.
@pytest.mark.parametrize("m,n,k", [(300, 2048, 2048), (536, 4096, 8192), (884, 3104, 4224), (629, 6504, 11840), (2305, 2048, 8192)])
@pytest.mark.parametrize("biased", [True, False])
@pytest.mark.parametrize("slices", [True, False])
def test_sums_for_a_reader_stay_float32(m, n, k, biased, slices):
    """A deferred product whose reader adds a bias, or slices that the library's product would leave, is handed on in float32."""
    from atom_amd.kernels.hip import DeferredSum

    ops = gpu_ops()
    x, w, b = operands(m, n, k, 0, 11)
    if not biased and not (slices and ops._library_slices(m, n, k) > 1):
        pytest.skip("the product is its tensor")
    lazy = ops.linear(x, w, b if biased else None, defer=True, slices=slices)
    assert isinstance(lazy, DeferredSum) and lazy.partial.dtype == torch.float32 and lazy.dtype == torch.bfloat16
    assert lazy.splits == 1 or slices
    assert (lazy.bias is b) if biased else (lazy.bias is None)
    want = x.double() @ w.double().T
    assert off(lazy.partial.double().sum(0), want) < 2e-7 * k ** 0.5
    assert off(ops.materialize(lazy), want + (b.double() if biased else 0)) < ROUNDED


# The lines of the rule that gives products to the kernel of large tiles: what the BLAS library finishes earlier stays with it.
@pytest.mark.parametrize("call,m,n,k,takes", [
    ("bias", 300, 640, 1536, False), ("bias", 384, 2048, 2048, True), ("bias32", 536, 1408, 1664, False), ("bias32", 300, 6144, 4096, False),
    ("bias32", 2048, 4096, 2048, True), ("bias deferred", 300, 2048, 2048, False), ("bias deferred", 300, 2048, 8192, True),
    ("relu", 384, 640, 1536, False), ("relu", 300, 6144, 4096, False), ("relu", 321, 6144, 4096, True), ("relu", 300, 2048, 8192, True),
    ("silu", 384, 640, 1536, False), ("silu", 320, 6144, 4096, False), ("silu", 321, 6144, 4096, True), ("silu bias", 321, 2048, 2048, True),
    ("gelu_tanh", 700, 640, 1536, False), ("gelu_tanh", 700, 4096, 2048, True),
    ("", 1024, 4096, 5120, True), ("", 1025, 4096, 5120, False), ("", 4111, 10240, 5120, True), ("", 2305, 10240, 5120, False),
    ("", 536, 16000, 3008, True), ("", 384, 16000, 3008, False), ("", 700, 4928, 4032, False), ("", 5569, 18704, 704, False),
    # K from 8,192 on: rounds of the library's tiles that are full, and single ones of more than nine 16ths of the CUs
    ("", 2048, 8192, 8192, False), ("", 1900, 7680, 8192, False), ("deferred", 4096, 8192, 8192, False), ("bias deferred", 2305, 4096, 8192, False),
    ("", 2304, 4096, 8192, True), ("deferred", 2048, 4096, 9728, True), ("", 4111, 8192, 8192, True), ("bias", 2048, 8192, 8192, True),
    ("relu", 2048, 8192, 8192, False), ("relu", 1900, 7680, 8192, True), ("", 6144, 8192, 5120, False), ("", 4111, 8192, 5120, True)])
def test_which_products_it_takes(call, m, n, k, takes, monkeypatch):
    ops = gpu_ops()
    x, w, b = operands(m, n, k, 0, 3)
    taken, launch = [], ops._many_launch
    monkeypatch.setattr(ops, "_many_launch", lambda *a, **kw: taken.append(1) or launch(*a, **kw))
    plain = x.double() @ w.double().T
    if call in ("silu", "silu bias", "gelu_tanh"):
        b = b if "bias" in call else None
        y = ops.linear_gated(x, w, b, call) if call == "gelu_tanh" else ops.linear_silu(x, w, b)
        gate, up = (plain if b is None else plain + b.double()).split(n // 2, 1)
        want = activation(call.split()[0])(gate) * up
    elif call == "relu":
        y, want = ops.linear_act(x, w, None, "relu"), torch.relu(plain)
    else:
        y = ops.linear(x, w, b if "bias" in call else None, out_dtype=torch.float32 if call == "bias32" else None, defer="deferred" in call)
        y, want = ops.materialize(y), plain + b.double() if "bias" in call else plain
    assert bool(taken) == takes
    assert off(y, want) < ROUNDED
