"""Kernels of small steps at the edges of the sizes where one variant gives way to another: layer norms whose row stays in
registers, gates folded into a product, keys written a group of four entries at a time, heads rotated by a wave each,
attention with the heads together in blocks of many and of few threads."""

import pytest
import torch

import plain_ralitar as pr
from helpers import gpu_ops
from test_gpu_lotorax import test_layernorm_modes as layernorm_modes
from test_gpu_savidra import test_attention_against_plain as attention_against_plain
from test_gpu_savidra import test_norm_rotation_blend_and_page_write as rotation_and_page_write

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [4, 1020, 1024, 1028, 2048, 4092, 8192, 8196])
def test_layernorm_groups_a_thread(dtype, width):
    layernorm_modes(dtype, width, 6)


@pytest.mark.parametrize("activation", ["silu", "relu", "gelu_tanh"])
@pytest.mark.parametrize("m,inter,k,biased", [(1, 24, 64, False), (3, 13, 136, True), (8, 520, 1032, True)])
def test_gate_in_the_product(activation, m, inter, k, biased):
    """A gate|up product of few rows that waits for its gate: the same as in float64 within one rounding of the result
    and the float32 sums."""
    ops = gpu_ops()
    x, w = rnd((m, k), 1).to(torch.bfloat16), rnd((2 * inter, k), 2, 0.1).to(torch.bfloat16)
    b = rnd((2 * inter,), 3) if biased else None
    both = ops.linear(x.to(DEV), w.to(DEV), b.to(DEV) if biased else None, defer=True, slices=False)
    out = torch.empty((m, inter), dtype=torch.bfloat16, device=DEV)
    ops.gated_act(both, out, activation)
    g, u = (x.double() @ w.double().T + (b.double() if biased else 0)).chunk(2, -1)
    act = {"silu": torch.nn.functional.silu, "relu": torch.relu,
           "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh")}[activation]
    want = act(g) * u
    assert bool(((out.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5 * float(want.abs().max())).all())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,inter", [(1, 8), (3, 264), (2, 12)])
def test_gated_act_groups(dtype, rows, inter):
    ops = gpu_ops()
    x = rnd((rows, 2 * inter), 4, 2.0).to(dtype)
    out = torch.empty((rows, inter), dtype=dtype, device=DEV)
    ops.gated_act(x.to(DEV), out, "relu")
    g, u = x.chunk(2, -1)
    assert torch.equal(out.cpu(), (torch.relu(g.float()) * u.float()).to(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,D,dims,normed", [(4, 2, 64, 32, True), (28, 4, 128, 128, True), (3, 1, 8, 4, False),
                                               (6, 2, 12, 0, True), (2, 1, 12, 6, True)])
def test_keys_as_values_in_groups_of_four(dtype, H, G, D, dims, normed):
    """(28 + 4) x 128 entries are the most a block holds in registers; 6 rotated entries take the general kernel."""
    ops = gpu_ops()
    T, page, eps = 5, 4, 1e-5
    proj = rnd((T, (H + G) * D + 4), 1, 2.0)
    positions, slots = torch.tensor([0, 1, 700, 40000, 5]), [3, 8, -1, 0, 11]
    qw, kw = (1 + rnd((H * D,), 2, 0.2), 1 + rnd((G * D,), 3, 0.2)) if normed else (None, None)
    freq = torch.tensor([300.0 ** (-2.0 * i / max(dims, 1)) for i in range(dims // 2)], dtype=torch.float64)
    k_cache = torch.zeros((3, G, page, D), dtype=dtype, device=DEV)
    v_cache = torch.zeros((3, G, D, page), dtype=dtype, device=DEV)
    q = torch.empty((T, H, D), dtype=dtype, device=DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    ops.keys_as_values_write(proj.to(DEV), q, k_cache, v_cache, qw.to(DEV) if normed else None, kw.to(DEV) if normed else None,
                             freq.to(DEV) if dims else None, dims, i32(positions.tolist()), i32(slots), H, G, D, page, eps)
    p = proj.double()
    qn, kn, raw = p[:, :H * D], p[:, H * D:(H + G) * D], p[:, H * D:(H + G) * D].view(T, G, D)
    if normed:
        qn, kn = pr.rms(qn, eps) * qw.double(), pr.rms(kn, eps) * kw.double()
    qn, kn = qn.view(T, H, D), kn.view(T, G, D)
    if dims:
        qn, kn = pr.rotate_pairs(qn, positions, freq), pr.rotate_pairs(kn, positions, freq)
    tol = {torch.float32: 2e-5, torch.bfloat16: 2.0 ** -8}[dtype]
    near = lambda got, want: bool(((got.double().cpu() - want).abs() <= tol * float(want.abs().max())).all())  # noqa: E731
    assert near(q, qn)
    for t, slot in enumerate(slots):
        if slot >= 0:
            pg, off = divmod(slot, page)
            assert near(k_cache[pg, :, off, :], kn[t]) and near(v_cache[pg, :, :, off], raw[t])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,D,DV,rot", [(2, 1, 320, 70, 320), (3, 1, 200, 64, 6), (1, 1, 130, 130, 128)])
def test_rotated_heads_wider_than_a_wave(dtype, H, G, D, DV, rot):
    rotation_and_page_write(dtype, H, G, D, DV, rot, 16, True, "blend")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("how", ["blocks", "parts"])
@pytest.mark.parametrize("H,G,D,DV,page,talk", [(16, 4, 64, 128, 16, True), (24, 2, 32, 128, 8, True), (6, 2, 16, 10, 24, False)])
def test_heads_together_by_pairs_a_thread(dtype, how, H, G, D, DV, page, talk):
    attention_against_plain(dtype, how, H, G, D, DV, page, 150, True, talk, True)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("how", ["blocks", "parts"])
@pytest.mark.parametrize("H,G,D,DV,page,talk", [(8, 2, 32, 64, 16, False), (4, 2, 32, 64, 6, True), (8, 2, 32, 66, 8, False),
                                                (10, 2, 16, 48, 16, False)])
def test_heads_together_by_threads_a_block(dtype, how, H, G, D, DV, page, talk):
    """Blocks of few threads up to 256 pairs and scores, of many from there on."""
    attention_against_plain(dtype, how, H, G, D, DV, page, 150, True, talk, True)


@pytest.mark.parametrize("wdtype", DTYPES)
@pytest.mark.parametrize("m,inter,k,biased", [(1, 13, 96, True), (5, 3080, 96, False), (5, 3081, 64, True), (17, 1, 20, True),
                                              (33, 160, 96, False), (65, 1003, 144, True), (130, 4100, 64, False),
                                              (200, 9000, 160, True), (300, 12300, 64, False)])
def test_float32_gate_in_the_product(m, inter, k, biased, wdtype):
    """The float32 product that gates where it writes: the bits of the plain product and SiLU-mul behind it, in the tiles of
    every height and width (the last two rows: through LDS with float32 weights)."""
    ops = gpu_ops()
    x, w = rnd((m, k), 5).to(DEV), rnd((2 * inter, k), 6, 0.2).to(DEV).to(wdtype)
    b = rnd((2 * inter,), 7).to(DEV) if biased else None
    act = ops.linear_silu(x, w, b)
    want = torch.empty_like(act)
    ops.silu_mul(ops.linear(x, w, b), want)
    assert act.shape == (m, inter) and act.dtype == torch.float32
    assert torch.equal(act, want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [53, 1024, 2050, 4096])
@pytest.mark.parametrize("init", [True, False])
def test_stream_norm_rows_do_not_depend_on_batch(dtype, width, init):
    """A row alone, among a few and among more than there are compute units: the same bits."""
    ops = gpu_ops()
    stream, x, w = rnd((600, width), 1).to(DEV), rnd((600, width), 2).to(DEV), (1 + rnd((width,), 3, 0.2)).to(DEV)
    got = []
    for rows in (slice(0, 600), slice(7, 12), slice(9, 10)):
        s, out = stream[rows].clone(), torch.empty((len(stream[rows]), width), dtype=dtype, device=DEV)
        ops.stream_norm(s, x[rows].contiguous(), w, 2e-5, out, init=init)
        got.append((s, out))
    for mine, few, alone in zip(*got):
        assert torch.equal(mine[7:12], few) and torch.equal(mine[9:10], alone)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [512, 1300])
@pytest.mark.parametrize("lens", [[1, 2, 1], [1020, 1, 2], [1021, 1, 2], [700, 800]])
def test_shifted_rows_in_pieces_and_whole(dtype, width, lens):
    """Rows cut over several blocks, and from four tokens a compute unit on whole: each mixed with the one before it, the
    first of a request with what its slot holds, which then holds the last."""
    ops = gpu_ops()
    T, S = sum(lens), len(lens)
    x, mu, kept = rnd((T, width), 1).to(dtype), torch.rand((width,), generator=torch.Generator().manual_seed(2)), rnd((S, 3 + width), 3)
    cu = [sum(lens[:i]) for i in range(S + 1)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    state, out = kept.to(DEV), torch.empty((T, width), dtype=dtype, device=DEV)
    ops.shift_rows(x.to(DEV), mu.to(DEV), out, state, 3, i32(cu), i32(list(range(S))), i32([s for s in range(S) for _ in range(lens[s])]))
    cur = x.double()
    prev = torch.cat((cur[:1], cur[:-1]))
    for s in range(S):
        prev[cu[s]] = kept[s, 3:].double()
    want = cur + (prev - cur) * mu.double()
    tol = {torch.float32: 1e-6, torch.bfloat16: 2.0 ** -8}[dtype]
    assert bool(((out.double().cpu() - want).abs() <= tol * (want.abs() + 1)).all())
    assert torch.equal(state.cpu()[:, 3:], x.float()[[c - 1 for c in cu[1:]]]) and torch.equal(state.cpu()[:, :3], kept[:, :3])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,D,DV", [(5, 2, 72, 40), (1, 1, 16, 20), (16, 4, 128, 128)])
def test_plain_heads_of_few_and_many_tokens(dtype, H, G, D, DV):
    """A wave a head up to four tokens a compute unit, a block a token from there on: the same bits, and every head there."""
    ops = gpu_ops()
    T, page, DP = 1100, 16, max(D, DV)
    proj = rnd((T, (H + G) * D + G * DV), 1).to(DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    slots = torch.randperm(T, generator=torch.Generator().manual_seed(2)).tolist()
    slots[7] = -1
    got = []
    for n in (T, 1023, 9):
        q = torch.full((n, H, DP), float("nan"), dtype=dtype, device=DEV)
        k_cache = torch.zeros((T // page + 1, G, page, DP), dtype=dtype, device=DEV)
        v_cache = torch.zeros((T // page + 1, G, DP, page), dtype=dtype, device=DEV)
        ops.qkv_plain_write(proj[:n].contiguous(), q, k_cache, v_cache, i32(list(range(n))), i32(slots[:n]), H, G, D, DV, page,
                            True, 1e-5, (0.1, 64))
        at = [slots[t] for t in range(9) if slots[t] >= 0]
        pg, off = torch.tensor(at, device=DEV) // page, torch.tensor(at, device=DEV) % page
        got.append((q[:9], k_cache[pg, :, off], v_cache[pg, :, :, off]))
    for few in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], few))
    x = proj[:9].double()
    k = x[:, H * D:(H + G) * D].view(9, G, D)
    k = k / torch.sqrt((k * k).mean(-1, keepdim=True) + 1e-5)
    keep = [t for t in range(9) if slots[t] >= 0]
    for mine, want in ((got[0][1][:, :, :D], k[keep]), (got[0][2][:, :, :DV], x[keep, (H + G) * D:].view(-1, G, DV))):
        assert bool(((mine.double() - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 1e-5) * want.abs().max()).all())
