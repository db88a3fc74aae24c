"""Kernels that take a decode step's single tokens through several operations in one launch, against the operations one by
one in float64."""

import pytest
import torch

from helpers import gpu_ops
from plain_kernels import PlainKernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PLAIN = PlainKernels()


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


def i32(values):
    return torch.tensor(values, dtype=torch.int32)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("per_channel,a_rank,g_rank,act", [(False, 0, 0, "silu"), (True, 64, 64, "sigmoid"), (True, 0, 16, "silu"),
                                                           (False, 48, 0, "sigmoid"), (True, 16, 0, "silu")])
@pytest.mark.parametrize("heads,kv_heads,dim", [(2, 2, 64), (6, 3, 64), (3, 3, 128), (4, 2, 128)])
def test_delta_step(heads, kv_heads, dim, per_channel, a_rank, g_rank, act, dtype):
    """Requests with and without a token, one that is padding; states beside theirs stay as they are."""
    ops = gpu_ops()
    lens, slots = [1, 1, 0, 1, 1], [4, 0, 2, -1, 1]
    T, C, decays = sum(lens), (2 * kv_heads + heads) * dim, heads * (dim if per_channel else 1)
    widths = [C, heads, a_rank or decays, g_rank or heads * dim]
    b_off, a_off, g_off = C, C + heads, C + heads + widths[2]
    proj = rnd((T, sum(widths) + 3), 1)
    taps = rnd((C, 4), 2, 0.5).to(dtype)
    decay2 = rnd((decays, a_rank), 3, 0.2).to(dtype) if a_rank else None
    gate2 = rnd((heads * dim, g_rank), 4, 0.2).to(dtype) if g_rank else None
    a_log, dt_bias, norm = rnd((heads,), 5, 0.5), rnd((decays,), 6) - 1, 1 + rnd((dim,), 7, 0.2)
    off = 3 * C + 4
    state = rnd((5, off + heads * dim * dim), 8, 0.3)
    cu = i32([0, 1, 2, 2, 3, 4])

    want_state, some, places = state.double(), i32([0, 1, 2, 3, 4]), i32([s for n, s in zip(lens, slots) if n])
    qkv = torch.empty((T, C), dtype=torch.float64)
    PLAIN.conv_silu_state(proj, C, taps, want_state, some, places, qkv)
    decay, d_off = (proj, a_off) if decay2 is None else (proj[:, a_off:a_off + a_rank].double() @ decay2.double().T, 0)
    gate, gate_off = (proj, g_off) if gate2 is None else (proj[:, g_off:g_off + g_rank].double() @ gate2.double().T, 0)
    read = torch.empty((T, heads, dim), dtype=torch.float64)
    PLAIN.delta_rule(qkv, proj, d_off, b_off, a_log, dt_bias, want_state, off, some, places, read, heads, kv_heads, dim, dim,
                     decay=decay, per_channel=per_channel)
    want = torch.empty((T, heads * dim), dtype=torch.float64)
    PLAIN.delta_out(read, gate, gate_off, norm, 1e-5, want, activation=act)

    dev = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    got, out = dev(state), torch.full((T, heads * dim), 7.0, dtype=dtype, device=DEV)
    assert ops.delta_step(dev(proj), dev(taps), got, off, dev(cu), dev(i32(slots)), b_off, a_off, dev(decay2), g_off, dev(gate2),
                          dev(a_log), dev(dt_bias), dev(norm), 1e-5, out, heads, kv_heads, dim, dim, per_channel, act) is out
    # sums of up to 128 float32 terms; the output is rounded to its type
    assert float((got.cpu().double() - want_state).norm() / want_state.norm()) <= 2e-6
    assert float((out.cpu().double() - want).norm() / want.norm()) <= (4e-3 if dtype == torch.bfloat16 else 4e-6)
    assert float(out[2].abs().max()) == 0
    assert torch.equal(got[2:4].cpu(), state[2:4]), "slots 2 (no token) and 3 (no request) are not touched"


def test_delta_step_leaves_other_sizes_alone():
    ops = gpu_ops()
    for sizes in ((4, 2, 32, 32, 4, 0, 0), (4, 2, 64, 128, 4, 0, 0), (6, 2, 64, 64, 4, 0, 0), (4, 2, 64, 64, 3, 0, 0),
                  (4, 2, 64, 64, 4, 24, 0), (4, 2, 64, 64, 4, 0, 80)):
        assert not ops.lib.atom_delta_step_supports(*sizes)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("blocks,part,lens,slots", [(3, 64, [1], [2]), (2, 128, [1, 0, 1, 1], [1, 2, -1, 0]),
                                                    (1, 256, [1] * 8, [7, 6, 5, 4, 3, 2, 1, 0]), (2, 512, [1, 1, 1], [0, -1, 3])])
def test_rglru_step(blocks, part, lens, slots, dtype):
    ops = gpu_ops()
    C, T = blocks * part, sum(lens)
    proj = rnd((T, 2 * C + 5), 1)
    taps, conv_bias = rnd((C, 4), 2, 0.5).to(dtype), rnd((C,), 3, 0.3)
    ra, ri = (rnd((blocks, part, part), s, part ** -0.5).to(dtype) for s in (4, 5))
    br, bi, lam = rnd((blocks, part), 6), rnd((blocks, part), 7), rnd((C,), 8) - 2
    off = 3 * C + 1
    state = rnd((8, off + C), 9, 0.5)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    some, places = i32(sorted(set(cu))), i32([s for n, s in zip(lens, slots) if n])

    want_state = state.double()
    u = torch.empty((T, C), dtype=torch.float64)
    PLAIN.conv_silu_state(proj, C, taps, want_state, some, places, u, bias=conv_bias, activation="none")
    parts = u.view(T, blocks, part).transpose(0, 1)
    gates = torch.stack([torch.matmul(parts, w.double().transpose(1, 2)).transpose(0, 1).reshape(T, C) for w in (ra, ri)])
    want = torch.empty((T, C), dtype=torch.float64)
    PLAIN.rglru_scan(u, gates, br, bi, lam, proj, C + 5, want_state, off, some, places, want, 8.0)

    dev = lambda t: t.to(DEV)  # noqa: E731
    got, out = dev(state), torch.full((T, C), 7.0, dtype=dtype, device=DEV)
    assert ops.rglru_step(dev(proj), C + 5, dev(taps), dev(conv_bias), got, off, dev(i32(cu)), dev(i32(slots)), dev(ra), dev(ri),
                          dev(br), dev(bi), dev(lam), out, 8.0) is out
    assert float((got.cpu().double() - want_state).norm() / want_state.norm()) <= 2e-6
    assert float((out.cpu().double() - want).norm() / want.norm()) <= (4e-3 if dtype == torch.bfloat16 else 4e-6)


@pytest.mark.parametrize("m,n,k", [(1, 256, 2048), (3, 37, 136), (8, 64, 512)])
def test_product_times_rows_of_a_table(m, n, k):
    ops = gpu_ops()
    x, w, table = rnd((m, k), 1).bfloat16(), rnd((n, k), 2, k ** -0.5).bfloat16(), rnd((50, 3 * n), 3).bfloat16()
    ids = i32([49, 0, -1, 7, 50, 3, 3, 1][:m])
    got = ops.linear_token_gate(x.to(DEV), w.to(DEV), table.to(DEV), n, ids.to(DEV))
    factor = torch.where(((ids >= 0) & (ids < 50))[:, None], table[ids.clamp(0, 49).long(), n:2 * n].double(), 0.0)
    want = torch.nn.functional.gelu(x.double() @ w.double().T, approximate="tanh") * factor
    assert float((got.cpu().double() - want).norm() / want.norm()) <= 4e-3


STEPS = [([1], [2]), ([1, 0, 1, 1], [1, 2, -1, 0])]


def places_of(lens, slots):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return cu, i32(sorted(set(cu))), i32([s for n, s in zip(lens, slots) if n])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,slots", STEPS)
@pytest.mark.parametrize("heads,groups,dim", [(4, 1, 64), (6, 2, 128), (70, 1, 128)])
def test_space_step(heads, groups, dim, lens, slots, dtype):
    ops = gpu_ops()
    V, T = 64, sum(lens)
    inner = heads * V
    C = inner + 2 * groups * dim
    proj = rnd((T, inner + C + (heads + 3) // 4 * 4), 1)
    taps, conv_bias = rnd((C, 4), 2, 0.5).to(dtype), rnd((C,), 3, 0.3)
    step_bias, a_log, skip, norm = rnd((heads,), 4) - 1, rnd((heads,), 5, 0.5), rnd((heads,), 6), 1 + rnd((inner,), 7, 0.2)
    off = 3 * C + 4
    state = rnd((4, off + inner * dim), 8, 0.3)
    cu, some, places = places_of(lens, slots)

    want_state = state.double()
    xbc, y, want = (torch.empty((T, n), dtype=torch.float64) for n in (C, inner, inner))
    PLAIN.conv_silu_state(proj, C, taps, want_state, some, places, xbc, bias=conv_bias, x_offset=inner)
    PLAIN.linear_scan(xbc, inner + groups * dim, groups, xbc, inner, groups, xbc, 0, proj, inner + C, want_state, off, some,
                      places, y, heads, dim, V, per_channel=False, skip=skip, step_bias=step_bias, a_log=a_log)
    PLAIN.group_norm_gate(y, 1, norm, 1e-5, want, gate=proj, gate_off=0, gate_first=True)

    dev = lambda t: t.to(DEV)  # noqa: E731
    got, out = dev(state), torch.full((T, inner), 7.0, dtype=dtype, device=DEV)
    assert ops.space_step(dev(proj), inner, dev(taps), dev(conv_bias), got, off, dev(i32(cu)), dev(i32(slots)), dev(step_bias),
                          dev(a_log), dev(skip), dev(norm), 1e-5, out, heads, groups, dim, V, 1) is out
    assert float((got.cpu().double() - want_state).norm() / want_state.norm()) <= 2e-6
    assert float((out.cpu().double() - want).norm() / want.norm()) <= (4e-3 if dtype == torch.bfloat16 else 4e-6)
    assert torch.equal(got[3].cpu(), state[3])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,slots", STEPS)
@pytest.mark.parametrize("heads,rank", [(1, 32), (5, 64), (3, 96), (32, 128)])
def test_mix_step(heads, rank, lens, slots, dtype):
    ops = gpu_ops()
    T, c = sum(lens), heads * 64
    r, k, v, g = (rnd((T, c), s) for s in (1, 2, 3, 4))
    squashed, decay2 = torch.tanh(rnd((T, rank), 5)), rnd((c, rank), 6, 0.2).to(dtype)
    bias, bonus, norm = rnd((c,), 7) - 2, rnd((heads, 64), 8, 0.3), 1 + rnd((c,), 9, 0.2)
    state = rnd((4, 8 + c * 64), 10, 0.3)
    cu, some, places = places_of(lens, slots)

    want_state = state.double()
    y, want = (torch.empty((T, c), dtype=torch.float64) for _ in range(2))
    PLAIN.linear_scan(r, 0, heads, k, 0, heads, v, 0, squashed.double() @ decay2.double().T, 0, want_state, 8, some, places, y,
                      heads, 64, 64, w_bias=bias, bonus=bonus)
    PLAIN.group_norm_gate(y, heads, norm, 1e-5, want, gate=g)

    dev = lambda t: t.to(DEV)  # noqa: E731
    got, out = dev(state), torch.full((T, c), 7.0, dtype=dtype, device=DEV)
    assert ops.mix_step(dev(r), dev(k), dev(v), dev(g), dev(squashed), dev(decay2), dev(bias), dev(bonus), dev(norm), got, 8,
                        dev(i32(cu)), dev(i32(slots)), out, heads, 64, 1e-5) is out
    assert float((got.cpu().double() - want_state).norm() / want_state.norm()) <= 2e-6
    assert float((out.cpu().double() - want).norm() / want.norm()) <= (4e-3 if dtype == torch.bfloat16 else 4e-6)
    assert torch.equal(got[3].cpu(), state[3])


@pytest.mark.parametrize("which", ["embedding", "embedding_scaled", "embedding_positions"])
def test_embeddings_of_tokens_still_on_the_device(which):
    """As after ``feed_tokens``, which it takes the place of: the rows, and the ids left for the kernels behind it.  Several
    blocks a row; sources that name no sampled row leave the id."""
    ops = gpu_ops()
    table, rows = rnd((40, 2500), 1).bfloat16().to(DEV), rnd((9, 2500), 2).bfloat16().to(DEV)
    ids, source, sampled = (i32(v).to(DEV) for v in ([7, 0, 39, 3, 1], [2, -1, 0, 3, 1], [11, 12, 13]))
    rest = {"embedding": (), "embedding_scaled": (2.5,), "embedding_positions": ()}[which]

    def run(ids, **kw):
        out = torch.empty((5, 2500), dtype=torch.float32, device=DEV)
        if which == "embedding_positions":
            return ops.embedding_positions(table, rows, ids, i32([0, 8, 3, 1, 2]).to(DEV), out, **kw)
        return getattr(ops, which)(table, ids, out, *rest, **kw)

    fed = ops.feed_tokens(ids.clone(), source, sampled)
    assert fed.tolist() == [13, 0, 11, 3, 12]
    assert torch.equal(run(ids, feed=(source, sampled)), run(fed)) and torch.equal(ids, fed)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,terms", [(4, 1), (1020, 2), (2048, 2), (4100, 1), (8192, 4)])
def test_sum_norm_shift(width, terms, dtype):
    """The bits of ``sum_norm`` and ``shift_rows`` in turn: rows with a slot, padding rows, a request that sits out."""
    ops = gpu_ops()
    dev = lambda t: t.to(DEV)  # noqa: E731
    stream, weight, mu = dev(rnd((4, width), 1)), dev(1 + rnd((width,), 2, 0.2)), dev(rnd((width,), 3, 0.5))
    ys = [dev(rnd((4, width), 4 + i).to(torch.bfloat16 if i % 2 else torch.float32)) for i in range(terms)]
    scales, state = [0.5 + i for i in range(terms)], dev(rnd((5, 8 + width), 9))
    cu, slots, seqs = dev(i32([0, 1, 2, 2, 3, 4])), dev(i32([3, 0, 1, -1, 4])), dev(i32([0, 1, -1, 4]))

    want_stream, want_state, want = stream.clone(), state.clone(), torch.empty((4, width), dtype=dtype, device=DEV)
    ops.sum_norm(want_stream, 1.5, ys, scales, weight, 1e-5)
    ops.shift_rows(want_stream, mu, want, want_state, 4, cu, slots, seqs)
    out = torch.empty((4, width), dtype=dtype, device=DEV)
    assert ops.sum_norm_shift(stream, 1.5, ys, scales, weight, 1e-5, mu, out, state, 4, slots, seqs) is out
    assert torch.equal(stream, want_stream) and torch.equal(state, want_state)
    # (a product and a sum may be one rounding in one kernel and two in the other)
    assert float((out.double() - want.double()).abs().max()) <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22) * float(want.abs().max())
    assert ops.sum_norm_shift(stream[:, :3].contiguous(), 1.5, [], [], weight[:3].clone(), 1e-5, mu[:3].clone(), out[:, :3].contiguous(),
                              state, 4, slots, seqs) is None


@pytest.mark.parametrize("tokens,heads,dim,rank,rot,dims", [(1, 16, 128, 512, 64, 64), (20, 3, 64, 40, 16, 8), (95, 2, 8, 128, 64, 0),
                                                            (33, 17, 24, 64, 32, 32)])
def test_latent_absorb(tokens, heads, dim, rank, rot, dims):
    """The bits of ``latent_prepare`` and ``heads_gemm`` in turn, tokens without a slot among them."""
    from atom_amd.kernels.hip import QueryTurn

    ops = gpu_ops()
    kv_off = heads * (dim + rot)
    ld = (kv_off + rank + rot + 7) // 4 * 4
    proj, norm = rnd((tokens, ld), 1).to(DEV), (1 + rnd((rank,), 2, 0.2)).to(DEV)
    weight = rnd((heads, rank, dim), 3, dim ** -0.5).bfloat16().to(DEV)
    turns = ops.rotation_table(torch.arange(tokens, dtype=torch.int32, device=DEV),
                               (0.7 ** torch.arange(dims // 2, dtype=torch.float64)).to(DEV), 1.1) if dims else None
    slots = torch.randperm(tokens + 5, generator=torch.Generator().manual_seed(4))[:tokens].int()
    slots[tokens // 2 + 1:tokens // 2 + 2] = -1
    slots = slots.to(DEV)
    pages = rnd((2, (tokens + 6) // 2, rank + rot), 5).bfloat16().to(DEV)
    want_pages, width = pages.clone(), rank + rot
    want, out = (torch.empty((tokens, heads, width), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.latent_prepare(proj, want_pages, slots, kv_off, rank, rot, norm, 1e-5, turns)
    ops.heads_gemm(proj, 0, ld, dim + rot, weight, want, 0, heads * width, width, heads, tokens, rank, dim, alpha=0.3,
                   turn=QueryTurn(dim, rank, rot, turns, 0.3))
    assert ops.latent_absorb(proj, pages, slots, kv_off, rank, rot, norm, 1e-5, turns, weight, out, heads, dim, 0.3) is out
    assert torch.equal(out, want) and torch.equal(pages, want_pages)
