"""General attention of many tokens, whose blocks take several query heads of one head of keys: bit for bit what a launch of a
single token, a block a head, gives."""

import pytest
import torch

from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# groups of one, two, three and four heads and more; head sizes of whole fours, of none and of more than a run; pages of few
# keys and of no whole four; contexts at the edges of a chunk of 512 keys
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d,page,longest", [(4, 1, 32, 16, 513), (8, 1, 36, 4, 300), (6, 3, 128, 16, 512), (6, 2, 65, 6, 77),
                                                   (12, 1, 300, 8, 40), (2, 2, 64, 16, 530)])
@pytest.mark.parametrize("extras", [{}, {"softcap": 3.0, "window": 100, "sink": 1, "slopes": 1, "gate": 1, "od": 1}])
def test_rows_are_those_of_single_tokens(dtype, hq, hkv, d, page, longest, extras):
    check_rows(dtype, hq, hkv, d, page, longest, extras, 1024 // hq + 7)             # more than the launches that take a block a head


def check_rows(dtype, hq, hkv, d, page, longest, extras, tokens):
    from atom_amd.kernels.hip import AttentionMeta

    ops = gpu_ops()
    ops.use_mfma_attention = False
    try:
        g = torch.Generator(device=DEV).manual_seed(3)
        lens = [longest, 1, longest // 2]
        blocks = -(-longest // page)
        pages = torch.randperm(3 * blocks, generator=torch.Generator().manual_seed(1)).to(torch.int32).view(3, blocks).to(DEV)
        k = torch.randn(3 * blocks, hkv, page, d, generator=g, device=DEV).to(dtype)
        v = torch.randn(3 * blocks, hkv, d, page, generator=g, device=DEV).to(dtype)
        q = torch.randn(tokens, hq, d, generator=g, device=DEV).to(dtype)
        seq = torch.arange(tokens, dtype=torch.int32, device=DEV) % 4 - 1        # every fourth a padding row
        pos = torch.tensor([(lens[s] - 1 - t // 4 % lens[s]) if s >= 0 else 0 for t, s in enumerate(seq.tolist())],
                           dtype=torch.int32, device=DEV)
        od = d - 3 if extras.get("od") else d
        opts = {"softcap": extras.get("softcap"), "window": extras.get("window")}
        if extras.get("sink"):
            opts["sink"], opts["slopes"] = torch.randn(hq, generator=g, device=DEV), torch.rand(hq, generator=g, device=DEV)
        gates = torch.randn(tokens, hq + 1, generator=g, device=DEV)

        def run(rows):
            n = len(rows)
            meta = AttentionMeta(token_seq=seq[rows].contiguous(), positions=pos[rows].contiguous(), block_tables=pages,
                                 cu_seqlens_q=torch.arange(n + 1, dtype=torch.int32, device=DEV), context_lens=None, num_seqs=3,
                                 num_tokens=n, max_q_len=n, max_context_len=longest, page_size=page)
            out = torch.full((n, hq, od), 7.0, device=DEV, dtype=dtype)
            if extras.get("gate"):
                opts["gate"], opts["gate_off"] = gates[rows].contiguous(), 1
            return ops.paged_attention(q[rows].contiguous(), k, v, out, meta, d ** -0.5, **opts)

        many = run(list(range(tokens)))
        assert bool(many.isfinite().all()) and bool((many[::4] == 0).all())
        for t in (1, 2, 3, tokens // 2, tokens - 3, tokens - 2, tokens - 1):
            assert torch.equal(run([t])[0], many[t])
    finally:
        ops.use_mfma_attention = True


# 600 blocks of four heads and a few more (fewer take two heads each), groups of four and eight
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d,page,longest", [(4, 1, 32, 16, 513), (8, 1, 36, 4, 300), (12, 3, 128, 16, 512), (24, 1, 65, 6, 77)])
@pytest.mark.parametrize("extras", [{}, {"softcap": 3.0, "window": 100, "sink": 1, "slopes": 1, "gate": 1, "od": 1}])
def test_rows_of_four_heads_a_block(dtype, hq, hkv, d, page, longest, extras):
    check_rows(dtype, hq, hkv, d, page, longest, extras, 2400 // hq + 7)


def test_heads_a_block():
    heads = gpu_ops().lib.atom_paged_attention_generic_heads
    assert heads(32, 32, 8) == 0                                                     # a block a head, 512 threads
    assert heads(33, 32, 8) == heads(74, 32, 8) == heads(2000, 6, 3) == 2            # few blocks of four; a group of two
    assert heads(75, 32, 8) == heads(461, 32, 8) == heads(38, 64, 8) == 4
    assert heads(33, 32, 32) == heads(500, 6, 2) == 1
