"""Heads worked through together for few tokens with their keys cut over several blocks, one walk over the keys and the heads mixed
behind the sums, against float64."""

import pytest
import torch

import plain_savidra as ps
from helpers import gpu_ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rnd(shape, seed, scale=1.0):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale


@pytest.mark.parametrize("parts", [2, 3, 9])
@pytest.mark.parametrize("H,G,D,DV,page,talk,sink,window", [
    (8, 2, 128, 128, 16, True, False, None), (16, 4, 64, 256, 8, True, True, None), (16, 1, 32, 16, 4, True, False, 70),
    (5, 5, 96, 80, 16, True, True, None), (6, 3, 64, 192, 32, True, False, None), (32, 2, 256, 48, 8, False, True, 100),
    (4, 4, 32, 1024, 64, False, False, None)])
def test_against_float64(H, G, D, DV, page, talk, sink, window, parts, monkeypatch):
    """Contexts at the edges of chunks of 64 keys and of pages, parts without keys, a padding row; places of a page that hold no
    key of the request hold NaN."""
    ops = gpu_ops()
    ran, kernel = [], ops.lib.atom_attention_together_few
    monkeypatch.setattr(ops.lib, "atom_attention_together_few", lambda *a: ran.append(1) or kernel(*a))
    lens, scale = [1, 63, 64, 65, 130, 257], 0.3
    dt, S = torch.bfloat16, 6
    blocks = -(-max(lens) // page)
    k_cache, v_cache = torch.full((S * blocks, G, page, D), float("nan")), torch.full((S * blocks, G, DV, page), float("nan"))
    tables = torch.randperm(S * blocks, generator=torch.Generator().manual_seed(1)).view(S, blocks).int()
    q = rnd((S + 1, H, D), 2, 128 ** -0.25).to(dt)
    temp, sk = 1 + 0.3 * rnd((H,), 4), 1.5 * rnd((H,), 5)
    tk = torch.eye(H) + 0.3 * rnd((H, H), 6)
    want = torch.zeros((S + 1, H, DV), dtype=torch.float64)
    for s, n in enumerate(lens):
        keys, values = rnd((n, G, D), 10 + s).to(dt), rnd((n, G, DV), 20 + s).to(dt)
        for j in range(n):
            k_cache[tables[s, j // page], :, j % page], v_cache[tables[s, j // page], :, :, j % page] = keys[j].float(), values[j].float()
        from_ = max(0, n - window) if window else 0
        w = ps.softmax_weights(q[s:s + 1].double(), keys[from_:].double(), torch.tensor([n - 1 - from_]), torch.arange(n - from_), scale,
                               sink=sk.double() if sink else None, temp=temp.double())
        if talk:
            w = torch.einsum("hg,gij->hij", tk.double(), w)
        want[s] = ps.apply_weights(w, values[from_:].double(), H).view(H, DV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    out = torch.full((S + 1, H, DV), float("nan"), dtype=dt, device=DEV)
    ops.attention_together(q.to(DEV), k_cache.to(dt).to(DEV), v_cache.to(dt).to(DEV), out, i32([0, 1, 2, 3, 4, 5, -1]),
                           i32([n - 1 for n in lens] + [0]), tables.to(DEV), scale, head_scale=temp.to(DEV),
                           sink=sk.to(DEV) if sink else None, talk=tk.to(DEV) if talk else None, window=window,
                           max_context_len=max(lens), parts=parts)
    assert ran == [1]
    got = out.double().cpu()
    # results rounded to bfloat16 once, float32 sums of up to 257 keys and 16 heads before
    assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 2e-5 * float(want.abs().max())).all())
