"""Prompt portions' attention in 32 bits, 32 queries to 256 keys: the bits of the kernel that takes each token on its own."""

import pytest
import torch

from test_kernels_gpu import DEV, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [32, 64, 128])
@pytest.mark.parametrize("H,Hkv,page,requests", [
    (3, 3, 16, [(0, 1)]), (2, 2, 4, [(0, 9), (31, 33)]), (4, 2, 24, [(0, 300), (5, 64)]), (3, 3, 64, [(255, 1), (256, 1), (250, 140), (700, 40)]), (12, 12, 16, [(0, 511), (0, 100), (3, 237)]),
])
def test_rows_have_the_bits_of_tokens_on_their_own(ops, H, Hkv, page, requests, tile):  # noqa: F811
    """requests: (cached, new) tokens: from one key to four splits, queries with none of a split's keys beside others with some, tiles' remainders of 1 to 33, pages that no
    load of four keys divides. A value that is no number, behind a token, changes nothing for the tokens ahead of it."""
    n, hd = sum(new for _, new in requests), 64
    blocks = max(-(-(past + new) // page) for past, new in requests) + 1
    pages = blocks * len(requests) + 2
    kc, vc = rnd(pages, Hkv, page, hd, seed=1), rnd(pages, Hkv, page, hd, seed=2)
    bt = torch.randperm(pages)[:blocks * len(requests)].reshape(len(requests), blocks).to(torch.int32).to(DEV)
    past, new = requests[-1]
    last = past + new - 1
    vc[bt[-1, last // page].item(), :, last % page, 5] = float("inf")
    q = rnd(n, H * hd, seed=3, scale=3.0)
    seq = torch.cat([torch.full((new,), r) for r, (_, new) in enumerate(requests)]).to(torch.int32).to(DEV)
    pos = torch.cat([torch.arange(past, past + new) for past, new in requests]).to(torch.int32).to(DEV)
    work, row = [], 0
    for r, (past, new) in enumerate(requests):
        for t0 in range(0, new, tile):
            work += [r, row + t0, past + t0, min(tile, new - t0)]
        row += new
    splits = -(-max(past + new for past, new in requests) // 256)
    want, got = torch.zeros(n, H * hd, device=DEV), torch.full((n, H * hd), float("nan"), device=DEV)
    partials = torch.empty(n, H, splits, hd + 4, device=DEV)
    common = dict(n_head=H, scale=0.125)
    ops.attention_decode(want, q, kc, vc, bt, seq, pos, n_splits=splits, partials=partials if splits > 1 else None, waves=4, chunk=256, **common)
    left = torch.full_like(partials, float("nan"))
    ops.attention_rows(got, q, kc, vc, bt, torch.tensor(work, dtype=torch.int32, device=DEV), len(work) // 4, tile=tile, n_splits=splits, partials=left, **common)
    if splits > 1:
        ops.attention_merge(got, left)
        assert torch.equal(left[..., :hd + 2].nan_to_num(7.0), partials[..., :hd + 2].nan_to_num(7.0))
    assert torch.equal(got[:-1], want[:-1]) and torch.isfinite(got[:-1]).all()
    assert torch.equal(got[-1].nan_to_num(7.0), want[-1].nan_to_num(7.0))
