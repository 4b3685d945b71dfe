"""Attention of prompt portions and single tokens in one launch."""

import pytest
import torch

from test_kernels_gpu import DEV, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [0, 100])
@pytest.mark.parametrize("tile,ksplit,waves,splits", [(64, 2, 4, 1), (64, 2, 4, 8), (64, 2, 8, 1), (64, 4, 4, 1), (64, 4, 4, 4), (64, 4, 8, 1), (64, 4, 8, 16), (128, 1, 4, 1), (128, 1, 4, 2)])
@pytest.mark.parametrize("H,Hkv,page,portions,singles", [
    (3, 3, 16, [(0, 9)], [0]),                                       # the least: one tile, one token at its first position
    (4, 2, 8, [(5, 64), (0, 65)], [31, 32, 700]),                    # shared keys, tiles' edges, pages of 8
    (5, 5, 64, [(300, 129), (63, 200)], [1, 63, 64, 255, 256, 257, 1010] * 3),
    (25, 25, 256, [(0, 1000)], [1500] * 2)])
def test_both_as_their_own_kernels_leave_them(ops, H, Hkv, page, portions, singles, tile, ksplit, waves, splits, window):  # noqa: F811
    """The bits of attention_prefill and attention_decode, row for row; nothing outside their rows is written."""
    hd, reqs = 64, portions + [(pos, 1) for pos in singles]
    blocks = -(-max(p + n for p, n in reqs) // page)
    pages = blocks * len(reqs) + 3
    tables = torch.randperm(pages)[:blocks * len(reqs)].reshape(len(reqs), blocks).to(torch.int32).to(DEV)
    kc, vc = (rnd(pages, Hkv, page, hd, seed=s, dtype=torch.bfloat16) for s in (1, 2))
    rows = sum(n for _, n in reqs)
    q = rnd(rows, H * hd, seed=3, dtype=torch.bfloat16)
    seq = torch.tensor([r for r, (_, n) in enumerate(reqs) for _ in range(n)], dtype=torch.int32, device=DEV)
    pos = torch.tensor([p + i for p, n in reqs for i in range(n)], dtype=torch.int32, device=DEV)
    work, row0 = [], 0
    for r, (p, n) in enumerate(portions):
        work += [[r, row0 + i, p + i, min(tile, n - i)] for i in range(0, n, tile)]
        row0 += n
    n_tiles = len(work)
    work = torch.tensor(work, dtype=torch.int32, device=DEV).reshape(-1)
    single = torch.arange(row0, rows, dtype=torch.int32, device=DEV)
    cut = dict(n_splits=splits, partials=torch.full((len(singles) * H * splits * (hd + 4),), float("nan"), device=DEV)) if splits > 1 else {}
    want, got = (torch.full((rows, H * hd), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.attention_prefill(want, q, kc, vc, tables, work, n_tiles, n_head=H, scale=0.125, window=window, tile=tile, ksplit=ksplit)
    ops.attention_decode(want, q, kc, vc, tables, seq, pos, n_head=H, scale=0.125, window=window, waves=waves, tok_list=single, n_tokens=len(singles), **cut)
    ops.attention_mixed(got, q, kc, vc, tables, work, n_tiles, single, len(singles), seq, pos, n_head=H, scale=0.125, window=window, tile=tile, ksplit=ksplit, waves=waves, **cut)
    assert torch.equal(got, want)
    got.fill_(7.0)
    # (one token of them, the other rows untouched)
    ops.attention_mixed(got, q, kc, vc, tables, work, n_tiles, single[-1:], 1, seq, pos, n_head=H, scale=0.125, window=window, tile=tile, ksplit=ksplit, waves=waves, **cut)
    want[row0:-1] = 7.0
    assert torch.equal(got, want)


def test_what_is_refused(ops):  # noqa: F811
    t = torch.zeros(4, dtype=torch.int32, device=DEV)
    bt = torch.zeros(1, 4, dtype=torch.int32, device=DEV)
    for hd, page, tile, ksplit, waves in ((64, 12, 64, 4, 8), (64, 4, 64, 4, 8), (64, 16, 128, 2, 8), (64, 16, 64, 1, 4), (128, 16, 64, 2, 4), (64, 16, 128, 1, 8), (64, 16, 64, 4, 16)):
        c = torch.zeros(2, 1, page, hd, dtype=torch.bfloat16, device=DEV)
        x = torch.zeros(4, hd, dtype=torch.bfloat16, device=DEV)
        with pytest.raises(Exception, match="attention_mixed"):
            ops.attention_mixed(x, x.clone(), c, c, bt, t, 1, t, 1, t, t, n_head=1, scale=1.0, tile=tile, ksplit=ksplit, waves=waves)
        assert not ops.mixed_pays(torch.bfloat16, hd, page, tile, ksplit, waves)
    assert all(ops.mixed_pays(torch.bfloat16, 64, 8, *form) for form in ((64, 2, 4), (64, 2, 8), (64, 4, 4), (64, 4, 8), (128, 1, 4))) and not ops.mixed_pays(torch.float32, 64, 16, 64, 4, 8)
    c = torch.zeros(2, 1, 16, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(Exception, match="partials"):
        ops.attention_mixed(c[0, 0, :4].contiguous(), c[1, 0, :4].contiguous(), c, c, bt, t, 1, t, 1, t, t, n_head=1, scale=1.0, n_splits=4)
