"""A small step's choice of experts in one launch: with the router's product, and with groups of experts."""

import pytest
import torch

from test_kernels_gpu import DEV, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


def route(ops, logits, n, E, top, block, router=None, **kw):  # noqa: F811
    rows = top + (1 if kw.get("extra") else 0)
    listed = E - kw.get("identity", 0) + (1 if kw.get("extra") else 0)
    tiles = ops.moe_tiles(n * rows, listed, block)
    ids, places, group = (torch.full((k,), 99, dtype=torch.int32, device=DEV) for k in (n * rows, tiles * block, tiles))
    weights = torch.full((n * rows,), float("nan"), device=DEV)
    ops.moe_route(logits, top, ids, weights, places, group, block=block, router=router, **kw)
    # every entry with an expert stands in one of its expert's tiles, once
    want = sorted((e, i) for i, e in enumerate(ids.tolist()) if e >= 0)
    got = sorted((group[p // block].item(), i) for p, i in enumerate(places.tolist()) if i >= 0)
    assert got == want
    used = [g for g in group.tolist() if g >= 0]
    assert used == sorted(used) and len(used) == sum(-(-sum(e == x for e, _ in want) // block) for x in range(listed)) and all(g == -1 for g in group.tolist()[len(used):])
    return ids, weights


@pytest.mark.parametrize("kw", [{}, dict(scores="logistic", groups=(4, 2)), dict(scores="softmax_all", scale=2.5, identity=2, extra=True), dict(scores="logistic", groups=(1, 1))])
@pytest.mark.parametrize("n,E,K,bias", [(1, 8, 64, False), (4, 8, 768, True), (7, 12, 1600, True), (8, 8, 192, False), (9, 14, 8256, True), (16, 12, 1088, False)])
def test_the_routers_product_inside(ops, n, E, K, bias, kw):  # noqa: F811
    """Logits, choices and weights of the product's own kernel and the choice behind it, bit for bit."""
    top, extra = 2, 1 if kw.get("extra") else 0
    if kw.get("groups", (1, 1))[0] == 4 and E != 8:
        E = 12 if E != 14 else 16  # (groups of three: the general kernel; of four)
    a, w = rnd(n, K, dtype=torch.bfloat16), rnd(E + extra, K, seed=1, scale=0.2, dtype=torch.bfloat16)
    b = rnd(E + extra, seed=2) if bias else None
    more = dict(kw, correction=rnd(E, seed=3, scale=0.1)) if kw else {}
    want = torch.full((n, E + extra), float("nan"), device=DEV)
    ops.gemm_skinny(a, w, b, out=want)
    first = route(ops, want, n, E, top, 16, **more)
    if not ops.router_product_takes(a, w, n, E, top, kw.get("groups"), kw.get("scores", "softmax")):
        assert kw.get("groups", (1, 1))[0] == 4 and E == 12
        return
    got = torch.full_like(want, float("nan"))
    second = route(ops, got, n, E, top, 16, router=(a, w, b), **more)
    assert torch.equal(got, want) and all(torch.equal(x, y) for x, y in zip(first, second))


def group_score(values):
    """The two largest, in the order of the kernel that walks a group."""
    a = b = float("-inf")
    for v in values:
        if v != v:
            b = max(b, a)
        else:
            b, a = max(b, min(a, v)), max(a, v)
    return a + b if len(values) > 1 else a


@pytest.mark.parametrize("n", [1, 5, 64])
@pytest.mark.parametrize("E,groups,top", [(2, (2, 1), 1), (8, (4, 2), 2), (64, (8, 3), 6), (64, (64, 7), 7), (48, (3, 2), 4), (32, (2, 2), 8)])
def test_groups_of_experts_in_lanes(ops, n, E, groups, top):  # noqa: F811
    """Against the rule in plain Python, with equal scores, infinities and a logit that is no number among them."""
    z, c = rnd(n, E), rnd(E, seed=3, scale=0.1)
    z[0, :] = 0.5
    c[:2] = 0.0
    if n > 1:
        z[1, 0], z[1, 1] = float("inf"), float("-inf")
        if groups[1] < groups[0]:  # (without a choice of groups the lanes' own order of what is no number holds)
            z[2, E // 2] = float("nan")
    ids, weights = route(ops, z, n, E, top, 16, scores="logistic", groups=groups, correction=c)
    score = 1.0 / (1.0 + torch.exp(-z.cpu()))
    per = E // groups[0]
    for t in range(n):
        # (what is no number is never chosen; in its group's score the largest ahead of it stands again)
        raw = (score[t] + c.cpu()).tolist()
        key = [(v if v == v else float("-inf")) for v in raw]
        best2 = [group_score(raw[g * per:(g + 1) * per]) for g in range(groups[0])]
        kept = sorted(range(groups[0]), key=lambda g: (-best2[g], g))[:groups[1]]
        want = sorted((e for e in range(E) if e // per in kept), key=lambda e: (-key[e], e))[:top]
        got = ids[t * top:(t + 1) * top].tolist()
        # (scores that the two exponentials round apart may change places)
        assert all(abs(key[x] - key[y]) < 1e-6 for x, y in zip(got, want)), (got, want)
        torch.testing.assert_close(weights[t * top:(t + 1) * top].cpu(), score[t][got], rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("groups", [(32, 9), (32, 5), (16, 3), (8, 2), (4, 3), (2, 1)])
def test_logits_that_are_no_numbers_choose_the_same_groups_in_lanes_and_in_a_walk(ops, groups):  # noqa: F811
    """64 experts, an expert a lane, against 64 and one group more that is never kept, which the kernel that walks takes: the same choices and weights, with none to five logits a
    token that are no numbers, and infinities."""
    n, E, per, top = 64, 64, 64 // groups[0], 5
    more, wide = per, (groups[0] + 1, groups[1])
    z, c = rnd(n, E, seed=7), rnd(E, seed=8, scale=0.1)
    g = torch.Generator().manual_seed(9)
    for t in range(n):
        z[t, torch.randperm(E, generator=g)[:t % 6].to(DEV)] = float("nan")
    z[3, 5], z[4, 9] = float("inf"), float("-inf")
    z2, c2 = torch.cat([z, torch.zeros(n, more, device=DEV)], 1).contiguous(), torch.cat([c, torch.full((more,), -10.0, device=DEV)])
    a = route(ops, z, n, E, top, 16, scores="logistic", groups=groups, correction=c)
    b = route(ops, z2, n, E + more, top, 16, scores="logistic", groups=wide, correction=c2)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
