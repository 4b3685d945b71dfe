"""Products of 17 to 64 rows from waves with rings of their own."""

import pytest
import torch

from test_kernels_gpu import DEV, close, gemm_reference, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


# a row and a tile's edge, one unit of K to more than eight, no whole number of strips, N with no wide stores (97), each of the four tiles (32 x 16 and 32 x 32 of few
# strips, 48 x 32, 64 x 32), more than one tile of rows
SHAPES = [(17, 97, 64), (1, 2064, 128), (33, 1284, 448), (32, 6152, 576), (31, 4808, 512), (48, 6400, 640), (40, 4999, 128), (64, 4808, 1600), (49, 8192, 192), (70, 520, 192),
          (48, 6408, 1344), (41, 4999, 1344)]


@pytest.mark.parametrize("epilogue", ["none", "gelu_tanh", "gelu_erf", "residual"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_products_of_a_tile_of_rows(ops, M, N, K, epilogue):  # noqa: F811
    """Against float64; tolerances: sums of K products of 32 bits, those of the tiles' tests. A row has the same bits among other rows."""
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    for dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 5e-3)):
        if epilogue == "residual" and dtype == torch.bfloat16:
            continue

        def run(rows):
            if epilogue == "residual":
                out = rnd(M, N, seed=3)[rows].contiguous()
                ops.gemm_mfma_dl(a[rows], w, bias, residual=out, epilogue=ops.EPI_RESIDUAL, tile=18)
            else:
                out = torch.full((a[rows].shape[0], N), float("nan"), dtype=dtype, device=DEV)
                ops.gemm_mfma_dl(a[rows], w, bias, out=out, epilogue=ops.ACTIVATION_EPILOGUE[epilogue], tile=18)
            return out

        got = run(slice(0, M))
        close(got, gemm_reference(a, w, bias, epilogue, rnd(M, N, seed=3)) if epilogue == "residual" else gemm_reference(a, w, bias, epilogue), tol, "tile 18")
        assert torch.equal(run(slice(M // 2, M // 2 + 1)), got[M // 2:M // 2 + 1])


@pytest.mark.parametrize("M,H,Hkv,hd,K,page", [(33, 3, 3, 16, 64, 4), (64, 25, 25, 64, 192, 16), (20, 6, 3, 64, 128, 16), (40, 40, 20, 64, 192, 48), (17, 5, 1, 80, 1600, 16),
                                                (40, 40, 20, 64, 1344, 48), (64, 25, 25, 64, 1344, 16)])
def test_they_write_pages(ops, M, H, Hkv, hd, K, page):  # noqa: F811
    """Queries to their rows, keys and values to their slots, and nothing anywhere else; a slot outside the pages is not written."""
    q_dim, kv_dim = H * hd, Hkv * hd
    N = q_dim + 2 * kv_dim
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    pages = -(-M // page) + 3
    slots = torch.randperm(pages * page)[:M].to(torch.int32).to(DEV)
    slots[1] = -1
    flat = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.gemm_mfma_dl(a, w, bias, out=flat, tile=18)
    kc = torch.full((pages, Hkv, page, hd), 7.0, dtype=torch.bfloat16, device=DEV)
    vc, q = kc.clone(), torch.zeros(M, q_dim, dtype=torch.bfloat16, device=DEV)
    want_k, want_v = kc.clone(), vc.clone()
    ops.gemm_mfma_dl(a, w, bias, out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, q_dim), tile=18)
    for m, s in enumerate(slots.tolist()):
        if s >= 0:
            want_k[s // page, :, s % page] = flat[m, q_dim:q_dim + kv_dim].view(Hkv, hd)
            want_v[s // page, :, s % page] = flat[m, q_dim + kv_dim:].view(Hkv, hd)
    assert torch.equal(q, flat[:, :q_dim]) and torch.equal(kc, want_k) and torch.equal(vc, want_v)


@pytest.mark.parametrize("n_base", [0, 1, 4, 6])
@pytest.mark.parametrize("M,N,K,parts", [(33, 768, 3072, 4), (64, 1600, 6400, 4), (64, 1284, 1280, 1), (24, 4096, 1024, 2), (50, 99, 320, 3), (45, 4099, 1344, 2), (60, 4100, 1344, 2)])
def test_cut_over_k(ops, M, N, K, parts, n_base):  # noqa: F811
    """The planes add up to base + a . w^T + bias."""
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    base = torch.stack([rnd(M, N, seed=4 + p) for p in range(n_base)]) if n_base else None
    planes = torch.full((parts, M, N), float("nan"), device=DEV)
    ops.gemm_mfma_dl_parts(a, w, planes, bias=bias if n_base else None, base=base, tile=18)
    want = gemm_reference(a, w, bias if n_base else torch.zeros_like(bias), "none")
    if n_base:
        want = want + base.double().sum(0).to(want.device)
    close(planes.double().sum(0), want, 1e-5, "planes")


@pytest.mark.parametrize("M,N,K", [(17, 2056, 64), (24, 4800, 1600), (33, 2304, 768), (48, 6400, 1600), (64, 4808, 832), (64, 1284, 448)])
def test_they_have_the_tiles_bits(ops, M, N, K):  # noqa: F811
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    base = rnd(3, M, N, seed=5)
    got = []
    for tile in (16, 17, 18):
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        ops.gemm_mfma_dl(a, w, bias, out=out, epilogue=ops.EPI_GELU_TANH, tile=tile)
        res = rnd(M, N, seed=3)
        ops.gemm_mfma_dl(a, w, bias, residual=res, epilogue=ops.EPI_RESIDUAL, tile=tile)
        planes = torch.empty(1 if K < 256 else 3, M, N, device=DEV)
        ops.gemm_mfma_dl_parts(a, w, planes, bias=bias, base=base, tile=tile)
        got.append((out, res, planes))
    for g in got[1:]:
        for x, y in zip(got[0], g):
            assert torch.equal(x, y)


def test_the_rule(ops):  # noqa: F811
    pay = ops.waves_pay
    assert pay(64, 1600) and pay(33, 768) and pay(64, 3072 * 4, 4) and pay(17, 4096) and pay(32, 4096 * 2, 2)
    assert not pay(64, 4096) and not pay(16, 1600) and not pay(65, 1600) and not pay(64, 1608) and not pay(20, 4160)
