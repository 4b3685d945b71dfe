"""The tiles of many rows: shapes and edges."""

import pytest
import torch

from test_kernels_gpu import DEV, close, gemm_reference, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("epilogue", ["none", "gelu_tanh", "gelu_erf", "residual"])
@pytest.mark.parametrize("M,N,K", [(1, 8, 64), (65, 97, 64), (330, 680, 128), (161, 321, 192), (300, 264, 832), (129, 1000, 1600), (520, 3000, 128), (2100, 1416, 192), (700, 4200, 1536)])
def test_tiles_of_every_shape(ops, M, N, K, epilogue):  # noqa: F811
    """Against float64, from one unit of K to more than the rings hold, no whole number of tiles, N with no wide stores (97) and a large
    `w` among them; a tile's bits do not depend on its shape. Tolerances: sums of K products of 32 bits, those of the tiles' other tests."""
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    for dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 5e-3)):
        if epilogue == "residual" and dtype == torch.bfloat16:
            continue
        first = None
        for tile in (6, 2, 7, 8, 9, 11, 15, 21):
            if epilogue == "residual":
                out = rnd(M, N, seed=3)
                want = gemm_reference(a, w, bias, epilogue, out)
                ops.gemm_mfma_dl(a, w, bias, residual=out, epilogue=ops.EPI_RESIDUAL, tile=tile)
            else:
                out = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
                want = gemm_reference(a, w, bias, epilogue)
                ops.gemm_mfma_dl(a, w, bias, out=out, epilogue=ops.ACTIVATION_EPILOGUE[epilogue], tile=tile)
            close(out, want, tol, f"tile {tile}")
            first = out if first is None else first
            assert torch.equal(out, first), f"tile {tile} against 6"


@pytest.mark.parametrize("tile", [2, 8, 15, 21])
@pytest.mark.parametrize("M,H,Hkv,hd,K,page", [(5, 3, 3, 16, 64, 4), (200, 5, 5, 48, 192, 8), (700, 6, 3, 64, 128, 16), (300, 4, 2, 64, 192, 48), (170, 5, 1, 80, 256, 16)])
def test_tiles_write_pages(ops, tile, M, H, Hkv, hd, K, page):  # noqa: F811
    """Queries, keys and values where 64 x 64 tiles put them, bit for bit."""
    q_dim, kv_dim = H * hd, Hkv * hd
    N = q_dim + 2 * kv_dim
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    pages = -(-M // page) + 3
    slots = torch.randperm(pages * page)[:M].to(torch.int32).to(DEV)
    got = []
    for t in (6, tile):
        kc = torch.zeros(pages, Hkv, page, hd, dtype=torch.bfloat16, device=DEV)
        vc, q = torch.zeros_like(kc), torch.zeros(M, q_dim, dtype=torch.bfloat16, device=DEV)
        ops.gemm_mfma_dl(a, w, bias, out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, q_dim), tile=t)
        got.append((q, kc, vc))
    for x, y in zip(*got):
        assert torch.equal(x, y)


@pytest.mark.parametrize("tile", [2, 6, 7, 8, 9, 11, 15, 21])
@pytest.mark.parametrize("M,H,Hkv,hd,K,page", [(70, 3, 3, 16, 64, 4), (300, 6, 3, 64, 192, 16), (20, 5, 1, 6, 128, 16)])
def test_tiles_write_pages_in_32_bits(ops, tile, M, H, Hkv, hd, K, page):  # noqa: F811
    """bfloat16 operands, queries and caches in 32 bits: the sums that stand in a plain output, in their places, and nothing elsewhere; heads that four outputs
    side by side do not divide (6) among them."""
    q_dim, kv_dim = H * hd, Hkv * hd
    N = q_dim + 2 * kv_dim
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    pages = -(-M // page) + 3
    slots = torch.randperm(pages * page)[:M].to(torch.int32).to(DEV)
    slots[1] = -1
    flat = torch.empty(M, N, device=DEV)
    ops.gemm_mfma_dl(a, w, bias, out=flat, tile=tile)
    kc = torch.full((pages, Hkv, page, hd), 7.0, device=DEV)
    vc, q = kc.clone(), torch.zeros(M, q_dim, device=DEV)
    want_k, want_v = kc.clone(), vc.clone()
    ops.gemm_mfma_dl(a, w, bias, out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, q_dim), tile=tile)
    real = (slots >= 0).nonzero()[:, 0]
    at = slots[real].long()
    want_k[at // page, :, at % page] = flat[real, q_dim:q_dim + kv_dim].view(-1, Hkv, hd)
    want_v[at // page, :, at % page] = flat[real, q_dim + kv_dim:].view(-1, Hkv, hd)
    assert torch.equal(q, flat[:, :q_dim]) and torch.equal(kc, want_k) and torch.equal(vc, want_v)
