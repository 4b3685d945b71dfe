"""Each kernel alone against a plain 32-bit PyTorch reference of the same operation, at
sizes other than the engine's (needs the GPU)."""

import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from liyab_amd.kernels import ops as o

    o.check_device()
    return o


def rnd(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator(device="cpu").manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def close(got, want, tol, what=""):
    got, want = got.double().cpu(), want.double().cpu()
    err = (got - want).abs().max().item() / max(want.abs().max().item(), 1e-30)
    assert math.isfinite(err) and err <= tol, f"{what}: relative error {err:.3e} > {tol:.1e}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,d", [(1, 64), (7, 100), (33, 1600), (5, 4096 + 24), (3, 4096), (2, 777), (4, 8200), (9, 768)])
def test_embed_and_add_rows(ops, dtype, n, d):
    V, P = 321, 77
    table, pos = rnd(V, d, dtype=dtype), rnd(P, d, dtype=dtype, seed=1)
    ids = torch.randint(0, V, (n,), dtype=torch.int32, device=DEV)
    positions = torch.randint(0, P, (n,), dtype=torch.int32, device=DEV)
    out = torch.empty(n, d, device=DEV)
    ops.embed(out, table, ids, 1.0, pos_table=pos, positions=positions)
    want = table.float()[ids.long()] + pos.float()[positions.long()]
    assert torch.equal(out, want)
    ops.embed(out, table, ids, 2.5)
    assert torch.equal(out, table.float()[ids.long()] * 2.5)
    ops.add_rows_(out, pos, positions)
    assert torch.equal(out, table.float()[ids.long()] * 2.5 + pos.float()[positions.long()])


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,d,eps", [(1, 64, 1e-5), (9, 96, 1e-6), (40, 1600, 1e-5), (3, 777, 1e-3), (5, 768, 1e-5),
                                     (70, 260, 1e-5), (6, 1028, 1e-6), (7, 2048, 1e-5), (2, 2052, 1e-5), (4, 4096, 1e-5), (3, 5120, 1e-6),
                                     (2, 16384, 1e-5), (2, 16388, 1e-5), (3, 4098, 1e-5)])
def test_layernorm(ops, out_dtype, n, d, eps):
    x = rnd(n + 3, d, scale=3.0) + 1.5
    w, b = rnd(d, seed=2) + 1.0, rnd(d, seed=3)
    out = torch.empty(n, d, dtype=out_dtype, device=DEV)
    ops.layernorm(out, x, w, b, eps)
    want = torch.nn.functional.layer_norm(x[:n].double(), (d,), w.double(), b.double(), eps)
    close(out, want, 1e-6 if out_dtype == torch.float32 else 5e-3, "layernorm")
    rows = torch.tensor([(i * 2) % (n + 3) for i in range(n)], dtype=torch.int32, device=DEV)
    ops.layernorm(out, x, w, None, eps, rows=rows)
    want = torch.nn.functional.layer_norm(x[rows.long()].double(), (d,), w.double(), None, eps)
    close(out, want, 1e-6 if out_dtype == torch.float32 else 5e-3, "layernorm gather")
    # eps is the kernel's argument, not a constant: a low-variance row shows it
    flat = torch.ones(1, d, device=DEV) + 1e-3 * rnd(1, d, seed=9)
    o1, o2 = torch.empty(1, d, device=DEV), torch.empty(1, d, device=DEV)
    ops.layernorm(o1, flat, None, None, 1e-5)
    ops.layernorm(o2, flat, None, None, 1e-6)
    assert (o1 - o2).abs().max() > 1e-2


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,d,parts", [(1, 64, 1), (9, 96, 4), (16, 768, 4), (5, 1600, 2), (7, 2048, 5), (6, 200, 16), (70, 768, 3),
                                       (5, 4096, 3), (2, 8192, 4), (3, 2052, 2)])
def test_layernorm_over_rows_in_planes(ops, out_dtype, n, d, parts):
    """Rows given as a sum of planes: the norm adds the planes up, in their order, as it loads a
    row, also over gathered rows; sum_parts alone does the same sum (into a tensor of its own or
    into the first plane); widths the kernel does not take in planes are refused."""
    tol = 1e-6 if out_dtype == torch.float32 else 5e-3
    planes = rnd(parts, n + 3, d, seed=4, scale=0.7)
    planes[0] += 1.5
    w, b = rnd(d, seed=2) + 1.0, rnd(d, seed=3)
    total = planes.double().sum(0)
    want = torch.nn.functional.layer_norm(total, (d,), w.double(), b.double(), 1e-5)
    out = torch.empty(n, d, dtype=out_dtype, device=DEV)
    before = planes.clone()
    ops.layernorm(out, planes, w, b, 1e-5)
    close(out, want[:n], tol, "layernorm over planes")
    assert torch.equal(planes, before)  # the planes stay as they are
    summed = torch.empty(n + 3, d, device=DEV)
    ops.sum_parts(summed, planes)
    close(summed, total, 1e-6, "sum of the planes")
    whole = torch.empty(n, d, dtype=out_dtype, device=DEV)
    ops.layernorm(whole, summed, w, b, 1e-5)
    assert torch.equal(whole, out)  # the same order of additions
    rows = torch.tensor([(i * 3) % (n + 3) for i in range(n + 2)], dtype=torch.int32, device=DEV)  # names rows twice
    out = torch.empty(n + 2, d, dtype=out_dtype, device=DEV)
    ops.layernorm(out, planes, w, b, 1e-5, rows=rows)
    close(out, want[rows.long()], tol, "gathered layernorm over planes")
    ops.sum_parts(planes[0], planes)
    assert torch.equal(planes[0], summed)
    if parts > 1:
        odd = rnd(parts, 3, 777, seed=6)
        assert not ops.norm_takes_planes(777)
        with pytest.raises(Exception, match="planes"):
            ops.layernorm(torch.empty(3, 777, device=DEV), odd, rnd(777), rnd(777), 1e-5)
    with pytest.raises(Exception, match="rows of d"):
        ops.layernorm(torch.empty(n, d, device=DEV), planes[:, :, :-4].contiguous(), w, b, 1e-5)


@pytest.mark.parametrize("M,N,K,parts", [(1, 64, 128, 2), (8, 768, 3072, 4), (16, 100, 200, 2), (5, 1600, 6400, 2), (40, 50, 448, 7),
                                         (64, 264, 1600, 3), (3, 40, 64, 1), (11, 130, 1032, 4)])
def test_gemm_skinny_parts(ops, M, N, K, parts):
    """The product cut over K: plane p holds the sums over the p-th part of K (whole units of
    64, the last one shorter); the planes add up to the product. With rows to add to (a tensor
    or planes of their own), the first plane also takes them and the bias, and the planes add
    up to rows + product + bias."""
    a, w = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16)
    planes = torch.full((parts, M, N), float("nan"), device=DEV)
    ops.gemm_skinny_parts(a, w, planes)
    units = (K + 63) // 64
    part_k = (units + parts - 1) // parts * 64
    for q in range(parts):
        lo, hi = q * part_k, min(K, (q + 1) * part_k)
        close(planes[q], a[:, lo:hi].double() @ w[:, lo:hi].double().t(), 1e-5, f"part {q}")
    product = a.double() @ w.double().t()
    close(planes.sum(0), product, 1e-5, "sum of the parts")
    bias = rnd(N, seed=7)
    for n_base in (0, 1, 3, 6):
        base = rnd(M, N, seed=8, scale=3.0) if n_base == 0 else rnd(n_base, M, N, seed=9, scale=3.0)
        for with_bias in (True, False):
            based = torch.full((parts, M, N), float("nan"), device=DEV)
            ops.gemm_skinny_parts(a, w, based, bias=bias if with_bias else None, base=base)
            assert torch.equal(based[1:], planes[1:])
            rows = base.double() if n_base == 0 else base.double().sum(0)
            want0 = planes[0].double() + rows + (bias.double() if with_bias else 0)
            close(based[0], want0, 1e-6, f"first plane over {n_base} planes of rows")
            close(based.double().sum(0), product + rows + (bias.double() if with_bias else 0), 1e-5, "sum with rows")
    with pytest.raises(Exception, match="parts"):
        ops.gemm_skinny_parts(a, w, torch.empty(K // 64 + 2, M, N, device=DEV))
    with pytest.raises(Exception, match="bias needs"):
        ops.gemm_skinny_parts(a, w, planes, bias=bias)
    with pytest.raises(Exception, match="overlap"):
        ops.gemm_skinny_parts(a, w, planes, base=planes[:1])


@pytest.mark.parametrize("tile", [6, 16, 17])
@pytest.mark.parametrize("M,N,K,parts", [(64, 768, 3072, 4), (2048, 768, 3072, 2), (200, 100, 448, 3), (33, 1600, 6400, 4), (1, 40, 64, 1),
                                         (130, 777, 1088, 5)])
def test_gemm_tiled_parts(ops, tile, M, N, K, parts):
    """The tiled product cut over K: plane p holds the sums over the p-th part of K (whole tiles
    of 64); with rows to add to, the first plane also takes them and the bias."""
    a, w = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16)
    planes = torch.full((parts, M, N), float("nan"), device=DEV)
    ops.gemm_mfma_dl_parts(a, w, planes, tile=tile)
    part_k = (K // 64 + parts - 1) // parts * 64
    for q in range(parts):
        lo, hi = q * part_k, min(K, (q + 1) * part_k)
        close(planes[q], a[:, lo:hi].double() @ w[:, lo:hi].double().t(), 1e-5, f"part {q}")
    product = a.double() @ w.double().t()
    bias = rnd(N, seed=7)
    for n_base in (0, 3):
        base = rnd(M, N, seed=8, scale=3.0) if n_base == 0 else rnd(n_base, M, N, seed=9, scale=3.0)
        for with_bias in (True, False):
            based = torch.full((parts, M, N), float("nan"), device=DEV)
            ops.gemm_mfma_dl_parts(a, w, based, bias=bias if with_bias else None, base=base, tile=tile)
            assert torch.equal(based[1:], planes[1:])
            rows = base.double() if n_base == 0 else base.double().sum(0)
            close(based[0], planes[0].double() + rows + (bias.double() if with_bias else 0), 1e-6, f"first plane over {n_base} planes of rows")
            close(based.double().sum(0), product + rows + (bias.double() if with_bias else 0), 1e-5, "sum with rows")
    with pytest.raises(Exception, match="parts"):
        ops.gemm_mfma_dl_parts(a, w, torch.empty(K // 64 + 2, M, N, device=DEV), tile=tile)
    with pytest.raises(Exception, match="overlap"):
        ops.gemm_mfma_dl_parts(a, w, planes, base=planes[:1], tile=tile)


def gemm_reference(a, w, bias, epilogue, residual=None):
    y = a.double() @ w.double().t()
    if bias is not None:
        y = y + bias.double()
    if epilogue == "gelu_tanh":
        y = torch.nn.functional.gelu(y, approximate="tanh")
    elif epilogue == "gelu_erf":
        y = torch.nn.functional.gelu(y)
    elif epilogue == "residual":
        y = residual.double() + y
    return y


GEMM_SHAPES = [(1, 64, 64), (7, 200, 96), (33, 777, 144), (130, 50, 320), (64, 1000, 96), (257, 130, 72)]


# beside those: strips of 16 rows by 4, 8 and 16 features, chunks of K with a tail, more chunks than waves, a K that is no multiple
# of 4 (element by element), products of many features
F32_SHAPES = GEMM_SHAPES + [(16, 1500, 100), (9, 2600, 260), (5, 3000, 72), (12, 40, 6), (40, 2561, 132), (3, 1024, 1028),
                            (16, 33, 3076), (20, 70, 50),
                            # two to four strips of rows: 16 features a strip on four and eight waves, 4 and 8 with a long K
                            (24, 4100, 200), (45, 4097, 68), (64, 4800, 324), (30, 2050, 1604), (17, 100, 3076),
                            # tiles of 64 x 64 (from 136 of them on): many of them with edges on both sides; a long K; just 136; a K that
                            # is no multiple of 4
                            (1100, 7300, 68), (700, 770, 3072), (65, 4352, 1604), (300, 2304, 770)]


@pytest.mark.parametrize("epilogue", ["none", "gelu_tanh", "gelu_erf", "residual"])
@pytest.mark.parametrize("M,N,K", F32_SHAPES)
def test_gemm_float32(ops, M, N, K, epilogue):
    a, w, bias = rnd(M, K), rnd(N, K, seed=1, scale=0.2), rnd(N, seed=2)
    if epilogue == "residual":
        res = rnd(M, N, seed=3)
        want = gemm_reference(a, w, bias, epilogue, res)
        ops.gemm(a, w, bias, residual=res, epilogue=ops.EPI_RESIDUAL)
        close(res, want, 2e-6, "gemm f32 residual")
    else:
        out = torch.empty(M, N, device=DEV)
        ops.gemm(a, w, bias, out=out, epilogue=ops.ACTIVATION_EPILOGUE[epilogue])
        close(out, gemm_reference(a, w, bias, epilogue), 2e-6, f"gemm f32 {epilogue}")
    # a row's result does not depend on the rows around it, nor on which kernel their number chooses
    if M > 1:
        one = torch.empty(1, N, device=DEV)
        ops.gemm(a[M // 2:M // 2 + 1], w, bias, out=one)
        full = torch.empty(M, N, device=DEV)
        ops.gemm(a, w, bias, out=full)
        assert torch.equal(one[0], full[M // 2])
        few = torch.empty(min(M, 40), N, device=DEV)  # strips, also of shapes that run in tiles
        ops.gemm(a[M - len(few):], w, bias, out=few)
        assert torch.equal(few, full[M - len(few):])
        many = torch.empty(70 + M, N, device=DEV)  # among 70 rows more: other strips, other tiles, or tiles instead of strips
        rows = torch.cat([rnd(70, K, seed=9), a])
        ops.gemm(rows, w, bias, out=many)
        assert torch.equal(many[70:], full)
        # from an address that is no multiple of 16 bytes operands are loaded element by element
        shifted = torch.empty(rows.numel() + 1, device=DEV)[1:].view_as(rows).copy_(rows)
        assert shifted.data_ptr() % 16 != 0
        ops.gemm(shifted, w, bias, out=many)
        assert torch.equal(many[70:], full)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (16, 1024, 63), (16, 1025, 65), (17, 1024, 64), (3, 2049, 130), (16, 6400, 128), (16, 6401, 68), (64, 3, 257),
                                   (65, 4288, 96), (65, 4289, 96), (65, 4352, 100), (129, 4351, 33), (700, 770, 200), (64, 8700, 64)])
def test_gemm_float32_at_the_edges_of_its_kernels(ops, M, N, K):
    """Strips of 4, 8 and 16 features, tiles of 64 x 64 (from 136 of them on), remainders in every direction, operands with
    16-byte loads and without, rows of outputs wider than N. The error of a chain of n multiply-adds is within n 2^-24 times
    the sum of |a w|: 64 a chunk, the chunks' sums, the bias."""
    a, w, bias = rnd(M, K), rnd(N, K, seed=1), rnd(N, seed=2)
    want = a.double() @ w.double().t() + bias.double()
    bound = (a.double().abs() @ w.double().abs().t() + bias.double().abs()) * ((min(K, 64) + K / 64 + 2) * 2.0 ** -24)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm_simple(a, w, bias, out=out)
    assert ((out.double() - want).abs() <= bound).all()
    shifted = torch.empty(M * K + 1, device=DEV)[1:].view(M, K).copy_(a)  # no 16-byte loads
    wider = torch.full((M, N + 3), float("nan"), device=DEV)
    ops.gemm_simple(shifted, w, bias, out=wider[:, :N])
    assert torch.equal(wider[:, :N], out) and wider[:, N:].isnan().all()
    res = rnd(M, N, seed=3)
    base = res.clone()
    ops.gemm_simple(a, w, bias, residual=res, epilogue=ops.EPI_RESIDUAL)
    assert torch.equal(res, base + out)
    one = torch.empty(1, N, device=DEV)  # a row alone: the kernel for few rows, in strips of its own
    ops.gemm_simple(a[M - 1:], w, bias, out=one)
    assert torch.equal(one[0], out[M - 1])


@pytest.mark.parametrize("K", [64, 130, 768])
@pytest.mark.parametrize("M,N", [(20, 70), (700, 770)])
def test_gemm_float32_is_chains_of_fused_multiply_adds(ops, M, N, K):
    """Every result has the bits of the chains it stands for, 64 k from zero each, the chunks' sums added in order, computed on the
    host with the C library's fmaf: for ordinary operands, for products below the normal numbers and for operands below them; in
    strips (20 x 70) and in tiles (143 of them)."""
    import ctypes

    fmaf = ctypes.CDLL("libm.so.6").fmaf
    fmaf.restype, fmaf.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    rng = np.random.default_rng(K + M)
    places = [(0, 0), (M - 1, N - 1)] + [(int(rng.integers(M)), int(rng.integers(N))) for _ in range(60)]
    for scale_a, scale_w in ((1.0, 1.0), (1e-20, 1e-20), (1e-40, 1.0)):
        a, w = (rng.standard_normal((M, K)) * scale_a).astype(np.float32), (rng.standard_normal((N, K)) * scale_w).astype(np.float32)
        out = torch.empty(M, N, device=DEV)
        ops.gemm_simple(torch.from_numpy(a).to(DEV), torch.from_numpy(w).to(DEV), None, out=out)
        got = out.cpu().numpy()
        for m, n in places:
            total = np.float32(0.0)
            for k0 in range(0, K, 64):
                chain = 0.0
                for x, y in zip(a[m, k0:k0 + 64].tolist(), w[n, k0:k0 + 64].tolist()):
                    chain = fmaf(x, y, chain)
                total = np.float32(total + np.float32(chain))
            assert got[m, n].tobytes() == total.tobytes(), (scale_a, scale_w, m, n, got[m, n], total)


@pytest.mark.parametrize("kernel", ["simple", "mfma128", "mfma64", "mfma128x64", "auto", "skinny1", "skinny4", "skinny16", "skinny4w", "skinny2w", "skinny8m1", "skinny4m2", "skinny2m4",
                                    "dl2", "dl6", "dl7", "dl8", "dl9", "dl11", "dl15", "dl16", "dl17"])
@pytest.mark.parametrize("epilogue", ["none", "gelu_tanh", "gelu_erf", "residual"])
@pytest.mark.parametrize("M,N,K", GEMM_SHAPES + [(300, 264, 1600), (2, 50257 // 16, 64), (8, 130, 3072), (16, 2304, 768), (3, 40, 200), (17, 100, 64), (40, 333, 768), (64, 257, 1600),
                                                 (500, 300, 128), (129, 193, 192), (20, 4800, 1600), (600, 520, 256), (1030, 770, 128), (5, 100, 16384)])
def test_gemm_bfloat16(ops, M, N, K, epilogue, kernel):
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    tiles = {"mfma128": 1, "mfma64": 2, "mfma128x64": 3}

    if kernel.startswith("skinny") and M > 64:
        pytest.skip("the skinny kernel takes at most 64 rows")

    if kernel.startswith("dl") and K % 64 != 0:
        pytest.skip("the direct-load kernel takes K in multiples of 64")

    def run(**kw):
        if kernel.startswith("dl"):
            ops.gemm_mfma_dl(a, w, bias, tile=int(kernel[2:]), **kw)
        elif kernel.startswith("skinny"):
            spec, _, mtile = kernel[6:].partition("m")  # split of K, "w" for wide tiles of N, "m<tiles of rows>"
            ops.gemm_skinny(a, w, bias, ksplit=int(spec.rstrip("w")), wide=1 if spec.endswith("w") else 0,
                            mtile=int(mtile or 0), **kw)
        elif kernel == "simple":
            ops.gemm_simple(a, w, bias, **kw)
        elif kernel == "auto":
            ops.gemm(a, w, bias, **kw)
        else:
            ops.gemm_mfma(a, w, bias, tile=tiles[kernel], **kw)

    if epilogue == "residual":
        res = rnd(M, N, seed=3)
        want = gemm_reference(a, w, bias, epilogue, res)
        run(residual=res, epilogue=ops.EPI_RESIDUAL)
        close(res, want, 1e-5, f"gemm bf16 residual {kernel}")
    else:
        for out_dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 5e-3)):
            out = torch.empty(M, N, dtype=out_dtype, device=DEV)
            run(out=out, epilogue=ops.ACTIVATION_EPILOGUE[epilogue])
            close(out, gemm_reference(a, w, bias, epilogue), tol, f"gemm bf16 {epilogue} {kernel} -> {out_dtype}")


@pytest.mark.parametrize("epilogue", ["none", "gelu_tanh", "gelu_erf"])
@pytest.mark.parametrize("M,N,K,eps,parts", [(1, 64, 64, 1e-5, 1), (8, 2304, 768, 1e-5, 4), (16, 100, 1600, 1e-6, 2), (5, 777, 144, 1e-5, 3),
                                             (3, 50, 2048, 1e-3, 5), (13, 520, 1024, 1e-5, 1), (9, 3072, 768, 1e-5, 2), (16, 48, 96, 1e-6, 16),
                                             (17, 200, 768, 1e-5, 2), (32, 2304, 768, 1e-5, 1), (24, 130, 1600, 1e-6, 3), (29, 3072, 768, 1e-5, 1),
                                             (32, 90, 1024, 1e-5, 4)])
def test_gemm_with_layernorm_folded_in(ops, M, N, K, eps, parts, epilogue):
    """The product kernel that normalises its own rows, given whole or as a sum of planes: the
    same bits as the standalone norm followed by the streaming product."""
    planes = rnd(parts, M, K, scale=2.0)
    planes[0] += 0.5
    lw, lb = rnd(K, seed=5) + 1.0, rnd(K, seed=6)
    w, bias = rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    x = planes if parts > 1 else planes[0]
    h = torch.nn.functional.layer_norm(planes.double().sum(0), (K,), lw.double(), lb.double(), eps).to(torch.bfloat16)
    epi = ops.ACTIVATION_EPILOGUE[epilogue]
    for out_dtype in (torch.float32, torch.bfloat16):
        out = torch.full((M, N), float("nan"), dtype=out_dtype, device=DEV)
        ops.gemm_skinny_ln(x, lw, lb, eps, w, bias, out=out, epilogue=epi, wide=0)
        if M <= 16:
            strips_of_32 = torch.full((M, N), float("nan"), dtype=out_dtype, device=DEV)
            ops.gemm_skinny_ln(x, lw, lb, eps, w, bias, out=strips_of_32, epilogue=epi, wide=1)
            assert torch.equal(out, strips_of_32)
        # the folded norm rounds to bfloat16 where the standalone kernel does: allow one ulp of the operand
        close(out, gemm_reference(h, w, bias, epilogue), 4e-3 if out_dtype == torch.float32 else 8e-3, f"gemm+ln {epilogue}")
        normed = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
        ops.layernorm(normed, x, lw, lb, eps)
        two = torch.empty(M, N, dtype=out_dtype, device=DEV)
        ops.gemm_skinny(normed, w, bias, out=two, epilogue=epi, ksplit=8, wide=0, mtile=1 if M <= 16 else 0)
        if M <= 16:
            assert torch.equal(out, two)
        else:  # more tiles of rows: the plain kernel deals K out to its waves in another order
            close(out, two, 1e-5 if out_dtype == torch.float32 else 8e-3, "folded against norm + product")
    with pytest.raises(Exception, match="residual"):
        ops.gemm_skinny_ln(x, lw, lb, eps, w, bias, out=out, epilogue=ops.EPI_RESIDUAL)
    with pytest.raises(Exception, match="outside"):
        ops.gemm_skinny_ln(rnd(33, K), lw, lb, eps, w, bias, out=torch.empty(33, N, device=DEV))


def test_gemm_strided_rows_and_refusals(ops):
    from liyab_amd import KernelError

    wide = rnd(20, 256, dtype=torch.bfloat16)
    a = wide[:, 64:128]  # a view into a wider buffer: rows strided
    w = rnd(48, 64, dtype=torch.bfloat16, seed=1)
    out = torch.empty(20, 48, device=DEV)
    ops.gemm(a, w, None, out=out)
    close(out, a.double() @ w.double().t(), 1e-5, "strided a")
    with pytest.raises(KernelError):
        ops.gemm(a, rnd(48, 63, dtype=torch.bfloat16), None, out=out)  # K mismatch
    with pytest.raises(KernelError):
        ops.gemm(a, w, rnd(47), out=out)  # bias length
    with pytest.raises(KernelError):
        ops.gemm(a.float(), w, None, out=out)  # mixed dtypes
    with pytest.raises(KernelError):
        ops.gemm_mfma(rnd(4, 20, dtype=torch.bfloat16), rnd(8, 20, dtype=torch.bfloat16), None, out=torch.empty(4, 8, device=DEV))  # K % 8
    with pytest.raises(KernelError):
        ops.gemm(a, w, None, out=torch.empty(20, 48))  # not on the GPU


# ---------------------------------------------------------------------------
# attention over pages
# ---------------------------------------------------------------------------
def paged_case(n_seqs, ctx_lens, q_lens, H, Hkv, hd, page, dtype, seed=0, shuffle=True):
    """Random requests in a shuffled page pool; returns everything the kernels take and a
    float64 reference per token."""
    g = torch.Generator().manual_seed(seed)
    n_pages_per = [-(-c // page) for c in ctx_lens]
    total_pages = sum(n_pages_per) + 3
    perm = torch.randperm(total_pages, generator=g).tolist() if shuffle else list(range(total_pages))
    kc = torch.full((total_pages, Hkv, page, hd), float("nan"), dtype=dtype)
    vc = torch.full((total_pages, Hkv, page, hd), float("nan"), dtype=dtype)
    W = max(n_pages_per) + 1
    bt = torch.full((n_seqs, W), -1, dtype=torch.int32)
    ks, vs = [], []
    nxt = 0
    for s in range(n_seqs):
        k = (torch.randn(ctx_lens[s], Hkv, hd, generator=g)).to(dtype)
        v = (torch.randn(ctx_lens[s], Hkv, hd, generator=g)).to(dtype)
        ks.append(k)
        vs.append(v)
        for lp in range(n_pages_per[s]):
            pg = perm[nxt]
            nxt += 1
            bt[s, lp] = pg
            a, b = lp * page, min((lp + 1) * page, ctx_lens[s])
            kc[pg, :, :b - a] = k[a:b].transpose(0, 1)
            vc[pg, :, :b - a] = v[a:b].transpose(0, 1)
    tok_seq, tok_pos = [], []
    for s in range(n_seqs):
        for i in range(q_lens[s]):
            tok_seq.append(s)
            tok_pos.append(ctx_lens[s] - q_lens[s] + i)
    n = len(tok_seq)
    q = torch.randn(n, H * hd + 16, generator=g).to(dtype)  # wider than the heads: a strided view
    return dict(q=q, kc=kc, vc=vc, bt=bt, tok_seq=tok_seq, tok_pos=tok_pos, ks=ks, vs=vs, n=n)


def attention_reference(case, H, Hkv, hd, scale, window=0):
    out = torch.zeros(case["n"], H * hd, dtype=torch.float64)
    for t, (s, p) in enumerate(zip(case["tok_seq"], case["tok_pos"])):
        first = max(0, p - window + 1) if window > 0 else 0
        for h in range(H):
            hk = h // (H // Hkv)
            qv = case["q"][t, h * hd:(h + 1) * hd].double()
            k = case["ks"][s][first:p + 1, hk].double()
            v = case["vs"][s][first:p + 1, hk].double()
            w = torch.softmax((k @ qv) * scale, dim=0)
            out[t, h * hd:(h + 1) * hd] = w @ v
    return out


def run_attention(ops, case, H, hd, scale, window, kernel, splits=1, tok_list=None, waves=4, ksplit=1):
    dev = lambda x: x.to(DEV)  # noqa: E731
    q, kc, vc, bt = dev(case["q"]), dev(case["kc"]), dev(case["vc"]), dev(case["bt"])
    tok_seq = torch.tensor(case["tok_seq"], dtype=torch.int32, device=DEV)
    tok_pos = torch.tensor(case["tok_pos"], dtype=torch.int32, device=DEV)
    out = torch.zeros(case["n"], H * hd, dtype=q.dtype, device=DEV)
    qv = q[:, :H * hd]
    if kernel == "generic":
        ops.attention_generic(out, qv, kc, vc, bt, tok_seq, tok_pos, n_head=H, scale=scale, window=window)
    elif kernel == "prefill":
        work, row = [], 0
        lens = {}
        for sidx in case["tok_seq"]:
            lens[sidx] = lens.get(sidx, 0) + 1
        tile = splits if splits in (64, 128) else 128
        for sidx, nq in sorted(lens.items()):
            p0 = case["tok_pos"][row]
            for t0 in range(0, nq, tile):
                work.extend((sidx, row + t0, p0 + t0, min(tile, nq - t0)))
            row += nq
        wk = torch.tensor(work, dtype=torch.int32, device=DEV)
        ops.attention_prefill(out, qv, kc, vc, bt, wk, len(work) // 4, n_head=H, scale=scale, window=window, tile=tile,
                              ksplit=ksplit)
    elif kernel == "decode":
        partials = torch.empty(case["n"] * H * splits * (hd + 4), device=DEV) if splits > 1 else None
        tl = torch.tensor(tok_list, dtype=torch.int32, device=DEV) if tok_list is not None else None
        ops.attention_decode(out, qv, kc, vc, bt, tok_seq, tok_pos, n_head=H, scale=scale, window=window,
                             n_splits=splits, partials=partials, tok_list=tl, waves=waves,
                             n_tokens=len(tok_list) if tok_list is not None else None)
    return out


ATT_CASES = [
    # ctx_lens, q_lens, H, Hkv, hd, page
    ([1, 17, 300], [1, 1, 1], 4, 4, 16, 16),
    ([40, 129, 5], [7, 1, 5], 3, 3, 32, 16),
    ([700, 64], [1, 64], 5, 5, 64, 64),
    ([33, 257], [2, 3], 6, 2, 48, 8),
    ([100], [100], 2, 1, 128, 16),
    ([90, 31], [1, 1], 2, 2, 256, 16),
    ([50, 3], [4, 3], 3, 3, 80, 4),
    ([300, 40, 90], [8, 8, 8], 4, 2, 64, 16),
    # pages that are no power of two: page and offset by division
    ([130, 24, 49], [3, 1, 8], 3, 3, 32, 24),
    ([200, 97], [1, 5], 4, 2, 64, 48),
]


@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case_id", range(len(ATT_CASES)))
def test_attention_generic(ops, case_id, dtype, window):
    ctx_lens, q_lens, H, Hkv, hd, page = ATT_CASES[case_id]
    case = paged_case(len(ctx_lens), ctx_lens, q_lens, H, Hkv, hd, page, dtype, seed=case_id)
    scale = 0.7 / math.sqrt(hd)
    out = run_attention(ops, case, H, hd, scale, window, "generic")
    close(out, attention_reference(case, H, Hkv, hd, scale, window), 2e-6 if dtype == torch.float32 else 8e-3, "generic")


@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("splits,waves", [(1, 4), (1, 16), (2, 4), (5, 16), (32, 4), (1, 8), (3, 8)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case_id", range(len(ATT_CASES)))
def test_attention_decode(ops, case_id, dtype, splits, waves, window):
    ctx_lens, q_lens, H, Hkv, hd, page = ATT_CASES[case_id]
    case = paged_case(len(ctx_lens), ctx_lens, q_lens, H, Hkv, hd, page, dtype, seed=case_id)
    scale = 0.7 / math.sqrt(hd)
    out = run_attention(ops, case, H, hd, scale, window, "decode", splits, waves=waves)
    assert torch.isfinite(out.float()).all()
    close(out, attention_reference(case, H, Hkv, hd, scale, window), 8e-3 if dtype == torch.bfloat16 else 2e-6, f"decode splits={splits}")
    # a subset of the rows through tok_list: the others stay untouched
    if case["n"] > 2:
        rows = list(range(case["n"]))[::2]
        part = run_attention(ops, case, H, hd, scale, window, "decode", splits, tok_list=rows, waves=waves)
        assert torch.equal(part[rows], out[rows]) and (part[1::2] == 0).all()


# contexts at and beside one, two and three trips of a workgroup over the keys, where a wave's walk ends: (head size, waves, heads, keys a trip)
TRIPS = [(64, 4, 2, 128), (64, 8, 2, 256), (64, 16, 2, 1024), (128, 4, 2, 64), (128, 16, 2, 512), (256, 4, 1, 32), (16, 4, 2, 512), (32, 8, 1, 512), (32, 4, 160, 256), (64, 4, 160, 128)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("scores", ["plain", "kept", "worked on"])
@pytest.mark.parametrize("hd,waves,H,trip", TRIPS)
def test_attention_decode_at_the_ends_of_its_trips(ops, hd, waves, H, trip, scores, dtype):
    """Trips whose keys are all there, the last one's first and last key and the waves that have none in it, with 16 waves a token too, and on both
    sides of the number of workgroups up to which four waves ask for the next trip's keys ahead."""
    if dtype == torch.float32 and waves == 16:
        trip //= 2
    ctx_lens = [trip - 1, trip, trip + 1, trip + 64 // max(1, hd // 8) + 1] + ([2 * trip, 2 * trip + 1, 3 * trip, 3 * trip + 7] if H <= 2 else [2 * trip + 1])
    case = paged_case(len(ctx_lens), ctx_lens, [1] * len(ctx_lens), H, H, hd, 16, dtype, seed=hd + waves)
    scale, window, keep = 0.7 / math.sqrt(hd), trip - 3 if scores == "kept" else 0, 5 if scores == "kept" else 0
    cap, sinks, table = 0.0, None, None
    if scores == "worked on":
        g = torch.Generator().manual_seed(1)
        cap, sinks, table = 2.0, torch.randn(H, generator=g), torch.randn(trip // 2, H, generator=g)
    want = torch.zeros(case["n"], H * hd, dtype=torch.float64)
    for t, p in enumerate(case["tok_pos"]):
        seen = torch.tensor([j for j in range(p + 1) if window == 0 or j > p - window or j < keep])
        s = torch.einsum("jhd,hd->hj", case["ks"][t][seen].double(), case["q"][t, :H * hd].double().view(H, hd)) * scale
        if scores == "worked on":
            s = cap * torch.tanh(s / cap) + table[(p - seen).clamp(max=len(table) - 1)].double().t()
            s = torch.cat([s, sinks.double()[:, None]], dim=1)
        w = torch.softmax(s, dim=1)[:, :len(seen)]
        want[t] = torch.einsum("hj,jhd->hd", w, case["vs"][t][seen].double()).flatten()
    dev = lambda x: None if x is None else x.to(DEV)  # noqa: E731
    out = torch.zeros(case["n"], H * hd, dtype=dtype, device=DEV)
    ops.attention_decode(out, dev(case["q"])[:, :H * hd], dev(case["kc"]), dev(case["vc"]), dev(case["bt"]), torch.arange(case["n"], dtype=torch.int32, device=DEV),
                         torch.tensor(case["tok_pos"], dtype=torch.int32, device=DEV), n_head=H, scale=scale, window=window, waves=waves, rows_are_requests=True,
                         keep_first=keep, softcap=cap, bias_table=dev(table), sinks=dev(sinks))
    close(out, want, 8e-3 if dtype == torch.bfloat16 else 3e-6, scores)


@pytest.mark.parametrize("window", [0, 37, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case_id", range(len(ATT_CASES)))
def test_attention_splits_by_position(ops, case_id, dtype, window):
    """Splits of a fixed number of keys from a token's first key on: right against the plain
    formula, and the same bits whether the step has just the splits the longest context needs or
    more (a longer context beside it), the later ones empty; a context within one split has the
    bits of the unsplit call."""
    ctx_lens, q_lens, H, Hkv, hd, page = ATT_CASES[case_id]
    case = paged_case(len(ctx_lens), ctx_lens, q_lens, H, Hkv, hd, page, dtype, seed=case_id)
    scale = 0.7 / math.sqrt(hd)
    dev = lambda x: x.to(DEV)  # noqa: E731
    q, kc, vc, bt = dev(case["q"]), dev(case["kc"]), dev(case["vc"]), dev(case["bt"])
    tok_seq = torch.tensor(case["tok_seq"], dtype=torch.int32, device=DEV)
    tok_pos = torch.tensor(case["tok_pos"], dtype=torch.int32, device=DEV)
    chunk = 64
    longest = max(ctx_lens) if window == 0 else min(max(ctx_lens), window)
    need = -(-longest // chunk)
    outs = []
    for splits in (need, need + 1, 2 * need + 3):
        out = torch.zeros(case["n"], H * hd, dtype=dtype, device=DEV)
        partials = torch.full((case["n"] * H * splits * (hd + 4),), float("nan"), device=DEV) if splits > 1 else None
        ops.attention_decode(out, q[:, :H * hd], kc, vc, bt, tok_seq, tok_pos, n_head=H, scale=scale, window=window,
                             n_splits=splits, partials=partials, waves=4, chunk=chunk)
        assert torch.isfinite(out.float()).all()
        outs.append(out)
    close(outs[0], attention_reference(case, H, Hkv, hd, scale, window), 8e-3 if dtype == torch.bfloat16 else 2e-6, "splits by position")
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    # launched as one split, a workgroup walking its token's splits in turn: the same bits again
    if need <= 16:
        out = torch.zeros(case["n"], H * hd, dtype=dtype, device=DEV)
        ops.attention_decode(out, q[:, :H * hd], kc, vc, bt, tok_seq, tok_pos, n_head=H, scale=scale, window=window,
                             n_splits=1, waves=4, chunk=chunk)
        assert torch.equal(out, outs[0]), "one workgroup walking the splits"
    # each request alone, with the splits its own context needs
    for s_, n_ctx in enumerate(ctx_lens):
        rows = [t for t, r in enumerate(case["tok_seq"]) if r == s_]
        own = -(-(n_ctx if window == 0 else min(n_ctx, window)) // chunk)
        out = torch.zeros(case["n"], H * hd, dtype=dtype, device=DEV)
        partials = torch.empty(len(rows) * H * own * (hd + 4), device=DEV) if own > 1 else None
        ops.attention_decode(out, q[:, :H * hd], kc, vc, bt, tok_seq, tok_pos, n_head=H, scale=scale, window=window,
                             n_splits=own, partials=partials, waves=4, chunk=chunk,
                             tok_list=torch.tensor(rows, dtype=torch.int32, device=DEV), n_tokens=len(rows))
        assert torch.equal(out[rows], outs[0][rows]), f"request {s_} alone"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_attention_order_of_the_grid(ops, dtype):
    """The grid runs along the heads or along the tokens first, by what a prompt's heads bring to an XCD's L2 (the width of the
    block table stands for the keys: five heads of 64 on either side of 4 MB) and by the number of single-token requests (16
    and 17): the same bits, and right against the plain formula."""
    H, hd, page = 5, 64, 16
    scale = 0.7 / math.sqrt(hd)
    case = paged_case(2, [300, 33], [40, 33], H, H, hd, page, dtype, seed=3)
    bt = case["bt"]
    outs = []
    for columns, reach in ((102, 0), (103, 0), (103, 512)):
        columns = columns * 4 // dtype.itemsize  # 4,177,920 bytes of keys and values, 4,218,880
        case["bt"] = torch.cat([bt, bt.new_zeros(bt.shape[0], columns - bt.shape[1])], dim=1)
        dev = [case[k].to(DEV) for k in ("q", "kc", "vc", "bt")] + [torch.tensor(case[k], dtype=torch.int32, device=DEV) for k in ("tok_seq", "tok_pos")]
        out = torch.zeros(case["n"], H * hd, dtype=dtype, device=DEV)
        ops.attention_decode(out, dev[0][:, :H * hd], *dev[1:], n_head=H, scale=scale, n_splits=1, waves=4, chunk=256, reach=reach)
        outs.append(out)
    close(outs[0], attention_reference(case, H, H, hd, scale), 8e-3 if dtype == torch.bfloat16 else 2e-6, "grid order")
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    case = paged_case(17, list(range(20, 20 + 17 * 9, 9)), [1] * 17, H, H, hd, page, dtype, seed=4)
    dev = [case[k].to(DEV) for k in ("q", "kc", "vc", "bt")] + [torch.tensor(case[k], dtype=torch.int32, device=DEV) for k in ("tok_seq", "tok_pos")]
    for splits in (1, 3):
        outs = []
        for n in (17, 16):
            out = torch.zeros(n, H * hd, dtype=dtype, device=DEV)
            partials = torch.empty(n * H * splits * (hd + 4), device=DEV) if splits > 1 else None
            ops.attention_decode(out, dev[0][:n, :H * hd], *dev[1:4], dev[4][:n], dev[5][:n], n_head=H, scale=scale, n_splits=splits, partials=partials,
                                 waves=4, rows_are_requests=True)
            outs.append(out)
        close(outs[0], attention_reference(case, H, H, hd, scale), 8e-3 if dtype == torch.bfloat16 else 2e-6, "single tokens")
        assert torch.equal(outs[0][:16], outs[1])


@pytest.mark.parametrize("waves", [4, 16])
@pytest.mark.parametrize("window", [0, 37])
@pytest.mark.parametrize("splits", [2, 4, 7, 8])
@pytest.mark.parametrize("case_id", [0, 1, 2, 3, 5, 6, 7, 8, 9])
def test_attention_splits_merged_by_the_projection(ops, case_id, splits, window, waves):
    """Attention that leaves each (token, head) pair's keys in splits, and the projection cut
    over its inner dimension that merges them as it loads them: the planes add up to rows +
    attention . W^T + bias; the merge kernel gives attention's output from the same splits.
    Contexts shorter than the number of splits leave splits empty."""
    ctx_lens, q_lens, H, Hkv, hd, page = ATT_CASES[case_id]
    case = paged_case(len(ctx_lens), ctx_lens, q_lens, H, Hkv, hd, page, torch.bfloat16, seed=case_id)
    scale = 0.7 / math.sqrt(hd)
    n = case["n"]
    dev = lambda x: x.to(DEV)  # noqa: E731
    q, kc, vc, bt = dev(case["q"]), dev(case["kc"]), dev(case["vc"]), dev(case["bt"])
    tok_seq = torch.tensor(case["tok_seq"], dtype=torch.int32, device=DEV)
    tok_pos = torch.tensor(case["tok_pos"], dtype=torch.int32, device=DEV)
    partials = torch.full((n, H, splits, hd + 4), float("nan"), device=DEV)
    untouched = torch.full((n, H * hd), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.attention_decode(untouched, q[:, :H * hd], kc, vc, bt, tok_seq, tok_pos, n_head=H, scale=scale, window=window,
                         n_splits=splits, partials=partials, waves=waves, leave_splits=True)
    assert (untouched == 7.0).all()
    want = attention_reference(case, H, Hkv, hd, scale, window)
    merged = torch.empty(n, H * hd, dtype=torch.bfloat16, device=DEV)
    ops.attention_merge(merged, partials)
    close(merged, want, 8e-3, "merged splits")
    N, K = 72, H * hd
    w, bias = rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    for parts in (1, 2, 3):
        if (parts - 1) * (((K + 63) // 64 + parts - 1) // parts) >= (K + 63) // 64:
            continue
        for n_base in (None, 0, 2):
            base = None if n_base is None else (rnd(n, N, seed=8, scale=3.0) if n_base == 0 else rnd(n_base, n, N, seed=9, scale=3.0))
            planes = torch.full((parts, n, N), float("nan"), device=DEV)
            if n > 32:
                with pytest.raises(Exception, match="outside"):
                    ops.gemm_att_parts(partials, w, planes, bias=bias if base is not None else None, base=base)
                continue
            ops.gemm_att_parts(partials, w, planes, bias=bias if base is not None else None, base=base)
            total = merged.double() @ w.double().t()
            if base is not None:
                total = total + bias.double() + (base.double() if n_base == 0 else base.double().sum(0))
            close(planes.double().sum(0), total, 1e-5, f"projection over splits, {parts} parts, base {n_base}")
            # the same bits as the plain cut product over the merged rows
            two = torch.empty_like(planes)
            ops.gemm_skinny_parts(merged, w, two, bias=bias if base is not None else None, base=base, ksplit=8)
            assert torch.equal(planes, two)


def test_projection_over_splits_with_rows_32_kb_apart(ops):
    """Heads x head size = 16,384: the weights' rows lie 32 KB apart, where the streaming kernels
    walk K in blocks from a place of each workgroup's own; the kernel that merges attention's
    splits as it loads them must still give the bits of the merge followed by the plain product."""
    M, H, S, hd, N = 3, 128, 2, 128, 40
    g = torch.Generator().manual_seed(3)
    partials = torch.randn(M, H, S, hd + 4, generator=g)
    partials[..., hd] = torch.randn(M, H, S, generator=g) * 2  # the splits' maxima
    partials[..., hd + 1] = torch.rand(M, H, S, generator=g) * 50 + 1  # and sums
    partials = partials.to(DEV)
    merged = torch.empty(M, H * hd, dtype=torch.bfloat16, device=DEV)
    ops.attention_merge(merged, partials)
    w, bias = rnd(N, H * hd, seed=1, scale=0.05, dtype=torch.bfloat16), rnd(N, seed=2)
    base = rnd(M, N, seed=8, scale=3.0)
    with pytest.raises(Exception, match="do not fit LDS"):  # whole rows of 16,384 are refused, not mangled
        ops.gemm_att_parts(partials, w, torch.empty(1, M, N, device=DEV), bias=bias, base=base)
    for parts in (2, 4):
        planes = torch.full((parts, M, N), float("nan"), device=DEV)
        ops.gemm_att_parts(partials, w, planes, bias=bias, base=base)
        want = merged.double() @ w.double().t() + bias.double() + base.double()
        close(planes.double().sum(0), want, 1e-5, f"projection over splits at K = 16,384, {parts} parts")
        two = torch.empty_like(planes)
        ops.gemm_skinny_parts(merged, w, two, bias=bias, base=base, ksplit=8)
        assert torch.equal(planes, two)


PREFILL_CASES = [
    # ctx_lens, q_lens, H, Hkv, hd, page
    ([1, 17, 300], [1, 17, 300], 4, 4, 16, 16),
    ([40, 129, 5], [7, 100, 5], 3, 3, 32, 16),
    ([700, 64], [130, 64], 5, 5, 64, 64),
    ([33, 257], [20, 129], 6, 2, 48, 8),
    ([300], [300], 2, 1, 128, 16),
    ([90, 31], [31, 9], 2, 2, 80, 16),
    ([1024], [1024], 1, 1, 64, 16),
    # pages that are no power of two
    ([130, 24, 49], [100, 24, 40], 3, 3, 32, 24),
    ([400, 97], [200, 97], 4, 2, 64, 48),
]


@pytest.mark.parametrize("tile,ksplit", [(64, 1), (64, 2), (64, 4), (128, 1), (128, 2)])
@pytest.mark.parametrize("window", [0, 37, 200])
@pytest.mark.parametrize("case_id", range(len(PREFILL_CASES)))
def test_attention_prefill(ops, case_id, window, tile, ksplit):
    ctx_lens, q_lens, H, Hkv, hd, page = PREFILL_CASES[case_id]
    if ksplit == 4 and hd > 64:
        pytest.skip("4 waves a query group are taken up to head size 64")
    case = paged_case(len(ctx_lens), ctx_lens, q_lens, H, Hkv, hd, page, torch.bfloat16, seed=case_id)
    scale = 0.7 / math.sqrt(hd)
    out = run_attention(ops, case, H, hd, scale, window, "prefill", splits=tile, ksplit=ksplit)
    assert torch.isfinite(out.float()).all()
    close(out, attention_reference(case, H, Hkv, hd, scale, window), 8e-3, "prefill")


@pytest.mark.parametrize("tile,ksplit", [(64, 1), (64, 2), (64, 4), (128, 1), (128, 2)])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("window,keep", [(0, 0), (100, 0), (100, 20), (70, 130)])
def test_attention_prefill_by_page_size(ops, window, keep, hd, tile, ksplit):
    """Contexts that end at and beside the blocks of 64 keys, in pages that a load of keys never crosses (8, 128), that it does (4), and
    of no power of two (24): the formula, and the same bits from each. What lies between the kept positions and every query's window is
    given back (no page, or NaN), and must not be read."""
    if ksplit == 4 and hd > 64:
        pytest.skip("4 waves a query group are taken up to head size 64")
    ctx_lens, q_lens, H, Hkv, scale = [63, 128, 193, 300], [63, 65, 1, 131], 2, 1, 0.7 / math.sqrt(hd)
    outs = []
    for page in (8, 4, 24, 128):
        case = paged_case(4, ctx_lens, q_lens, H, Hkv, hd, page, torch.bfloat16, seed=5, shuffle=False)  # (the same values whatever the pages)
        case["bt"] = torch.where(case["bt"] >= 0, case["kc"].shape[0] - 1 - case["bt"], case["bt"])
        case["kc"], case["vc"] = case["kc"].flip(0), case["vc"].flip(0)
        row, work, want = 0, [], torch.zeros(case["n"], H * hd, dtype=torch.float64)
        for s, (c, n) in enumerate(zip(ctx_lens, q_lens)):
            for t0 in range(0, n, tile):
                work += [s, row + t0, c - n + t0, min(tile, n - t0)]
            for t in range(row, row + n):
                p = case["tok_pos"][t]
                seen = [j for j in range(p + 1) if window == 0 or j > p - window or j < keep]
                for h in range(H):
                    w = torch.softmax(case["ks"][s][seen, 0].double() @ case["q"][t, h * hd:(h + 1) * hd].double() * scale, dim=0)
                    want[t, h * hd:(h + 1) * hd] = w @ case["vs"][s][seen, 0].double()
            for j in range(keep, c - n - window + 1 if window else 0):  # no query sees position j
                pg = int(case["bt"][s, j // page])
                case["kc"][pg, :, j % page], case["vc"][pg, :, j % page] = float("nan"), float("nan")
            row += n
        out = torch.zeros(case["n"], H * hd, dtype=torch.bfloat16, device=DEV)
        kw = {k: case[k].to(DEV) for k in ("kc", "vc", "bt")}
        ops.attention_prefill(out, case["q"].to(DEV)[:, :H * hd], kw["kc"], kw["vc"], kw["bt"], torch.tensor(work, dtype=torch.int32, device=DEV),
                              len(work) // 4, n_head=H, scale=scale, window=window, tile=tile, ksplit=ksplit, keep_first=keep)
        close(out, want, 8e-3, f"pages of {page}")
        outs.append(out)
    assert all(torch.equal(outs[0], o) for o in outs[1:])


@pytest.mark.parametrize("tile,ksplit", [(64, 1), (64, 2), (64, 4), (128, 1), (128, 2)])
@pytest.mark.parametrize("hd,padded", [(48, 64), (112, 128)])
@pytest.mark.parametrize("scores", ["plain", "window", "kept", "worked on"])
def test_attention_prefill_of_padded_heads_has_the_same_bits(ops, scores, hd, padded, tile, ksplit):
    """Heads of 48 and of 112 run in the kernel that keeps its keys in registers; with zeros behind them, as heads of 64 and of 128, in the one that takes them
    straight into LDS. The sums are in one order, and the zeros add nothing."""
    if ksplit == 4 and hd > 64:
        pytest.skip("4 waves a query group are taken up to head size 64")
    ctx_lens, q_lens, H, Hkv, scale = [63, 129, 300, 520], [63, 65, 131, 301], 4, 2, 0.7 / math.sqrt(hd)
    kw = dict(window=100) if scores == "window" else dict(window=100, keep_first=20) if scores == "kept" else {}
    if scores == "worked on":
        kw = dict(softcap=2.0, bias_table=rnd(65, H, seed=1), sinks=rnd(H, seed=2))
    for page in (16, 24, 4):
        case = paged_case(4, ctx_lens, q_lens, H, Hkv, hd, page, torch.bfloat16, seed=5)
        row, work = 0, []
        for s, (c, n) in enumerate(zip(ctx_lens, q_lens)):
            for t0 in range(0, n, tile):
                work += [s, row + t0, c - n + t0, min(tile, n - t0)]
            row += n
        outs = []
        for d in (hd, padded):
            wider = lambda x: torch.nn.functional.pad(x, (0, d - hd)).contiguous().to(DEV)  # noqa: E731
            out = torch.zeros(case["n"], H * d, dtype=torch.bfloat16, device=DEV)
            ops.attention_prefill(out, wider(case["q"][:, :H * hd].reshape(-1, H, hd)).view(-1, H * d), wider(case["kc"]), wider(case["vc"]), case["bt"].to(DEV),
                                  torch.tensor(work, dtype=torch.int32, device=DEV), len(work) // 4, n_head=H, scale=scale, tile=tile, ksplit=ksplit, **kw)
            outs.append(out.view(-1, H, d)[:, :, :hd])
        assert torch.isfinite(outs[0].float()).all() and torch.equal(outs[0], outs[1]), f"pages of {page}"


@pytest.mark.parametrize("K", [64, 192, 832, 72])
@pytest.mark.parametrize("N", [33, 64, 72, 200])
@pytest.mark.parametrize("form", ["one", "relu2", "two", "clamped", "heads", "gated heads"])
def test_products_of_listed_rows_and_heads(ops, form, N, K):
    """Tiles of 64 places with one, some and all of them taken, one in the middle that nobody uses and some at the end; features that fill no
    tile; K of one stage, of three, of a wide tile's 13, and of no whole stage. Against 32-bit sums of the same bfloat16 operands: the results'
    rounding to bfloat16 (2^-9) and a sum's order."""
    E, n = 3, 150
    if "heads" in form:
        a, w = rnd(n, E * K, dtype=torch.bfloat16), rnd(E, N, K, seed=1, scale=0.2, dtype=torch.bfloat16)
        gate = rnd(n, E * N + 3, seed=2)[:, :E * N] if form == "gated heads" else None
        out = torch.full((n, E * N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.heads_product(out, a, w, gate)
        want = torch.cat([a[:, h * K:(h + 1) * K].float() @ w[h].float().t() for h in range(E)], dim=1)
        close(out, want * torch.sigmoid(gate) if gate is not None else want, 4e-3, form)
        return
    a = rnd(n, K, dtype=torch.bfloat16)
    w0, w1 = rnd(E, N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(E, N, K, seed=2, scale=0.2, dtype=torch.bfloat16)
    expert = torch.tensor([0] * 65 + [1] * 1 + [2] * (2 * n - 66))
    expert = expert[torch.randperm(2 * n, generator=torch.Generator().manual_seed(3))]
    tiles = ops.moe_tiles(2 * n, E, 64)
    rows, group, at = torch.full((tiles, 64), -1, dtype=torch.int32), torch.full((tiles,), -1, dtype=torch.int32), 0
    for e in range(E):
        mine = (expert == e).nonzero().flatten().int()
        for c in mine.split(64):
            rows[at, :len(c)], group[at], at = c, e, at + 1
        at += 1 if e == 0 and at + 1 + -(-int((expert > 0).sum()) // 64) < tiles else 0  # a tile nobody uses
    scale = rnd(2 * n, seed=4)
    two, clamp = form in ("two", "clamped"), (1.5, 1.7, 1.0) if form == "clamped" else None
    x = a.float().repeat_interleave(2, 0)
    u, v = (torch.stack([x[i] @ w[e].float().t() for i, e in enumerate(expert.tolist())]) for w in (w0, w1))
    if form == "clamped":
        g = u.clamp(max=1.5)
        want = g * torch.sigmoid(1.7 * g) * (v.clamp(-1.5, 1.5) + 1.0)
    else:
        want = u * torch.sigmoid(u) * v if two else torch.relu(u) ** 2 if form == "relu2" else u
    for dtype, tol in ((torch.bfloat16, 4e-3), (torch.float32, 1e-5)):
        out = torch.full((2 * n, N), float("nan"), dtype=dtype, device=DEV)
        ops.moe_product(out, a, w0, w1 if two else None, rows.to(DEV).flatten(), group.to(DEV), a_div=2, row_scale=scale, act="relu2" if form == "relu2" else "none", clamp=clamp)
        close(out, want * scale[:, None], tol, form)


@pytest.mark.parametrize("K,N", [(64, 130), (192, 200), (832, 200), (832, 70)])
@pytest.mark.parametrize("form", ["one", "two", "heads"])
@pytest.mark.parametrize("E", [3, 400])
def test_products_of_long_lists(ops, form, E, N, K):
    """Lists and heads of many tiles, whose XCDs take stretches of several tiles, the last one shorter: with a hole inside a stretch, and with more spare tiles
    at the end than a workgroup looks at. Bounds as above."""
    n, H = 550 if E == 3 else 1100, 3
    if form == "heads":
        a, w = rnd(n, H * K, dtype=torch.bfloat16), rnd(H, N, K, seed=1, scale=0.2, dtype=torch.bfloat16)
        out = torch.full((n, H * N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.heads_product(out, a, w, None)
        close(out, torch.cat([a[:, h * K:(h + 1) * K].float() @ w[h].float().t() for h in range(H)], dim=1), 4e-3, form)
        return
    a = rnd(n, K, dtype=torch.bfloat16)
    w0, w1 = rnd(E, N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(E, N, K, seed=2, scale=0.2, dtype=torch.bfloat16)
    expert = torch.randint(0, 3, (2 * n,), generator=torch.Generator().manual_seed(3)) * (E // 3)
    tiles = ops.moe_tiles(2 * n, E, 64)
    rows, group, at = torch.full((tiles, 64), -1, dtype=torch.int32), torch.full((tiles,), -1, dtype=torch.int32), 0
    for e in sorted(set(expert.tolist())):
        for c in (expert == e).nonzero().flatten().int().split(64):
            at += at == 4  # a tile nobody uses
            rows[at, :len(c)], group[at], at = c, e, at + 1
    scale = rnd(2 * n, seed=4)
    x, want = a.float().repeat_interleave(2, 0), torch.empty(2 * n, N, device=DEV)
    for e in sorted(set(expert.tolist())):
        mine = (expert == e).nonzero().flatten().to(DEV)
        u, v = x[mine] @ w0[e].float().t(), x[mine] @ w1[e].float().t()
        want[mine] = u * torch.sigmoid(u) * v if form == "two" else u
    out = torch.full((2 * n, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_product(out, a, w0, w1 if form == "two" else None, rows.to(DEV).flatten(), group.to(DEV), a_div=2, row_scale=scale)
    close(out, want * scale[:, None], 4e-3, form)


def test_products_of_more_tiles_than_a_grid_dimension_holds(ops):
    """17 million tiles of places and features, all but one column of them spare."""
    n, tiles, N, K = 4, 1100, 1_000_000, 64
    a, w = rnd(n, K, dtype=torch.bfloat16), rnd(1, N, K, seed=1, dtype=torch.bfloat16)
    rows, group = torch.full((tiles * 64,), -1, dtype=torch.int32), torch.full((tiles,), -1, dtype=torch.int32)
    rows[:n], group[0] = torch.arange(n), 0
    out = torch.full((n, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.moe_product(out, a, w, None, rows.to(DEV), group.to(DEV))
    close(out, a.float() @ w[0].float().t(), 4e-3, "spare tiles")


def reference_from_pages(case, kc, vc, bt, H, Hkv, hd, page, scale, window=0):
    """The plain formula over whatever pages a block table names (float64)."""
    out = torch.zeros(case["n"], H * hd, dtype=torch.float64)
    for t, (s, p) in enumerate(zip(case["tok_seq"], case["tok_pos"])):
        first = max(0, p - window + 1) if window > 0 else 0
        pos = torch.arange(first, p + 1)
        pages, offs = bt[s, pos // page].long(), pos % page
        for h in range(H):
            hk = h // (H // Hkv)
            k, v = kc[pages, hk, offs].double(), vc[pages, hk, offs].double()
            w = torch.softmax((k @ case["q"][t, h * hd:(h + 1) * hd].double()) * scale, dim=0)
            out[t, h * hd:(h + 1) * hd] = w @ v
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kernel", ["generic", "decode", "decode in splits", "prefill"])
def test_a_page_id_past_the_counted_pages_is_not_followed(ops, kernel, dtype):
    """The caches hold eight pages more than the launcher is told of, and block tables name ids
    in that slack (and a -1 in a place that is read): told the count, a kernel reads the last
    counted page instead; told of all pages it reads the slack page. Either way every fetch
    stays inside the caches: an id that a table should never hold costs a wrong number, not
    the machine."""
    if kernel == "prefill" and dtype != torch.bfloat16:
        pytest.skip("the tiled kernel is bfloat16 only")
    ctx_lens, q_lens, H, Hkv, hd, page = ([300, 70], [9, 40], 4, 2, 64, 16) if kernel == "prefill" else ([300, 70], [3, 1], 4, 2, 64, 16)
    case = paged_case(len(ctx_lens), ctx_lens, q_lens, H, Hkv, hd, page, dtype, seed=11)
    counted = case["kc"].shape[0]
    g = torch.Generator().manual_seed(5)
    kc = torch.cat([torch.nan_to_num(case["kc"].float(), nan=0.5), torch.randn(8, Hkv, page, hd, generator=g)]).to(dtype)
    vc = torch.cat([torch.nan_to_num(case["vc"].float(), nan=-0.5), torch.randn(8, Hkv, page, hd, generator=g)]).to(dtype)
    bt = case["bt"].clone()
    bt[0, 2], bt[0, 7], bt[1, 1] = counted + 3, counted + 7, -1
    case = dict(case, kc=kc, vc=vc, bt=bt)
    scale = 0.7 / math.sqrt(hd)
    tol = 8e-3 if dtype == torch.bfloat16 else 2e-6

    def run(num_pages):
        dev = lambda x: x.to(DEV)  # noqa: E731
        q = dev(case["q"])[:, :H * hd]
        tok_seq = torch.tensor(case["tok_seq"], dtype=torch.int32, device=DEV)
        tok_pos = torch.tensor(case["tok_pos"], dtype=torch.int32, device=DEV)
        out = torch.zeros(case["n"], H * hd, dtype=dtype, device=DEV)
        kw = dict(n_head=H, scale=scale, num_pages=num_pages)
        if kernel == "generic":
            ops.attention_generic(out, q, dev(kc), dev(vc), dev(bt), tok_seq, tok_pos, **kw)
        elif kernel == "prefill":
            work = torch.tensor([0, 0, ctx_lens[0] - q_lens[0], q_lens[0], 1, q_lens[0], ctx_lens[1] - q_lens[1], q_lens[1]],
                                dtype=torch.int32, device=DEV)
            ops.attention_prefill(out, q, dev(kc), dev(vc), dev(bt), work, 2, tile=64, **kw)
        else:
            splits = 3 if kernel == "decode in splits" else 1
            partials = torch.empty(case["n"] * H * splits * (hd + 4), device=DEV) if splits > 1 else None
            ops.attention_decode(out, q, dev(kc), dev(vc), dev(bt), tok_seq, tok_pos, n_splits=splits, partials=partials, **kw)
        assert torch.isfinite(out.float()).all()
        return out

    told = run(counted)
    close(told, reference_from_pages(case, kc, vc, bt.clamp(0, counted - 1), H, Hkv, hd, page, scale), tol, "ids brought into the counted pages")
    whole = run(None)
    close(whole, reference_from_pages(case, kc, vc, bt.clamp(0, counted + 7), H, Hkv, hd, page, scale), tol, "every page counted")
    assert not torch.equal(told, whole)
    with pytest.raises(Exception, match="pages"):
        run(counted + 9)


@pytest.mark.parametrize("kernel", ["kv_write", "skinny", "dl", "dl6", "dl7", "dl9", "dl11", "dl15", "mfma", "folded norm"])
def test_a_slot_past_the_counted_pages_is_not_written(ops, kernel):
    """Slots in the eight pages the launcher is not told of (and a -1) are skipped; told of all
    pages, the same call writes them."""
    M, H, Hkv, hd, K, page = 24, 3, 3, 32, 128, 8
    q_dim, kv_dim = H * hd, Hkv * hd
    N = q_dim + 2 * kv_dim
    counted = 6
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    slots = torch.randperm(counted * page)[:M].to(torch.int32)
    slots[3], slots[10], slots[17] = counted * page, (counted + 8) * page - 1, -1
    slots = slots.to(DEV)

    def run(num_pages):
        kc = torch.zeros(counted + 8, Hkv, page, hd, dtype=torch.bfloat16, device=DEV)
        vc = torch.zeros_like(kc)
        q = torch.zeros(M, q_dim, dtype=torch.bfloat16, device=DEV)
        kw = dict(out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, q_dim, num_pages))
        if kernel == "kv_write":
            full = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
            ops.gemm_simple(a, w, bias, out=full)
            ops.kv_write(kc, vc, full, q_dim, q_dim + kv_dim, slots, num_pages=num_pages)
        elif kernel == "skinny":
            ops.gemm_skinny(a, w, bias, **kw)
        elif kernel.startswith("dl"):
            ops.gemm_mfma_dl(a, w, bias, tile=int(kernel[2:] or 2), **kw)
        elif kernel == "mfma":
            ops.gemm_mfma(a, w, bias, tile=2, **kw)
        else:
            x = rnd(M, K, scale=2.0, seed=4)
            ops.gemm_skinny_ln(x, rnd(K, seed=5) + 1.0, rnd(K, seed=6), 1e-5, w, bias, **kw)
        return kc, vc

    for num_pages, written in ((counted, M - 3), (None, M - 1)):
        kc, vc = run(num_pages)
        for c in (kc, vc):
            assert (c[:counted] != 0).any(dim=(1, 3)).sum().item() == M - 3  # the tokens with a slot in the counted pages
            assert (c != 0).any(dim=(1, 3)).sum().item() == written


@pytest.mark.parametrize("T,targets", [(700, [0, 15, 16, 31, 32, 255, 256, 511, 559, 560, 561, 600, 640, 687, 698, 699]),
                                       (5000, [0, 17, 1023, 1024, 2047, 2048, 3000, 4095, 4096, 4097, 4859, 4860, 4900, 4959, 4998, 4999])])
def test_attention_prefill_finds_one_far_key(ops, T, targets):
    """A portion's queries each with one outstanding key, at page and block edges; in a context of
    700 positions and in one of 5,000 (313 pages)."""
    H = Hkv = 2
    hd, page, nq = 64, 16, 140
    case = paged_case(1, [T], [nq], H, Hkv, hd, page, torch.bfloat16, seed=3)
    k = case["ks"][0]
    for n, target in enumerate(targets):
        row = nq - 1 - n * 3  # the query at position T - 1 - 3 n looks for `target` if it may see it
        qpos = T - nq + row
        if target > qpos:
            continue
        qv = case["q"][row, :hd].float()
        # orthogonalise against earlier planted keys is not needed: random 64-vectors are nearly orthogonal
        k[target, 0] = (qv * 4).to(torch.bfloat16)
        lp, off = divmod(target, page)
        case["kc"][case["bt"][0, lp], 0, off] = k[target, 0]
    out = run_attention(ops, case, H, hd, 1.0, 0, "prefill")
    ref = attention_reference(case, H, Hkv, hd, 1.0, 0)
    close(out, ref, 8e-3, "prefill far keys")


@pytest.mark.parametrize("T,targets", [(700, (0, 15, 16, 17, 255, 256, 511, 512, 687, 688, 698, 699)),
                                       (5000, (0, 255, 256, 2047, 2048, 4095, 4096, 4863, 4864, 4998, 4999))])
@pytest.mark.parametrize("kernel", ["generic", "decode", "decode by position", "decode walking its splits"])
def test_attention_finds_one_far_key(ops, kernel, T, targets):
    """Random values average a wrong key away; here one key's score stands out, at a page's
    first and last slot, in the first page and the last, at the edges of splits, and the output
    must be its value row; in a context of 700 positions and in one of 5,000."""
    H = Hkv = 2
    hd, page = 64, 16
    if kernel == "decode walking its splits" and T > 16 * 256:
        pytest.skip("one workgroup walks at most 16 splits")
    for target in targets:
        case = paged_case(1, [T], [1], H, Hkv, hd, page, torch.bfloat16, seed=target)
        qv = case["q"][0, :hd].float()
        k = case["ks"][0]
        k[target, 0] = (qv * 4).to(torch.bfloat16)  # head 0: score ~ 4 |q|^2 ~ 250, all others ~ N(0, 8)
        lp, off = divmod(target, page)
        case["kc"][case["bt"][0, lp], 0, off] = k[target, 0]
        if kernel.startswith("decode "):
            dev = lambda x: x.to(DEV)  # noqa: E731
            splits = -(-T // 256) if kernel == "decode by position" else 1
            out = torch.zeros(1, H * hd, dtype=torch.bfloat16, device=DEV)
            ops.attention_decode(out, dev(case["q"])[:, :H * hd], dev(case["kc"]), dev(case["vc"]), dev(case["bt"]),
                                 torch.zeros(1, dtype=torch.int32, device=DEV), torch.tensor([T - 1], dtype=torch.int32, device=DEV),
                                 n_head=H, scale=1.0, n_splits=splits, waves=4, chunk=256,
                                 partials=torch.empty(H * splits * (hd + 4), device=DEV) if splits > 1 else None)
        else:
            out = run_attention(ops, case, H, hd, 1.0, 0, kernel, splits=(3 if T < 1000 else 11) if kernel == "decode" else 1)
        want = case["vs"][0][target, 0].float()
        assert torch.allclose(out[0, :hd].float().cpu(), want, atol=2e-2), f"{kernel}: key {target} was not found"


# ---------------------------------------------------------------------------
# sampling
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("rows,V", [(1, 50257), (9, 1000), (64, 777), (3, 5)])
def test_argmax_ties_go_to_the_lowest_id(ops, rows, V):
    logits = rnd(rows, V + 3)[:, :V]  # strided rows
    logits[:, V // 2] = 50.0
    logits[:, V - 1] = 50.0  # a tie: the lower id wins
    if rows > 1:
        logits[1, 0] = 50.0
    out = torch.empty(rows, dtype=torch.int32, device=DEV)
    ops.argmax(out, logits)
    want = [V // 2] * rows
    if rows > 1:
        want[1] = 0
    assert out.tolist() == want
    ops.argmax(out, rnd(rows, V, seed=4))
    assert out.tolist() == rnd(rows, V, seed=4).argmax(dim=1).tolist()


@pytest.mark.parametrize("V", [1000, 50257, 53250, 60000, 70001])
def test_sampler_against_the_plain_sampler(ops, V):
    """Temperature, top-k and top-p per row against the plain implementation's rules, at
    vocabularies that take each of the sampling kernels (the row in registers with a one-wave
    finish for top-k <= 64, the same with many candidates, and the general kernel)."""
    import plain_gpt2 as plain

    logits = rnd(14, V, scale=2.0, seed=11)
    logits[5, 100:140] = 3.0  # many ties at the top-k boundary
    logits[12, :] = 0.25  # all equal: ties everywhere
    logits[3, 7:60:2] = 9.0  # ties above the top-k boundary: all kept
    logits[4, 10:50] = 8.0  # ties at the top: the 5 of the lowest ids are kept
    logits[13, 300:900] = 7.5  # more ties at the boundary than keys the one-wave pool would hold at the large vocabularies
    params = [(0.0, 0, 1.0), (1.0, 0, 1.0), (0.8, 0, 1.0), (0.8, 40, 0.95), (1.3, 5, 1.0), (0.7, 20, 1.0), (1.0, 0, 0.5),
              (1.0, 0, 0.05), (0.5, 1, 1.0), (2.0, 999, 0.9), (1.0, 40, 0.0), (0.8, 0, 0.999), (1.0, 64, 0.7), (0.9, 65, 0.9)]
    cpu = logits.cpu().numpy()
    for trial in range(6):
        u = [plain.uniform(7 + trial, r) for r in range(len(params))]
        out = torch.empty(len(params), dtype=torch.int32, device=DEV)
        ops.sample(out, logits,
                   torch.tensor([p[0] for p in params], dtype=torch.float32, device=DEV),
                   torch.tensor([p[1] for p in params], dtype=torch.int32, device=DEV),
                   torch.tensor([p[2] for p in params], dtype=torch.float32, device=DEV),
                   torch.tensor(u, dtype=torch.float64, device=DEV))
        got = out.tolist()
        for r, (T, k, p) in enumerate(params):
            probs = plain.probabilities(cpu[r], T, k, p)
            want = plain.sample(probs, u[r])
            if got[r] != want:
                cdf = np.cumsum(probs)
                assert probs[got[r]] > 0 and np.abs(cdf - u[r]).min() < 1e-5, (V, r, params[r], got[r], want)


@pytest.mark.parametrize("V", [3000, 50257, 53250, 65533])
def test_top_p_over_many_candidates_keeps_exactly_the_nucleus(ops, V):
    """Top-p alone (and with a top-k too wide for one wave) at rows made so that a wrong cut shows
    in the draws: a few heavy ids over a light floor, the cut falling between them, inside a run
    of ties (the lowest ids of the run are kept), on the top-k boundary's ties, in a flat row where
    every key shares a bin, and in a peaked row whose masses span every bin. 48 draws a row are
    compared with the plain sampler's; a draw may differ only where the uniform number lies
    within rounding of a boundary between two ids."""
    import plain_gpt2 as plain

    g = torch.Generator().manual_seed(V)
    cases = []  # (logits row, temperature, top_k, top_p)
    floor = torch.randn(V, generator=g) * 0.5 - 12.0
    heavy = floor.clone()
    heavy[[5, 900, 1777, 2500, 40, 41]] = torch.tensor([3.0, 2.9, 2.5, 2.45, 1.0, 0.9])
    for p in (0.2, 0.4, 0.63, 0.8, 0.97, 0.99999):
        cases.append((heavy, 1.0, 0, p))
    ties = floor.clone()
    ties[[10, 20, 30]] = 6.0
    ties[100:2100:250] = 5.0  # eight ties: the cut falls among them
    for p in (0.3, 0.5, 0.7, 0.85, 0.95):
        cases.append((ties, 1.0, 0, p))
    cases.append((ties, 0.5, 0, 0.9))
    wide = torch.randn(V, generator=g) * 2.0
    wide[200:330] = 4.0  # 130 ties on the boundary of top-k 100: 100 - (keys above) of them are in the set
    for k, p in ((100, 0.5), (100, 0.9), (100, 0.999), (400, 0.3), (V - 1, 0.6)):
        cases.append((wide, 1.0, k, p))
    cases.append((torch.full((V,), 0.25), 1.0, 0, 0.5))  # every key in one bin: more than the pool holds
    zeros = (torch.randn(V, generator=g) * 1.5).round()  # thousands of ties a value, and both zeros, which are one value
    assert (zeros == 0).sum() > 100 and torch.signbit(zeros[zeros == 0]).any() and not torch.signbit(zeros[zeros == 0]).all()
    for T, k, p in ((1.0, 0, 0.6), (1.7, 0, 0.95), (1.0, 200, 0.9), (0.0, 0, 1.0), (1.0, 30, 1.0)):
        cases.append((zeros.clamp(max=0.0) if T == 0.0 else zeros, T, k, p))
    cases.append((torch.randn(V, generator=g) * 0.01, 1.0, 0, 0.9))  # nearly flat: a few bins hold the row
    peaked = torch.linspace(0.0, -40.0, V)[torch.randperm(V, generator=g)]
    for T, p in ((1.0, 0.9), (0.3, 0.5), (3.0, 0.95)):
        cases.append((peaked, T, 0, p))
    draws = 48
    for row, T, k, p in cases:
        logits = row.to(DEV).repeat(draws, 1)
        u = [plain.uniform(1000 + k, i) for i in range(draws)]
        u[0], u[1] = 0.0, 1.0 - 2.0 ** -40  # the first and the last id that are kept
        out = torch.empty(draws, dtype=torch.int32, device=DEV)
        ops.sample(out, logits, torch.full((draws,), T, dtype=torch.float32, device=DEV),
                   torch.full((draws,), k, dtype=torch.int32, device=DEV),
                   torch.full((draws,), p, dtype=torch.float32, device=DEV), torch.tensor(u, dtype=torch.float64, device=DEV))
        probs = plain.probabilities(row.numpy(), T, k, p)
        cdf = np.cumsum(probs)
        for i, got in enumerate(out.tolist()):
            want = plain.sample(probs, u[i])
            if got != want:
                assert probs[got] > 0 and np.abs(cdf - u[i]).min() < 1e-5, (V, T, k, p, i, got, want)


@pytest.mark.parametrize("V", [1000, 50257, 70001])
def test_sampler_without_cuts(ops, V):
    """Temperature alone, called without top-k and top-p: the shorter kernel draws what the
    plain sampler draws, also from a row of ties and beside a greedy row."""
    import plain_gpt2 as plain

    temps = [1.0, 0.8, 0.0, 1.7, 0.3, 1.0, 0.05]
    logits = rnd(len(temps), V, scale=2.0, seed=13)
    logits[5, :] = -1.5  # all equal
    logits[3, 40:90] = 6.0
    cpu = logits.cpu().numpy()
    with pytest.raises(ops.KernelError):
        ops.sample(torch.empty(len(temps), dtype=torch.int32, device=DEV), logits,
                   torch.tensor(temps, dtype=torch.float32, device=DEV), None,
                   torch.ones(len(temps), dtype=torch.float32, device=DEV),
                   torch.zeros(len(temps), dtype=torch.float64, device=DEV))
    for trial in range(8):
        u = [plain.uniform(23 + trial, r) for r in range(len(temps))]
        out = torch.empty(len(temps), dtype=torch.int32, device=DEV)
        ops.sample(out, logits, torch.tensor(temps, dtype=torch.float32, device=DEV), None, None,
                   torch.tensor(u, dtype=torch.float64, device=DEV))
        got = out.tolist()
        for r, T in enumerate(temps):
            probs = plain.probabilities(cpu[r], T, 0, 1.0)
            want = plain.sample(probs, u[r])
            if got[r] != want:
                cdf = np.cumsum(probs)
                assert probs[got[r]] > 0 and np.abs(cdf - u[r]).min() < 1e-5, (V, r, T, got[r], want)


@pytest.mark.parametrize("K", [64, 768, 832, 3072])
def test_tiles_of_every_shape_give_a_row_the_same_bits(ops, K):
    """The tiled products of the batch-invariant mode: the small tiles whose four groups of waves
    walk K side by side (16, 17) and the large ones whose one group keeps four sums by unit of K
    (102, 106, 108) leave the same bits in a row, whatever rows are beside it; K of one unit, of
    whole rounds of four units and of 13 units."""
    M, N = 200, 320
    a, w, bias = rnd(M, K, dtype=torch.bfloat16, seed=K), rnd(N, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2), rnd(N, seed=2)
    want = gemm_reference(a.float(), w.float(), bias, "none")
    full = {}
    for tile in (102, 106, 108, 16, 17):
        out = torch.empty(M, N, device=DEV)
        ops.gemm_mfma_dl(a, w, bias, out=out, tile=tile)
        close(out, want, 2e-5, f"tile {tile}")
        full[tile] = out
    for tile in (106, 108, 16, 17):
        assert torch.equal(full[tile], full[102]), f"tile {tile} against 102"
    for rows in (slice(0, 8), slice(37, 38), slice(100, 164)):
        for tile in (16, 17):
            out = torch.empty(rows.stop - rows.start, N, device=DEV)
            ops.gemm_mfma_dl(a[rows], w, bias, out=out, tile=tile)
            assert torch.equal(out, full[108][rows]), f"rows {rows} in tiles {tile}"


@pytest.mark.parametrize("K", [64, 192, 768, 832, 1600, 3072])
def test_rows_give_the_bits_of_the_tiles(ops, K):
    """The product of few rows leaves the bits of the tiles of four sums (held to the 32-bit reference above): rings of every
    depth (up to 3, 6 and 12 units a wave, and around them again), every strip, rows and features at the edges of both."""
    for M in (1, 8, 9, 17, 32, 33, 64):
        for N in (3, 40, 301):
            a, w, bias = rnd(M, K, dtype=torch.bfloat16, seed=K), rnd(N, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2), rnd(N, seed=2)
            want, base = torch.empty(M, N, device=DEV), rnd(M, N, seed=3)
            ops.gemm_mfma_dl(a, w, bias, out=want, tile=17)
            added = base.clone()
            ops.gemm_mfma_dl(a, w, bias, residual=added, epilogue=ops.EPI_RESIDUAL, tile=17)
            for strip in (0, 8, 16, 32):
                out, res = torch.full((M, N), float("nan"), device=DEV), base.clone()
                ops.gemm_rows(a, w, bias, out=out, strip=strip)
                ops.gemm_rows(a, w, bias, residual=res, epilogue=ops.EPI_RESIDUAL, strip=strip)
                assert torch.equal(out, want) and torch.equal(res, added), (M, N, strip)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K", [64, 768, 832, 1024, 1600, 2048])
def test_a_norm_inside_the_product_leaves_its_own_kernels_bits(ops, dtype, K):
    """The norm computed inside the product of few rows (the batch-invariant mode's and the 32-bit one) against the norm's kernel and the
    plain product: the same bits, with and without weight and bias, GELU behind it, keys and values to their pages."""
    with ops.batch_invariant(dtype == torch.bfloat16):
        for M in (1, 3, 4, 5, 9, 16, 17, 33):
            x, lw, lb = rnd(M, K, seed=K, scale=3.0), rnd(K, seed=4), rnd(K, seed=5)
            w, bias = rnd(3 * 32, K, dtype=dtype, seed=6, scale=0.2), rnd(3 * 32, seed=7)
            slots = torch.randperm(40)[:M].to(torch.int32).to(DEV)
            slots[M // 2] = -1
            for weight, shift in ((lw, lb), (None, None)):
                normed, want, out = torch.empty(M, K, dtype=dtype, device=DEV), torch.empty(M, 96, dtype=dtype, device=DEV), torch.empty(M, 96, dtype=dtype, device=DEV)
                fused = ops.gemm_f32_ln if dtype == torch.float32 else ops.gemm_rows_ln
                ops.layernorm(normed, x, weight, shift, 1e-5)
                ops.gemm(normed, w, bias, out=want, epilogue=ops.EPI_GELU_TANH)
                fused(x, weight, shift, 1e-5, w, bias, out=out, epilogue=ops.EPI_GELU_TANH)
                assert torch.equal(out, want), (M, weight is None)
                got = []
                for one in (False, True):
                    q, kc, vc = (torch.zeros(s, dtype=dtype, device=DEV) for s in ((M, 32), (10, 2, 4, 16), (10, 2, 4, 16)))
                    kv = dict(out=q, kv=(kc, vc, slots, 32))
                    if one:
                        fused(x, weight, shift, 1e-5, w, bias, epilogue=ops.EPI_QKV_PAGED, **kv)
                    elif dtype == torch.float32:
                        ops.gemm_f32_qkv(normed, w, bias, **kv)
                    else:
                        ops.gemm(normed, w, bias, epilogue=ops.EPI_QKV_PAGED, **kv)
                    got.append((q, kc, vc))
                assert all(torch.equal(a, b) for a, b in zip(*got)), (M, weight is None)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,hd,S", [(1, 64, 2), (12, 64, 4), (5, 128, 3), (8, 16, 8), (25, 64, 5)])
def test_splits_merged_inside_the_product_leave_the_merges_bits(ops, dtype, H, hd, S):
    """Attention's splits merged inside the output projection against the merge's kernel and the plain product, splits without keys among them."""
    K, N = H * hd, 72
    with ops.batch_invariant(dtype == torch.bfloat16):
        for M in (1, 3, 4, 9, 17, 33):
            p = rnd(M, H, S, hd + 4, seed=M)
            p[..., hd + 1] = p[..., hd + 1].abs() + 0.5
            p[::2, :, S - 1, hd], p[::2, :, S - 1, hd + 1] = -float("inf"), 0.0
            w, bias, base = rnd(N, K, dtype=dtype, seed=1, scale=0.2), rnd(N, seed=2), rnd(M, N, seed=3)
            att, want, got = torch.empty(M, K, dtype=dtype, device=DEV), base.clone(), base.clone()
            ops.attention_merge(att, p)
            ops.gemm(att, w, bias, residual=want, epilogue=ops.EPI_RESIDUAL)
            ops.gemm_splits(p, w, bias, residual=got)
            assert torch.equal(got, want), M


def test_rows_made_inside_a_product_are_as_many_as_lds_holds(ops):
    """16 rows of 1,664, or 13 of 2,048, beside a workgroup's weights in 32 bits; 8 of 8,192 as merged splits in bfloat16, 4 in 32 bits: they run. More are refused, not run past it."""
    for M, K, runs in ((16, 1664, True), (13, 2048, True), (14, 2048, False), (16, 2048, False)):
        x, w = rnd(M, K, seed=1), rnd(2064, K, seed=2, scale=0.2)
        rows, want, got = torch.empty(M, K, device=DEV), torch.empty(M, 2064, device=DEV), torch.zeros(M, 2064, device=DEV)
        if not runs:
            with pytest.raises(ops.KernelError, match="LDS"):
                ops.gemm_f32_ln(x, None, None, 1e-5, w, None, out=got)
            assert not got.any()
            continue
        ops.layernorm(rows, x, None, None, 1e-5)
        ops.gemm(rows, w, None, out=want)
        ops.gemm_f32_ln(x, None, None, 1e-5, w, None, out=got)
        assert torch.equal(got, want), (M, K)
    for M, H, dtype, runs in ((8, 64, torch.bfloat16, True), (32, 64, torch.bfloat16, False), (4, 64, torch.float32, True), (16, 64, torch.float32, False)):
        p, w, base = rnd(M, H, 2, 132, seed=3), rnd(40, H * 128, dtype=dtype, seed=4, scale=0.2), rnd(M, 40, seed=5)
        p[..., 129] = p[..., 129].abs() + 0.5
        att, want, got = torch.empty(M, H * 128, dtype=dtype, device=DEV), base.clone(), base.clone()
        with ops.batch_invariant(dtype == torch.bfloat16):
            if not runs:
                with pytest.raises(ops.KernelError, match="LDS"):
                    ops.gemm_splits(p, w, None, residual=got)
                assert torch.equal(got, base)
                continue
            ops.attention_merge(att, p)
            ops.gemm(att, w, None, residual=want, epilogue=ops.EPI_RESIDUAL)
            ops.gemm_splits(p, w, None, residual=got)
            assert torch.equal(got, want), (M, H, dtype)


@pytest.mark.parametrize("K", [64, 768, 3072])
def test_tiles_of_one_sum_give_a_row_the_same_bits(ops, K):
    """The tiles of many rows take K in one chain of the same steps whatever their shape: the same bits from each, inside the
    output and at its edges, in 32 bits and in bfloat16."""
    M, N = 300, 520
    a, w, bias = rnd(M, K, dtype=torch.bfloat16, seed=K), rnd(N, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2), rnd(N, seed=2)
    want = gemm_reference(a.float(), w.float(), bias, "none")
    for dtype, tol in ((torch.float32, 2e-5), (torch.bfloat16, 8e-3)):
        first = None
        for tile in (2, 6, 7, 8, 9, 11, 15):
            out = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
            ops.gemm_mfma_dl(a, w, bias, out=out, tile=tile)
            close(out, want, tol, f"tile {tile}")
            first = out if first is None else first
            assert torch.equal(out, first), f"tile {tile} against 2"


@pytest.mark.parametrize("kernel", ["skinny", "mfma128", "mfma64", "dl2", "dl6", "dl7", "dl8", "dl9", "dl11", "dl15", "dl16", "dl17", "auto"])
@pytest.mark.parametrize("M,H,Hkv,hd,K,page", [(5, 3, 3, 16, 64, 4), (40, 4, 2, 32, 128, 16), (200, 5, 5, 48, 192, 8), (130, 2, 1, 64, 64, 64), (700, 6, 3, 64, 128, 16),
                                               (50, 3, 3, 32, 128, 24), (300, 4, 2, 64, 192, 48),
                                               (780, 16, 16, 64, 1024, 16)])  # (the size at which `auto` takes tiles of 128 x 128)
def test_gemm_paged_qkv_epilogue(ops, kernel, M, H, Hkv, hd, K, page):
    """Queries to a dense buffer, keys and values straight into shuffled cache slots, against
    the plain product followed by the scatter kernel."""
    if kernel == "skinny" and M > 64:
        pytest.skip("at most 64 rows")
    q_dim, kv_dim = H * hd, Hkv * hd
    N = q_dim + 2 * kv_dim
    a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    pages = -(-M // page) + 3
    slots = torch.randperm(pages * page)[:M].to(torch.int32).to(DEV)
    kc = torch.zeros(pages, Hkv, page, hd, dtype=torch.bfloat16, device=DEV)
    vc = torch.zeros_like(kc)
    q = torch.zeros(M, q_dim, dtype=torch.bfloat16, device=DEV)
    kw = dict(out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, q_dim))
    if kernel == "skinny":
        ops.gemm_skinny(a, w, bias, **kw)
    elif kernel == "auto":
        ops.gemm(a, w, bias, **kw)
    elif kernel.startswith("dl"):
        ops.gemm_mfma_dl(a, w, bias, tile=int(kernel[2:]), **kw)
    else:
        ops.gemm_mfma(a, w, bias, tile=1 if kernel == "mfma128" else 2, **kw)
    full = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.gemm_simple(a, w, bias, out=full)
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    ops.kv_write(kc2, vc2, full, q_dim, q_dim + kv_dim, slots)
    close(q, full[:, :q_dim], 1e-2, "queries")
    close(kc, kc2, 1e-2, "keys")
    close(vc, vc2, 1e-2, "values")
    assert (kc == 0).sum() == (kc2 == 0).sum()  # nothing written outside the tokens' slots


@pytest.mark.parametrize("M,H,Hkv,hd,K,page", [(1, 4, 4, 16, 64, 16), (9, 6, 2, 32, 192, 8), (16, 12, 12, 64, 768, 64), (27, 5, 5, 48, 240, 16),
                                               (32, 12, 12, 64, 768, 64)])
def test_folded_norm_with_the_paged_qkv_epilogue(ops, M, H, Hkv, hd, K, page):
    """The product that normalises its own rows, writing queries to a dense buffer and keys and
    values into shuffled cache slots: what the standalone norm followed by the streaming
    product writes."""
    q_dim, kv_dim = H * hd, Hkv * hd
    N = q_dim + 2 * kv_dim
    x = rnd(2, M, K, scale=2.0)
    lw, lb = rnd(K, seed=5) + 1.0, rnd(K, seed=6)
    w, bias = rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
    pages = -(-M // page) + 3
    slots = torch.randperm(pages * page)[:M].to(torch.int32).to(DEV)
    got = [torch.zeros(pages, Hkv, page, hd, dtype=torch.bfloat16, device=DEV) for _ in range(2)] + [torch.zeros(M, q_dim, dtype=torch.bfloat16, device=DEV)]
    ops.gemm_skinny_ln(x, lw, lb, 1e-5, w, bias, out=got[2], epilogue=ops.EPI_QKV_PAGED, kv=(got[0], got[1], slots, q_dim))
    normed = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
    ops.layernorm(normed, x, lw, lb, 1e-5)
    want = [torch.zeros_like(got[0]), torch.zeros_like(got[1]), torch.zeros_like(got[2])]
    ops.gemm_skinny(normed, w, bias, out=want[2], epilogue=ops.EPI_QKV_PAGED, kv=(want[0], want[1], slots, q_dim), ksplit=8, wide=0,
                    mtile=1 if M <= 16 else 0)
    for g, t, what in zip(got, want, ("keys", "values", "queries")):
        if M <= 16:
            assert torch.equal(g, t), what
        else:
            close(g, t, 8e-3, what)
    assert (got[0] == 0).sum() == (want[0] == 0).sum()  # nothing written outside the tokens' slots


@pytest.mark.parametrize("seed", range(4))
def test_drawn_shapes_of_the_folded_and_the_cut_products(ops, seed):
    """Shapes drawn at random (rows, widths that are multiples of 8 only, any number of output
    features, planes up to 16, rows to add to in up to 9 planes): the folded norm against norm +
    product, the cut products against the whole product."""
    import random

    rng = random.Random(seed)
    for _ in range(12):
        M = rng.choice([1, 2, 7, 8, 9, 16, 17, 31, 32])
        K, N, P = 8 * rng.randint(1, 256), rng.randint(1, 700), rng.choice([1, 1, 2, 4, 5, 16])
        planes = rnd(P, M, K, scale=2.0, seed=rng.randint(0, 99))
        planes[0] += 0.5
        x = planes if P > 1 else planes[0]
        lw, lb = rnd(K, seed=5) + 1.0, rnd(K, seed=6)
        w, bias = rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        ops.gemm_skinny_ln(x, lw, lb, 1e-5, w, bias, out=out, epilogue=ops.EPI_GELU_TANH, wide=rng.choice([0, 1]) if M <= 16 else 0)
        normed = torch.empty(M, K, dtype=torch.bfloat16, device=DEV)
        ops.layernorm(normed, x, lw, lb, 1e-5)
        two = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        ops.gemm(normed, w, bias, out=two, epilogue=ops.EPI_GELU_TANH)
        close(out, two, 1e-2, f"folded norm M={M} K={K} N={N} planes={P}")
    for _ in range(12):
        M, K, N = rng.choice([1, 5, 16, 33, 64]), 8 * rng.randint(8, 400), rng.randint(1, 300)
        units = (K + 63) // 64
        parts = rng.randint(1, min(8, units))
        if (parts - 1) * ((units + parts - 1) // parts) >= units:
            parts = 1
        a, w, bias = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(N, seed=2)
        base = rnd(rng.choice([1, 2, 4, 5, 9]), M, N, seed=3)
        want = a.double() @ w.double().t() + bias.double() + base.double().sum(0)
        planes = torch.full((parts, M, N), float("nan"), device=DEV)
        ops.gemm_skinny_parts(a, w, planes, bias=bias, base=base)
        close(planes.double().sum(0), want, 1e-5, f"streaming product in parts M={M} K={K} N={N} parts={parts}")
        if K % 64 == 0 and parts <= K // 64 and (parts - 1) * ((K // 64 + parts - 1) // parts) < K // 64:
            planes = torch.full((parts, M, N), float("nan"), device=DEV)
            ops.gemm_mfma_dl_parts(a, w, planes, bias=bias, base=base, tile=rng.choice([6, 16]))
            close(planes.double().sum(0), want, 1e-5, f"tiled product in parts M={M} K={K} N={N} parts={parts}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,d,indexed", [(1, 16, True), (7, 100, True), (33, 1600, False), (5, 257, True)])
def test_gather_rows(dtype, n, d, indexed):
    """out[r] = x[rows[r]] in the output's dtype; without rows the first n rows."""
    from liyab_amd.kernels import ops

    g = torch.Generator().manual_seed(n * 1000 + d)
    x = torch.randn(n + 9, d, generator=g).to(DEV)
    rows = torch.randint(0, n + 9, (n,), generator=g, dtype=torch.int32).to(DEV) if indexed else None
    out = torch.full((n, d), 7.0, dtype=dtype, device=DEV)
    ops.gather_rows(out, x, rows)
    want = (x[rows.long()] if indexed else x[:n]).to(dtype)
    assert torch.equal(out, want)


@pytest.mark.parametrize("n", [1, 255, 50257 * 3, 4096 * 256 + 5])
def test_scale_in_place(n):
    from liyab_amd.kernels import ops

    x = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(DEV)
    want = x * 0.37
    ops.scale_(x, 0.37)
    assert torch.equal(x, want)


@pytest.mark.parametrize("n,d,n_sum", [(1, 3, 1), (5, 768, 2), (3, 769, 3), (7, 1024, 1), (2, 1600, 2), (4, 2048, 3), (513, 260, 1), (1025, 65, 2),
                                     (2, 256, 3), (3, 1280, 1), (600, 1281, 2), (2, 1700, 3)])
@pytest.mark.parametrize("also", ["nothing", "gate", "centred", "next"])
def test_rows_update_by_waves_is_the_one_by_workgroups(ops, n, d, n_sum, also):
    """A wave a row for up to three rows of y a token, a workgroup a row for more: with rows of zeros added to make four, the same
    update (x + 0 is x)."""
    x, y = rnd(n, d), rnd(n, n_sum, d, seed=1, scale=2.0) + 0.5
    more = torch.cat([y, torch.zeros(n, 4 - n_sum, d, device=DEV)], dim=1)
    w, kw = rnd(d, seed=2) + 1.0, {}
    if also == "gate":
        kw["gate"] = rnd(n, d + 4, seed=5)[:, 3:3 + d]
    elif also == "centred":
        kw.update(bias=rnd(d, seed=3), centred=True)
    elif also == "next":
        kw["next_norm"] = (rnd(d, seed=4) + 1.0, 1e-6)
    for cast in (torch.bfloat16, torch.float32):
        got = []
        for rows, k in ((y, n_sum), (more, 4)):
            into, out = x.clone(), torch.full((n, d), float("nan"), dtype=cast, device=DEV)
            ops.gated_norm_add(into, rows.reshape(n * k, d), w, 1e-5, n_sum=k, cast_out=out, **kw)
            got.append((into, out))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("M,H,Hkv,hd,K,page", [(1, 4, 4, 16, 64, 16), (4, 12, 12, 64, 768, 64), (17, 5, 5, 48, 100, 16), (65, 6, 2, 32, 130, 24), (300, 12, 12, 64, 96, 16), (3, 3, 1, 10, 30, 7)])
def test_float32_qkv_product_into_the_pages(ops, M, H, Hkv, hd, K, page):
    """Queries to a dense buffer, keys and values straight into shuffled slots: the bits of the product followed by the
    scatter, in strips and in tiles, heads that are no multiple of four; slots of no token or outside the caches stay unwritten."""
    q_dim, kv_dim = H * hd, Hkv * hd
    a, w, bias = rnd(M, K), rnd(q_dim + 2 * kv_dim, K, seed=1), rnd(q_dim + 2 * kv_dim, seed=2)
    pages = -(-M // page) + 3
    slots = torch.randperm(pages * page)[:M].to(torch.int32)
    if M > 16:
        slots[3], slots[10] = -1, pages * page
    slots = slots.to(DEV)
    full = torch.empty(M, q_dim + 2 * kv_dim, device=DEV)
    ops.gemm_simple(a, w, bias, out=full)
    want = [torch.zeros(pages, Hkv, page, hd, device=DEV) for _ in range(2)]
    ops.kv_write(*want, full, q_dim, q_dim + kv_dim, slots)
    got = [torch.zeros_like(want[0]) for _ in range(2)]
    q = torch.full((M, q_dim), float("nan"), device=DEV)
    ops.gemm_f32_qkv(a, w, bias, out=q, kv=(*got, slots, q_dim))
    assert torch.equal(q, full[:, :q_dim]) and torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("d", [64, 768, 1300])
@pytest.mark.parametrize("also", ["nothing", "gate"])
def test_rows_update_by_waves_keeps_the_rows(ops, d, also):
    """The rows kept as a convolution's history before the update, by the kernel of a wave a row (two rows of y a token) and by the
    one of a workgroup a row (four, two of them zeros): the last `ring` rows of each request, of no request without a slot, and
    none of the rows behind the step's tokens."""
    from types import SimpleNamespace

    lens, contexts, slots, ring, n_slots, n = [1, 5, 2, 4], [9, 5, 40, 30], [2, 0, -1, 7], 3, 5, 15
    real = sum(lens)
    tok_seq = [r for r, q in enumerate(lens) for _ in range(q)] + [0] * (n - real)
    positions = [contexts[r] - q + i for r, q in enumerate(lens) for i in range(q)] + [8] * (n - real)
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    ctx = SimpleNamespace(n_tokens=n, n_seqs=len(lens), tok_seq=dev(tok_seq), positions=dev(positions), context_lens=dev(contexts), state_slots=dev(slots),
                          seq_starts=dev([0, 1, 6, 8, 12]))
    x, y, w = rnd(n, d), rnd(n, 2, d, seed=1), rnd(d, seed=2) + 1.0
    gate = rnd(n, d, seed=3) if also == "gate" else None
    want = torch.full((n_slots, ring, d), 7.0, device=DEV)
    for t in range(real):
        r = tok_seq[t]
        if positions[t] >= contexts[r] - ring and 0 <= slots[r] < n_slots:
            want[slots[r], positions[t] % ring] = x[t]
    got = []
    for rows in (y, torch.cat([y, torch.zeros_like(y)], dim=1)):
        into, state = x.clone(), torch.full((n_slots, ring, d), 7.0, device=DEV)
        ops.gated_norm_add(into, rows.reshape(-1, d), w, 1e-5, n_sum=rows.shape[1], gate=gate, keep=(state, ctx))
        assert torch.equal(state, want)
        got.append(into)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("V", [330, 600, 4093, 4100, 9000, 20000])
def test_sampler_at_few_ids_a_thread(ops, V):
    """The same rules where the floor for the k-th largest is found among the threads' largest keys and among those of four neighbours (from 512 such
    values on), with ties at the boundary inside and outside the pool."""
    test_sampler_against_the_plain_sampler(ops, V)


@pytest.mark.parametrize("form", ["one", "relu2", "two", "clamped", "heads", "gated heads"])
@pytest.mark.parametrize("K", [64, 192, 256, 448, 832, 1600])
def test_products_of_whole_units_leave_the_bits_of_the_others(ops, form, K):
    """Tiles of 16 places: the kernel for whole units of 64 k against the one for any K (held to the 32-bit reference above), which gets eight zeros more
    a row: units a wave of none, one, and around the ring; rows and features at the edges of a tile, empty places, an unused tile."""
    pad = lambda t: torch.nn.functional.pad(t, (0, 8)).contiguous()  # noqa: E731
    for n, N in ((1, 3), (5, 40), (33, 16), (17, 130)):
        if "heads" in form:
            H = 3
            a, w = rnd(n, H, K, dtype=torch.bfloat16), rnd(H, N, K, seed=1, scale=0.2, dtype=torch.bfloat16)
            for gate in ((rnd(n, H * N, seed=2), rnd(n, H * N, seed=2, dtype=torch.bfloat16)) if form == "gated heads" else (None,)):
                got, want = (torch.full((n, H * N), float("nan"), device=DEV) for _ in range(2))
                ops.heads_product(got, a.reshape(n, H * K), w, gate)
                ops.heads_product(want, pad(a).reshape(n, H * (K + 8)), pad(w), gate)
                assert torch.equal(got, want), (n, N)
            continue
        E, two = 5, form in ("two", "clamped")
        a, w0, w1 = rnd(n, K, dtype=torch.bfloat16), rnd(E, N, K, seed=1, scale=0.2, dtype=torch.bfloat16), rnd(E, N, K, seed=2, scale=0.2, dtype=torch.bfloat16)
        expert = torch.randint(0, E - 1, (2 * n,), generator=torch.Generator().manual_seed(3))
        tiles = ops.moe_tiles(2 * n, E, 16) + 1
        rows, group, at = torch.full((tiles, 16), -1, dtype=torch.int32), torch.full((tiles,), -1, dtype=torch.int32), 0
        for e in sorted(set(expert.tolist())):
            for c in (expert == e).nonzero().flatten().int().split(16):
                at += at == 1  # a tile nobody uses
                rows[at, :len(c)], group[at], at = c, e, at + 1
        for scale in (None, rnd(2 * n, seed=4)):
            got, want = (torch.full((2 * n, N), float("nan"), device=DEV) for _ in range(2))
            for out, x, u, v in ((got, a, w0, w1), (want, pad(a), pad(w0), pad(w1))):
                ops.moe_product(out, x, u, v if two else None, rows.to(DEV).flatten(), group.to(DEV), a_div=2, row_scale=scale, block=16,
                                act="relu2" if form == "relu2" else "none", clamp=(0.7, 1.702, 1.0) if form == "clamped" else None)
            assert torch.equal(got, want), (n, N)


@pytest.mark.parametrize("activation", ["silu", "gelu_tanh"])
@pytest.mark.parametrize("K,ff", [(192, 1), (192, 24), (768, 2048), (832, 17), (1600, 100), (2048, 5504), (8192, 40)])
def test_an_activation_inside_its_product_leaves_its_own_kernels_bits(ops, K, ff, activation):
    """A gated feed-forward's first product with the activation in its epilogue against the product to 32-bit rows and the
    activation's kernel: the same bits, at the edges of a strip of features and of the waves that share K."""
    for M in (1, 3, 8):
        a, w = rnd(M, K + 8, dtype=torch.bfloat16, seed=K)[:, :K], rnd(2 * ff, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2)
        assert ops.glu_in_product_takes(a, w)
        both, want, got = torch.empty(M, 2 * ff, device=DEV), torch.empty(M, ff, dtype=torch.bfloat16, device=DEV), torch.zeros(M, ff, dtype=torch.bfloat16, device=DEV)
        ops.gemm(a, w, None, out=both)
        ops.glu(want, both, activation)
        ops.gemm_glu(got, a, w, activation)
        assert torch.equal(got, want), M


@pytest.mark.parametrize("K", [64, 192, 1728, 2048])
def test_an_activation_inside_its_product_takes_eight_rows_at_most(ops, K):
    """What the entry says of itself at every K: nine rows are refused by their number (16 waves' rings of 16 rows would pass a workgroup's LDS), eight run."""
    a, w = rnd(9, K, dtype=torch.bfloat16, seed=1), rnd(2 * 24, K, dtype=torch.bfloat16, seed=2, scale=0.2)
    out = torch.zeros(9, 24, dtype=torch.bfloat16, device=DEV)
    assert not ops.glu_in_product_takes(a, w)
    with pytest.raises(ops.KernelError, match="at most 8"):
        ops.gemm_glu(out, a, w, "silu")
    ops.gemm_glu(out[:8], a[:8], w, "silu")
    y = a[:8].double() @ w.double().T
    want = torch.nn.functional.silu(y[:, :24]) * y[:, 24:]
    assert (out[:8].double() - want).norm() <= 1e-2 * want.norm() and not out[8].any()


@pytest.mark.parametrize("form", ["one", "centred", "gate", "next"])
def test_rows_update_shares_a_row_among_four_waves_with_the_same_bits(ops, form):
    """Up to 1,536 rows a row belongs to four waves, beyond to one: what a row becomes does not depend on how many there are."""
    for d in (64, 256, 260, 768, 1021, 2048):
        x, y, w, b, gate = rnd(1537, d), rnd(1537 * 3, d, seed=1), rnd(d, seed=2), rnd(d, seed=3), rnd(1537, d + 3, seed=4)[:, :d]
        for k in (1, 2, 3):
            got = []
            for n in (1537, 1536, 3):
                into, cast = x[:n].clone(), torch.empty(n, d, dtype=torch.bfloat16, device=DEV)
                ops.gated_norm_add(into, y[:n * k], w, 1e-5, n_sum=k, cast_out=cast, gate=gate[:n] if form == "gate" else None,
                                   **({"bias": b, "centred": True} if form == "centred" else {"next_norm": (b, 1e-5)} if form == "next" else {}))
                got.append((into, cast))
            for into, cast in got[1:]:
                assert torch.equal(into, got[0][0][:len(into)]) and torch.equal(cast, got[0][1][:len(into)]), (d, k, len(into))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [260, 516, 768, 1028, 1600, 2048])
def test_norm_of_few_rows_shares_a_row_among_waves_with_the_same_bits(ops, d, dtype):
    """Where the rows are few, each piece of 256 entries has a wave of its own; among many a row has one: the same bits, rows in planes too."""
    n, w, b = 1100, rnd(d, seed=1), rnd(d, seed=2)
    for planes in (1, 2, 5, 8):
        x = rnd(planes, n, d, seed=3)
        picked = torch.tensor([3, 0, 1099], dtype=torch.int32, device=DEV)
        for weights in ((w, b), (w, None)):
            many, few, gathered = (torch.empty(rows, d, dtype=dtype, device=DEV) for rows in (n, 5, 3))
            if planes == 1:
                ops.layernorm(many, x[0], *weights, 1e-5)
                ops.layernorm(few, x[0, :5], *weights, 1e-5)
                ops.layernorm(gathered, x[0], *weights, 1e-5, rows=picked)
            else:
                ops.layernorm(many, x, *weights, 1e-5)
                ops.layernorm(few, x[:, :5].contiguous(), *weights, 1e-5)
                ops.layernorm(gathered, x, *weights, 1e-5, rows=picked)
            assert torch.equal(few, many[:5]) and torch.equal(gathered, many[picked.long()]), planes


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,dk,dv", [(12, 12, 64, 64), (6, 2, 40, 40), (5, 1, 30, 33), (8, 8, 256, 256), (32, 8, 128, 64)])
def test_prepared_rows_do_not_depend_on_how_many_there_are(ops, H, G, dk, dv, dtype):
    """Queries, keys and values of up to 256 rows have 256 threads each and stay in registers, those of more (and of wider rows) do not: the same bits;
    turned as neighbours and as halves, rows wider than the heads, slots outside the pages, queries alone."""
    n, page = 259, 16
    src, q_norm, k_norm = rnd(n, (H + G) * dk + G * dv), rnd(H * dk, seed=1), rnd(G * dk, seed=2)
    slots = torch.randperm(20 * page, generator=torch.Generator().manual_seed(3))[:n].int()
    slots[1], slots[2] = -1, 20 * page + 2
    slots, positions = slots.to(DEV), torch.arange(n, dtype=torch.int32, device=DEV) * 37
    for rot, halves in ((0, False), (dk // 2 * 2, False), (dk // 4 * 2, True)):
        freqs = torch.rand(max(rot // 2, 1), dtype=torch.float64, generator=torch.Generator().manual_seed(4)).to(DEV) if rot else None
        for wide in (0, 7):
            for keys in (True, False):
                got = []
                for rows in (n, 3):
                    q = torch.full((rows, H * (dk + wide)), 7.0, dtype=dtype, device=DEV)
                    kc, vc = (torch.full((20, G, page, w + wide), 7.0, dtype=dtype, device=DEV) for w in (dk, dv))
                    ops.qk_prepare_rows(src[:rows], q, kc if keys else None, vc if keys else None, slots[:rows], positions[:rows], q_off=0, k_off=H * dk, v_off=(H + G) * dk,
                                        n_head=H, n_kv_head=G, head_dim=dk, value_dim=dv, q_norm=q_norm, k_norm=k_norm if keys else None, eps=1e-5, freqs=freqs, rot_dims=rot,
                                        rot_halves=halves)
                    got.append((q, kc, vc))
                assert torch.equal(got[1][0], got[0][0][:3])
                for few, many in zip(got[1][1:], got[0][1:]):
                    at = slots[:1].long()
                    rows_of = lambda c: c.transpose(1, 2).flatten(0, 1)  # noqa: E731
                    assert torch.equal(rows_of(few)[at], rows_of(many)[at]) and (rows_of(few) != 7.0).any(dim=2).any(dim=1).sum().item() == (1 if keys else 0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [5, 256, 770])
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_a_short_convolution_with_its_inputs_ahead_has_the_general_kernels_bits(ops, taps, C, dtype):
    """Two to four taps against six, the first ones zeros (the kernel that walks the taps): tokens whose inputs lie in the step, in the ring, in
    both, before position 0, and of a request without a slot."""
    from types import SimpleNamespace

    lens, contexts, slots = [1, 1, 4, 2, 1], [0, 9, 2, 1, 7], [2, 0, 4, 1, -1]
    n = sum(lens)
    seq = [r for r, q in enumerate(lens) for _ in range(q)]
    dev = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    ctx = SimpleNamespace(n_tokens=n, n_seqs=len(lens), max_q=max(lens), tok_seq=dev(seq), positions=dev([contexts[r] + i for r, q in enumerate(lens) for i in range(q)]),
                          seq_starts=dev([sum(lens[:r]) for r in range(len(lens) + 1)]), state_slots=dev(slots), context_lens=dev([c + q for c, q in zip(contexts, lens)]))
    x, weight, before = rnd(n, C), rnd(C, taps, seed=1), rnd(len(lens), 10, C, seed=2)
    for bias in (rnd(C, seed=3), None):
        got = []
        for t, w in ((taps, weight), (6, torch.cat([torch.zeros(C, 6 - taps, device=DEV), weight], dim=1).contiguous())):
            state = torch.full((5, (t - 1) * C), 7.0, device=DEV)
            for r, slot in enumerate(slots):
                for at in range(max(0, contexts[r] - (t - 1)), contexts[r]):
                    if slot >= 0:
                        state[slot, at % (t - 1) * C:(at % (t - 1) + 1) * C] = before[r, at]
            out = torch.empty(n, C, dtype=dtype, device=DEV)
            ops.conv_act(out, x, w, bias, state, 0, ctx)
            got.append(out)
        assert torch.equal(*got)


@pytest.mark.parametrize("K", [64, 192, 832, 1600, 3072])
def test_streamed_products_of_17_rows_and_more_leave_the_bits_of_the_others(ops, K):
    """17 to 64 rows: the kernel whose operands come through rings in LDS (whole units of 64 k) against the one that holds them in registers, which gets
    eight zeros more a row; blocks of rows and strips of features at their edges, sums, the residual stream and parts of K."""
    pad = lambda t: torch.nn.functional.pad(t, (0, 8)).contiguous()  # noqa: E731
    for M in (17, 32, 33, 64):
        for N in (3, 40, 768, 2310):
            a, w, bias = rnd(M, K, dtype=torch.bfloat16, seed=K), rnd(N, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2), rnd(N, seed=2)
            got = []
            for x, y in ((a, w), (pad(a), pad(w))):
                out, half, added = torch.empty(M, N, device=DEV), torch.empty(M, N, dtype=torch.bfloat16, device=DEV), rnd(M, N, seed=3)
                ops.gemm_skinny(x, y, bias, out=out)
                ops.gemm_skinny(x, y, None, out=half)
                ops.gemm_skinny(x, y, bias, residual=added, epilogue=ops.EPI_RESIDUAL)
                planes = torch.empty(1, M, N, device=DEV)
                ops.gemm_skinny_parts(x, y, planes, bias=bias, base=rnd(2, M, N, seed=4))
                got.append((out, half, added, planes))
            assert all(torch.equal(p, q) for p, q in zip(*got)), (M, N)


@pytest.mark.parametrize("ksplit", [1, 4, 16])
@pytest.mark.parametrize("K", [64, 192, 832, 1600])
def test_streamed_products_of_up_to_16_rows_leave_the_bits_of_the_others(ops, K, ksplit):
    """As above for 1 to 16 rows, both kernels on the same waves: one strip of 16 features a workgroup and two (5,000 features), rings of two units and of four, every
    epilogue, K in one part and in two."""
    pad = lambda t: torch.nn.functional.pad(t, (0, 8)).contiguous()  # noqa: E731
    for M in (1, 8, 9, 16):
        for N in (48, 768, 5000):  # whole heads of 16 below, for the pages
            a, w, bias, base = rnd(M, K, dtype=torch.bfloat16, seed=K), rnd(N, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2), rnd(N, seed=2), rnd(5, M, N, seed=4)
            slots = torch.randperm(40)[:M].to(torch.int32).to(DEV)
            slots[M // 2] = -1
            got = []
            for x, y in ((a, w), (pad(a), pad(w))):
                out, half, added = torch.empty(M, N, device=DEV), torch.empty(M, N, dtype=torch.bfloat16, device=DEV), rnd(M, N, seed=3)
                gelu, erf = torch.empty(M, N, device=DEV), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
                ops.gemm_skinny(x, y, bias, out=out, ksplit=ksplit)
                ops.gemm_skinny(x, y, None, out=half, ksplit=ksplit)
                ops.gemm_skinny(x, y, bias, out=gelu, epilogue=ops.EPI_GELU_TANH, ksplit=ksplit)
                ops.gemm_skinny(x, y, bias, out=erf, epilogue=ops.EPI_GELU_ERF, ksplit=ksplit)
                ops.gemm_skinny(x, y, bias, residual=added, epilogue=ops.EPI_RESIDUAL, ksplit=ksplit)
                one, two = torch.empty(1, M, N, device=DEV), torch.empty(2, M, N, device=DEV)
                ops.gemm_skinny_parts(x, y, one, bias=bias, base=base, ksplit=ksplit)
                if K > 64:  # (an odd number of units: the eight zeros leave the parts' border where it is)
                    ops.gemm_skinny_parts(x, y, two, bias=bias, base=base[:2], ksplit=ksplit)
                else:
                    two.zero_()
                outs = [out, half, gelu, erf, added, one, two]
                if N == 768:
                    q, kc, vc = (torch.zeros(s, dtype=torch.bfloat16, device=DEV) for s in ((M, 256), (10, 16, 4, 16), (10, 16, 4, 16)))
                    ops.gemm_skinny(x, y, bias, out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, 256), ksplit=ksplit)
                    outs += [q, kc, vc]
                got.append(outs)
            assert all(torch.equal(p, q) for p, q in zip(*got)), (M, N, [torch.equal(p, q) for p, q in zip(*got)])


@pytest.mark.parametrize("K", [768, 1280])
@pytest.mark.parametrize("M", [17, 32])
def test_streamed_products_with_one_unit_in_flight_keep_every_epilogues_bits(ops, M, K):
    """More than 256 blocks of 16 rows and 16 features, of a wave a unit or two: each epilogue has a kernel of its own there; against the kernel that holds its operands
    in registers, which gets eight zeros more a row."""
    pad = lambda t: torch.nn.functional.pad(t, (0, 8)).contiguous()  # noqa: E731
    N = 3 * 704
    a, w, bias = rnd(M, K, dtype=torch.bfloat16, seed=K), rnd(N, K, dtype=torch.bfloat16, seed=K + 1, scale=0.2), rnd(N, seed=2)
    slots = torch.randperm(60)[:M].to(torch.int32).to(DEV)
    slots[M // 2] = -1
    got = []
    for x, y in ((a, w), (pad(a), pad(w))):
        outs = []
        for dtype in (torch.float32, torch.bfloat16):
            for epilogue in (ops.EPI_NONE, ops.EPI_GELU_TANH, ops.EPI_GELU_ERF):
                out = torch.empty(M, N, dtype=dtype, device=DEV)
                ops.gemm_skinny(x, y, bias, out=out, epilogue=epilogue, ksplit=16)
                outs.append(out)
        added = rnd(M, N, seed=3)
        ops.gemm_skinny(x, y, bias, residual=added, epilogue=ops.EPI_RESIDUAL, ksplit=16)
        q, kc, vc = (torch.zeros(s, dtype=torch.bfloat16, device=DEV) for s in ((M, 704), (15, 44, 4, 16), (15, 44, 4, 16)))
        ops.gemm_skinny(x, y, bias, out=q, epilogue=ops.EPI_QKV_PAGED, kv=(kc, vc, slots, 704), ksplit=16)
        got.append(outs + [added, q, kc, vc])
    assert all(torch.equal(p, q) for p, q in zip(*got)), [torch.equal(p, q) for p, q in zip(*got)]


@pytest.mark.parametrize("K", [64, 512, 576, 768, 832, 1000, 1024])
def test_steps_of_13_to_16_rows_keep_the_folded_norms_bits(ops, K, monkeypatch):
    """A norm and the product behind it as the parts run them, against the kernel that folds them: the same bits on either side of the rows (13 to 16) and widths
    (513 to 1,024) that take the norm's own kernel instead, in planes too. From 8,177 features on four waves share K and not eight: another order of the same
    sum, no further from the 64-bit product."""
    from types import SimpleNamespace

    from liyab_amd.parts import linear as lin
    from liyab_amd.parts.norms import LayerNorm, Normed

    taken = []
    for name in ("gemm_skinny_ln", "layernorm"):
        monkeypatch.setattr(ops, name, (lambda f, n: lambda *a, **k: (taken.append(n), f(*a, **k))[1])(getattr(ops, name), name))
    norm = LayerNorm.__new__(LayerNorm)
    norm.width, norm.eps, norm.dtype, norm.weight, norm.bias = K, 1e-5, torch.bfloat16, rnd(K, seed=1) + 1.0, rnd(K, seed=2)
    for M in (12, 13, 16, 17):
        for N in (16, 300, 8176, 8177, 8192):
            if not ops.skinny_ln_pays(M, N, K):
                continue
            w, bias = rnd(N, K, dtype=torch.bfloat16, seed=3, scale=0.2), rnd(N, seed=4)
            for planes in (1, 4):
                x = rnd(planes, M, K, seed=5) if planes > 1 else rnd(M, K, seed=5)
                ctx = SimpleNamespace(workspace=SimpleNamespace(get=lambda name, shape, dtype: torch.empty(shape, dtype=dtype, device=DEV)))
                got, want = torch.empty(M, N, device=DEV), torch.empty(M, N, device=DEV)
                taken.clear()
                lin.linear(Normed(norm, x, ctx), w, bias, out=got)
                own_kernel = 12 < M <= 16 and 512 < K <= 1024 and K % 64 == 0
                assert taken == (["layernorm"] if own_kernel else ["gemm_skinny_ln"]), (M, N)
                ops.gemm_skinny_ln(x, norm.weight, norm.bias, 1e-5, w, bias, out=want)
                if N <= 8176 or not own_kernel:
                    assert torch.equal(got, want), (M, N, planes)
                    continue
                rows = torch.nn.functional.layer_norm(x.sum(0) if planes > 1 else x, (K,), norm.weight, norm.bias, 1e-5).bfloat16()
                exact = rows.double() @ w.double().T + bias.double()
                err = lambda t: ((t.double() - exact).norm() / exact.norm()).item()  # noqa: E731
                assert err(got) <= 1.1 * err(want) + 1e-7, (M, N, planes, err(got), err(want))
