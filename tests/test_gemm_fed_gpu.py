"""The GEMM tiles whose copies other waves make (gemm_fed_tiles.h, and the 256 x 128 tile), at the edges of every tile,
in one part and in several, with contractions of fewer stages than their rings hold.  Whole numbers: products and
sums are exact, operands lie in buffers of NaN and outputs in canvases."""

import re

import pytest
import torch

import test_kernel_codegen as codegen
from axonn_amd import _native as nv
from launches import launches
from test_gemm_edge_gpu import canvas, check, numbers


@pytest.mark.parametrize("source", ["gemm_fed_nt_f16", "gemm_fed_nn_tn_bf16"])
def test_fed_kernels_keep_the_properties_of_the_others(tmp_path_factory, source):
    kernels = {k: v for k, v in codegen._device_asm(tmp_path_factory, source).items() if "gemm_fed_edge" in k}
    assert len(kernels) == (80 if "nt" in source.split("_")[2] else 40), len(kernels)   # 10 tiles x 8 or 4 products
    codegen.test_solo_kernels_do_not_spill(kernels)
    codegen.test_accumulators_stay_in_their_registers_until_the_last_mfma_has_retired(kernels)


def product(op, a, b, c, M, N, K, code, out, ldc, ws, beta=0, bias=None, z=None, epilogue=nv.EPI_NONE):
    nv.call("axn_gemm_any_n", op, nv.ptr(a), nv.ptr(b), nv.ptr(bias), nv.ptr(c), nv.ptr(z), code, M, N, K, a.stride(0),
            b.stride(0), ldc, epilogue, beta, out, nv.ptr(ws), 0 if ws is None else ws.numel() * 4, nv.current_stream())


@pytest.mark.gpu
@pytest.mark.parametrize("op,M,N,K,tile,parts", [
    (0, 161, 808, 200, "64, 64", 1), (0, 372, 168, 1944, None, 3), (0, 1423, 792, 320, "96, 64", 1),
    (0, 673, 2096, 552, "64, 128", 1), (0, 124, 1824, 2816, None, 5), (0, 1382, 1416, 832, "96, 128", 1),
    (0, 1525, 2152, 1024, "128, 128", 1), (0, 2125, 2088, 656, "96, 192", 1), (0, 1442, 3672, 704, "128, 192", 1),
    (0, 1594, 3880, 1024, "160, 192", 1), (0, 1887, 2488, 488, "256, 128", 1),
    (0, 70, 136, 8, "64, 64", 1), (0, 70, 200, 72, "64, 64", 1),        # one and two stages
    (0, 256, 512, 512, "64, 64", 1),                                    # whole tiles
    (1, 153, 840, 104, "64, 64", 1), (1, 460, 1728, 168, None, 3), (1, 1820, 592, 576, "96, 64", 1),
    (1, 625, 2624, 160, "64, 128", 1), (1, 1127, 1024, 2328, "96, 128", 1), (1, 1444, 1600, 2064, "128, 128", 1),
    (1, 1791, 2432, 2384, "96, 192", 1), (1, 2079, 960, 2232, "128, 192", 1), (1, 1802, 2176, 3672, "160, 192", 1),
    (1, 1600, 472, 2504, "256, 128", 1),
    (2, 193, 1440, 96, "64, 64", 1), (2, 2856, 240, 536, None, 5), (2, 264, 128, 2832, "96, 64", 1),
    (2, 1544, 272, 176, "64, 128", 1), (2, 447, 2000, 1048, "96, 128", 1), (2, 583, 2064, 1672, "128, 128", 1),
    (2, 207, 1200, 3320, "96, 192", 1), (2, 199, 1944, 2624, "128, 192", 1), (2, 1471, 2080, 3824, "128, 256", 1),
    (2, 927, 1832, 3280, "160, 192", 1),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_products_on_every_fed_tile(op, M, N, K, tile, parts, dtype):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    shapes = (((M, K), (N, K), (M, N)), ((M, N), (N, K), (M, K)), ((M, N), (M, K), (N, K)))[op]
    a, b = (numbers(r, c, dtype, gen, 16) for r, c in shapes[:2])
    code, (rows, cols) = nv.dtype_code(dtype), shapes[2]
    nbytes = nv.load().axn_gemm_workspace_bytes(op, M, N, K) if parts > 1 else 0
    ws = torch.full((nbytes // 4,), float("nan"), device="cuda") if nbytes else None
    want = {0: lambda: a.double() @ b.double().t(), 1: lambda: a.double() @ b.double(),
            2: lambda: a.double().t() @ b.double()}[op]()
    full, c = canvas(rows, cols, dtype)
    call = lambda: product(op, a, b, c, M, N, K, code, code, c.stride(0), ws)   # noqa: E731
    found = launches(call)
    m = re.search(r"gemm_(?:fed_)?edge_kernel(?:<|ILi)(\d+)(?:, |ELi)(\d+)", found[0][0])
    assert m and tile in ("%s, %s" % m.groups(), None) and len(found) == (2 if parts > 1 else 1), found
    check(full, c, want)
    if op == 2:
        for out in (dtype, torch.float32):
            full, c = canvas(rows, cols, out)
            c.fill_(3.0)
            product(op, a, b, c, M, N, K, code, nv.dtype_code(out), c.stride(0), ws, beta=1)
            check(full, c, want + 3.0)
    if op == 0:
        bias = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
        for out in (dtype, torch.float32):
            full, c = canvas(rows, cols, out)
            product(op, a, b, c, M, N, K, code, nv.dtype_code(out), c.stride(0), ws, bias=bias, epilogue=nv.EPI_BIAS)
            check(full, c, want + bias)
        fy, y = canvas(rows, cols, dtype)
        fz, z = canvas(rows, cols, dtype)
        product(op, a, b, y, M, N, K, code, code, y.stride(0), ws, bias=bias, z=z, epilogue=nv.EPI_BIAS_GELU)
        gelu = torch.nn.functional.gelu(want + bias)   # within one rounding and the erf's 1.5e-7
        eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        assert bool(((y.double() - gelu).abs() <= eps * gelu.abs() + 2e-7 * (want + bias).abs().clamp(min=1)).all())
        check(fz, z, want + bias)
        flat = torch.full((M * (N + 3) + 8,), 7.0, dtype=dtype, device="cuda")   # rows that start anywhere
        product(op, a, b, flat, M, N, K, code, code, N + 3, ws)
        assert torch.equal(flat[:M * (N + 3)].view(M, N + 3)[:, :N].double(), want.to(dtype).double())
        assert bool((flat[:M * (N + 3)].view(M, N + 3)[:, N:] == 7).all()) and bool((flat[M * (N + 3):] == 7).all())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(300, 1000, 1608), (512, 4096, 2560), (250, 1024, 1024)])
def test_a_workspace_that_a_smaller_tile_does_without(M, N, K):
    """Sizes that have a workspace and are faster in one part on a small tile: accepted and refused as before."""
    nbytes = nv.load().axn_gemm_workspace_bytes(0, M, N, K)
    gen = torch.Generator(device="cuda").manual_seed(M)
    a, b = (numbers(r, K, torch.bfloat16, gen, 16) for r in (M, N))
    ws = torch.full((max(nbytes // 4, 1),), float("nan"), device="cuda")
    full, c = canvas(M, N, torch.bfloat16)
    call = lambda: product(0, a, b, c, M, N, K, nv.BF16, nv.BF16, c.stride(0), ws if nbytes else None)   # noqa: E731
    found = launches(call)
    assert len(found) == 1 and "gemm_fed_edge_kernel" in found[0][0], found
    check(full, c, a.double() @ b.double().t())
    if nbytes:
        with pytest.raises(nv.AxnError, match="workspace too small"):
            product(0, a, b, c, M, N, K, nv.BF16, nv.BF16, c.stride(0), ws[:-4])


@pytest.mark.gpu
@pytest.mark.parametrize("op,M,N,K,workgroups", [
    (1, 640, 3176, 7936, 186), (0, 704, 9856, 7392, 231),                           # one part, with bounds
    (1, 1216, 5208, 2816, 220), (1, 320, 3648, 5376, 252), (2, 4263, 15872, 256, 248),   # parts
    (1, 5120, 256, 1536, 240), (0, 256, 4096, 15360, 256),                          # whole tiles, and parts of them
])
def test_tiles_of_256_by_128_that_are_not_fed(op, M, N, K, workgroups):
    """Where the estimate of the one-wave tile picks 256 x 128, that tile runs: four waves, not eight."""
    shapes = (((M, K), (N, K), (M, N)), ((M, N), (N, K), (M, K)), ((M, N), (M, K), (N, K)))[op]
    a, b, c = (torch.zeros(*s, device="cuda", dtype=torch.bfloat16) for s in shapes)
    nbytes = nv.load().axn_gemm_workspace_bytes(op, M, N, K)
    ws = torch.empty(nbytes // 4, device="cuda") if nbytes else None
    found = launches(lambda: product(op, a, b, c, M, N, K, nv.BF16, nv.BF16, c.stride(0), ws), threads=True)
    assert re.search(r"gemm_(edge|bf16_rest)_kernel", found[0][0]) and "fed" not in found[0][0], found
    assert found[0][1:] == (workgroups, 256) and len(found) == (2 if nbytes else 1), found


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,epilogue", [(2366, 256, 3712, nv.EPI_GELU), (1007, 512, 3200, nv.EPI_GELU),
                                            (3211, 1024, 5504, nv.EPI_BIAS | nv.BIAS_16BIT)])
def test_a_round_of_tiles_has_its_epilogue_counted(M, N, K, epilogue):
    """One part without an epilogue; parts, whose sum has it for little, with one.  Both are right."""
    gen = torch.Generator(device="cuda").manual_seed(M)
    x, w = numbers(M, K, torch.bfloat16, gen, 16), numbers(N, K, torch.bfloat16, gen, 16)
    bias = torch.randint(-3, 4, (N,), generator=gen, device="cuda").bfloat16() if epilogue & nv.BIAS_16BIT else None
    y = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    nbytes = nv.load().axn_gemm_workspace_bytes(0, M, N, K)
    ws = torch.empty(nbytes // 4, device="cuda")
    call = lambda epi: product(0, x, w, y, M, N, K, nv.BF16, nv.BF16, N, ws, bias=bias if epi else None, epilogue=epi)   # noqa: E731
    assert [len(launches(lambda: call(epi))) for epi in (nv.EPI_NONE, epilogue)] == [1, 2]
    call(epilogue)
    want = (x.double() @ w.double().t())
    want = want + bias.double() if bias is not None else torch.nn.functional.gelu(want)
    # exact sums, one rounding to 8 bits; the activation's own error is 2^-20 of its argument at most
    assert float(((y.double() - want).abs() / want.abs().clamp(min=1.0)).max()) <= 2.0 ** -8


@pytest.mark.gpu
@pytest.mark.parametrize("op,M,N,K,fed", [(2, 2048, 6144, 4096, True), (2, 4096, 6144, 4096, True), (2, 1984, 6144, 4096, False),
                                          (0, 4096, 6144, 2048, False), (1, 4096, 2048, 6144, False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rests_of_more_than_64_large_tiles(op, M, N, K, fed, dtype):
    """One whole round and 128 tiles: those of a weight gradient of 2048 tokens on are the ones with copying waves."""
    out, beta = (torch.float32, 1) if op == 2 and dtype == torch.float16 else (dtype, 0)
    gen = torch.Generator(device="cuda").manual_seed(M)
    shapes = (((M, K), (N, K), (M, N)), ((M, N), (N, K), (M, K)), ((M, N), (M, K), (N, K)))[op]
    a, b = (torch.randint(-2, 3, s, generator=gen, device="cuda").to(dtype) for s in shapes[:2])
    c = torch.full(shapes[2], 3.0, device="cuda", dtype=out)
    call = lambda: product(op, a, b, c, M, N, K, nv.dtype_code(dtype), nv.dtype_code(out), c.stride(0), None, beta=beta)   # noqa: E731
    (first, n1, t1), (rest, n2, t2) = launches(call, threads=True)
    assert "solo_kernel" in first and (n1, t1) == (256, 256) and n2 == 256, (first, n1, t1)
    assert t2 == (512 if fed else 256) and ("gemm_fed_edge" in rest) == fed, (rest, t2)
    c.fill_(3.0)
    call()
    rows = torch.randint(0, shapes[2][0], (128,), generator=gen, device="cuda")
    left = {0: lambda: a[rows], 1: lambda: a[rows], 2: lambda: a[:, rows].t()}[op]().double().contiguous()
    right = (b.t() if op == 0 else b).double().contiguous()
    want = left @ right + 3.0 * beta
    # whole numbers: exact in fp32 (the sums are below 2^24), one rounding to a 16-bit result
    assert torch.equal(c[rows].double(), want.to(out).double())
