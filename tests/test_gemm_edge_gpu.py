"""The GEMM kernels with bounds (shapes that are not made of whole tiles) at the sizes where
they can go wrong: one element around tile edges, contractions that end inside a 64-deep
stage, outputs that need one, several and cut rounds of tiles.

Operands are small whole numbers, so every partial sum is exact in fp32 and the expected
result is exact too: the float64 product rounded once to the storage type.  The operands are
views into buffers whose other elements are NaN, and the outputs views into buffers filled
with a canary: what lies outside a view is neither read into a result nor written."""

import threading

import pytest
import torch

from axonn_amd import _native as nv
from launches import launches

pytestmark = pytest.mark.gpu

CANARY = 7.0


def numbers(rows, cols, dtype, gen, pad):
    """A [rows, cols] view of whole numbers -2 .. 2, NaN around it."""
    full = torch.full((rows + 3, cols + pad), float("nan"), dtype=dtype, device="cuda")
    view = full[:rows, :cols]
    view.copy_(torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda"))
    return view


def canvas(rows, cols, dtype):
    full = torch.full((rows + 2, cols + 8), CANARY, dtype=dtype, device="cuda")
    return full, full[:rows, :cols]


def check(full, view, want):
    assert torch.equal(view.double(), want.to(view.dtype).double())
    view.fill_(CANARY)
    assert torch.equal(full, torch.full_like(full, CANARY)), "written outside the output"


@pytest.mark.parametrize("M,N,K", [
    (1, 8, 8), (127, 120, 56), (129, 136, 72), (255, 264, 64), (257, 248, 136), (300, 392, 200),
    (64, 1000, 24), (1000, 128, 1032), (777, 2056, 328),
    (2049, 2304, 128),      # 9 x 9 tiles of 256 x 128 columns and rows
    (4000, 4360, 72),       # 288 large tiles: a full round and a cut rest
    (4100, 4104, 64),       # 289 large tiles that no cut divides
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_edge_kernels_are_exact_and_stay_inside_their_operands(M, N, K, dtype):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    X, W, dY = (numbers(r, c, dtype, gen, 16) for r, c in ((M, K), (N, K), (M, N)))
    code, ld = nv.dtype_code(dtype), lambda t: t.stride(0)
    sfx = "" if dtype == torch.bfloat16 else "_f16"
    stream = nv.current_stream()
    bias = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()

    full, y = canvas(M, N, dtype)
    nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(W), None, nv.ptr(y), None, M, N, K, ld(X), ld(W),
            ld(y), nv.EPI_NONE, stream)
    product = X.double() @ W.double().t()
    check(full, y, product)
    nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(W), nv.ptr(bias), nv.ptr(y), None, M, N, K, ld(X),
            ld(W), ld(y), nv.EPI_BIAS, stream)
    check(full, y, product + bias)
    full32, y32 = canvas(M, N, torch.float32)
    nv.call("axn_gemm_fwd_f32out", nv.ptr(X), nv.ptr(W), nv.ptr(bias), nv.ptr(y32), None, code, M, N, K,
            ld(X), ld(W), ld(y32), nv.EPI_BIAS, stream)
    check(full32, y32, product + bias)

    full, dx = canvas(M, K, dtype)
    nv.call("axn_gemm_dgrad" + sfx, nv.ptr(dY), nv.ptr(W), nv.ptr(dx), M, N, K, ld(dY), ld(W), ld(dx), stream)
    want_dx = dY.double() @ W.double()
    check(full, dx, want_dx)

    full, dw = canvas(N, K, torch.float32)
    want_dw = dY.double().t() @ X.double()
    for beta in (0, 1):
        dw.fill_(3.0)
        nv.call("axn_gemm_wgrad" + sfx, nv.ptr(dY), nv.ptr(X), nv.ptr(dw), M, N, K, ld(dY), ld(X), ld(dw),
                beta, nv.F32, stream)
        check(full, dw, want_dw + 3.0 * beta)
    # both gradients through the joint entry point, dW in the operands' type
    fullx, dx = canvas(M, K, dtype)
    fullw, dw = canvas(N, K, dtype)
    nv.call("axn_gemm_bwd", nv.ptr(dY), nv.ptr(W), nv.ptr(X), nv.ptr(dx), nv.ptr(dw), code, M, N, K, ld(dY),
            ld(W), ld(X), ld(dx), ld(dw), 0, code, stream)
    check(fullx, dx, want_dx)
    check(fullw, dw, want_dw)


@pytest.mark.parametrize("M,N,K", [(129, 136, 72), (300, 2056, 200)])
def test_edge_epilogues_keep_the_pre_activation(M, N, K):
    """GELU on whole-number pre-activations: the saved Z is exact, Y within one rounding of
    the exact function of Z (2^-8 relative for bfloat16) plus the erf's 1.5e-7."""
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    X, W = (numbers(r, c, torch.bfloat16, gen, 8) for r, c in ((M, K), (N, K)))
    bias = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
    for b, epi in ((bias, nv.EPI_BIAS_GELU), (None, nv.EPI_GELU)):
        fz, z = canvas(M, N, torch.bfloat16)
        fy, y = canvas(M, N, torch.bfloat16)
        nv.call("axn_gemm_fwd", nv.ptr(X), nv.ptr(W), nv.ptr(b), nv.ptr(y), nv.ptr(z), M, N, K, X.stride(0),
                W.stride(0), y.stride(0), epi, nv.current_stream())
        pre = X.double() @ W.double().t() + (0 if b is None else b)
        want = torch.nn.functional.gelu(pre)
        assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2e-7 * pre.abs().clamp(min=1)).all())
        check(fz, z, pre)


@pytest.mark.parametrize("op,M,N,K", [
    (0, 65, 136, 2056), (0, 129, 392, 4104), (0, 300, 1000, 1608),      # 128 x 128 tiles
    (0, 520, 2560, 8200), (1, 300, 8200, 2568), (2, 4104, 136, 264),    # 256 wide ones
    (0, 24, 520, 16384), (0, 1, 8, 200000), (0, 64, 4096, 8200),         # few rows, a long contraction
    (0, 128, 384, 12224),    # whole tiles whose 191 stages no number of parts divides
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split_contraction_of_any_shape_with_its_epilogue(op, M, N, K, dtype):
    """The contraction cut into parts of unequal length; the pass that adds them applies bias,
    GELU (pre-activation kept) and beta.  Whole-number operands: every partial sum is exact."""
    lib, code = nv.load(), nv.dtype_code(dtype)
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    nbytes = lib.axn_gemm_workspace_bytes(op, M, N, K)
    assert nbytes > 0, "this shape is meant to be split"
    ws = torch.full((nbytes // 4 + 8,), float("nan"), device="cuda")
    stream = nv.current_stream()
    shapes = (((M, K), (N, K), (M, N)), ((M, N), (N, K), (M, K)), ((M, N), (M, K), (N, K)))[op]
    a, b = (numbers(r, c, dtype, gen, 16) for r, c in shapes[:2])
    full, c = canvas(*shapes[2], torch.float32 if op == 2 else dtype)
    tail = (nv.ptr(ws), nbytes, stream)
    if op == 0:
        bias = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
        pre = a.double() @ b.double().t()
        for bb, epi, want in ((None, nv.EPI_NONE, pre), (bias, nv.EPI_BIAS, pre + bias)):
            nv.call("axn_gemm_fwd_ws", nv.ptr(a), nv.ptr(b), nv.ptr(bb), nv.ptr(c), None, code, M, N, K, a.stride(0),
                    b.stride(0), c.stride(0), epi, *tail)
            check(full, c, want)
        fz, z = canvas(M, N, dtype)
        nv.call("axn_gemm_fwd_ws", nv.ptr(a), nv.ptr(b), nv.ptr(bias), nv.ptr(c), nv.ptr(z), code, M, N, K,
                a.stride(0), b.stride(0), c.stride(0), nv.EPI_BIAS_GELU, *tail)
        want = torch.nn.functional.gelu(pre + bias)   # within one rounding and the erf's 1.5e-7
        eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        assert bool(((c.double() - want).abs() <= eps * want.abs() + 2e-7 * pre.abs().clamp(min=1)).all())
        check(fz, z, pre + bias)
    elif op == 1:
        nv.call("axn_gemm_dgrad_ws", nv.ptr(a), nv.ptr(b), nv.ptr(c), code, M, N, K, a.stride(0), b.stride(0),
                c.stride(0), *tail)
        check(full, c, a.double() @ b.double())
    else:
        c.fill_(3.0)
        nv.call("axn_gemm_wgrad_ws", nv.ptr(a), nv.ptr(b), nv.ptr(c), code, M, N, K, a.stride(0), b.stride(0),
                c.stride(0), 1, nv.F32, *tail)
        check(full, c, a.double().t() @ b.double() + 3.0)
    assert bool(torch.isnan(ws[nbytes // 4:]).all()), "written behind the workspace"


@pytest.mark.parametrize("M,N,K,epi", [(256, 512, 4096, nv.EPI_BIAS), (300, 1000, 1608, nv.EPI_NONE)])
@pytest.mark.parametrize("nbytes,offset", [(64, 0), (1 << 24, 4)])
def test_a_workspace_too_small_or_misaligned_with_an_epilogue_or_a_ragged_shape(M, N, K, epi, nbytes, offset):
    """The plain GEMM, bit for bit, and the workspace is left alone."""
    assert nv.load().axn_gemm_workspace_bytes(0, M, N, K) > 64
    gen = torch.Generator(device="cuda").manual_seed(N)
    x, w = (numbers(r, K, torch.bfloat16, gen, 16) for r in (M, N))
    bias = torch.randn(N, generator=gen, device="cuda")
    ws = torch.full((nbytes + 16,), 7, dtype=torch.uint8, device="cuda")
    got, want = (torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    args = (M, N, K, x.stride(0), w.stride(0), N, epi)
    nv.call("axn_gemm_fwd_ws", nv.ptr(x), nv.ptr(w), nv.ptr(bias), nv.ptr(got), None, nv.BF16, *args,
            ws.data_ptr() + offset, nbytes, nv.current_stream())
    nv.call("axn_gemm_fwd", nv.ptr(x), nv.ptr(w), nv.ptr(bias), nv.ptr(want), None, *args, nv.current_stream())
    assert torch.equal(got, want) and bool((ws == 7).all())


def test_the_longest_contractions():
    """A weight gradient over 2^31 - 8 tokens: the stages of 64 and their parts are counted past 2^31.  Zeros
    but for the first and the last rows and one in each part."""
    M = 2 ** 31 - 8
    if torch.cuda.mem_get_info()[0] < 90e9:
        pytest.skip("needs 69 GB")
    from axonn_amd import ops

    dy, x = (torch.zeros((M, 8), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    want = torch.zeros(8, 8, dtype=torch.float64, device="cuda")
    for i, row in enumerate([0, 1, M - 1, M - 2, M - 70] + [p * (M // 16) + 5 for p in range(16)]):
        dy[row, i % 8], x[row, (3 * i) % 8] = 1, i + 1
        want[i % 8, (3 * i) % 8] += i + 1
    assert torch.equal(ops.gemm_wgrad(dy, x, out_dtype=torch.float32).double(), want)


def backward(M, N, K, dtype=torch.bfloat16):
    """A call of the joint entry point on operands of ones."""
    dy, w, x = (torch.ones(s, dtype=dtype, device="cuda") for s in ((M, N), (N, K), (M, K)))
    dx, dw = torch.empty(M, K, dtype=dtype, device="cuda"), torch.empty(N, K, dtype=dtype, device="cuda")
    return lambda: nv.call("axn_gemm_bwd", nv.ptr(dy), nv.ptr(w), nv.ptr(x), nv.ptr(dx), nv.ptr(dw),
                           nv.dtype_code(dtype), M, N, K, N, K, K, K, K, 0, nv.dtype_code(dtype), nv.current_stream())


@pytest.mark.parametrize("M,N,K", [(2210, 2160, 2088), (3001, 10240, 2560),   # one of either order: the weight
                                   (1402, 2056, 4024), (3783, 2520, 3208)])   # gradient's tiles longer, or not
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_both_gradients_of_a_ragged_shape_in_one_launch(M, N, K, dtype):
    """Workgroups of both products side by side: exact, inside their views, equal to the separate calls."""
    names = launches(backward(M, N, K, dtype))
    assert len(names) == 1 and "gemm_edge_backward_kernel" in names[0][0], "this shape is meant to go together"
    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    dY, W, X = (numbers(r, c, dtype, gen, 16) for r, c in ((M, N), (N, K), (M, K)))
    code, ld, stream = nv.dtype_code(dtype), lambda t: t.stride(0), nv.current_stream()
    sfx = "" if dtype == torch.bfloat16 else "_f16"
    want_dx, want_dw = dY.double() @ W.double(), dY.double().t() @ X.double()
    for out, beta in ((dtype, 0), (dtype, 1), (torch.float32, 0), (torch.float32, 1)):
        fullx, dx = canvas(M, K, dtype)
        fullw, dw = canvas(N, K, out)
        dw.fill_(3.0)
        nv.call("axn_gemm_bwd", nv.ptr(dY), nv.ptr(W), nv.ptr(X), nv.ptr(dx), nv.ptr(dw), code, M, N, K, ld(dY),
                ld(W), ld(X), ld(dx), ld(dw), beta, nv.dtype_code(out), stream)
        alone_x, alone_w = torch.empty(M, K, dtype=dtype, device="cuda"), torch.full((N, K), 3.0, dtype=out, device="cuda")
        nv.call("axn_gemm_dgrad" + sfx, nv.ptr(dY), nv.ptr(W), nv.ptr(alone_x), M, N, K, ld(dY), ld(W), K, stream)
        nv.call("axn_gemm_wgrad" + sfx, nv.ptr(dY), nv.ptr(X), nv.ptr(alone_w), M, N, K, ld(dY), ld(X), K, beta,
                nv.dtype_code(out), stream)
        assert torch.equal(dx, alone_x) and torch.equal(dw, alone_w)
        check(fullx, dx, want_dx)
        check(fullw, dw, want_dw + 3.0 * beta)


def test_a_shape_is_planned_alike_whatever_was_asked_before():
    """Two ragged shapes with the same numbers of tiles and stages, one of them better in one launch: the plan
    that a thread keeps for the first is not taken for the second."""
    shapes = [(3783, 2520, 3080), (3783, 2520, 3208)]
    found = {}

    def plan(order):
        found[tuple(order)] = [launches(backward(*shapes[i])) for i in order]

    for order in ((0, 1), (1, 0)):   # a thread's plans are its own
        t = threading.Thread(target=plan, args=(order,))
        t.start()
        t.join()
    assert found[0, 1] == found[1, 0][::-1]
    assert [len(f) for f in found[0, 1]] != [1, 1], "the second is meant to differ from the first"


@pytest.mark.parametrize("op,M,N,K", [(0, 256, 512, 4160), (1, 128, 8896, 256), (2, 4160, 256, 384),   # an odd number of stages
                                      (0, 640, 3584, 8192)])                                         # 140 tiles
def test_a_workspace_too_small_for_whole_tiles_that_do_not_halve_or_are_many(op, M, N, K):
    """The plain GEMM, bit for bit."""
    assert nv.load().axn_gemm_workspace_bytes(op, M, N, K) > 64
    gen = torch.Generator(device="cuda").manual_seed(N)
    rows = {0: ((M, K), (N, K), (M, N)), 1: ((M, N), (N, K), (M, K)), 2: ((M, N), (M, K), (N, K))}[op]
    a, b = (torch.randn(s, generator=gen, device="cuda").bfloat16() for s in rows[:2])
    ws = torch.zeros(64, dtype=torch.uint8, device="cuda")
    got, want = (torch.empty(rows[2], dtype=torch.bfloat16, device="cuda") for _ in range(2))
    name, none, last = {0: ("axn_gemm_fwd", (None,), (nv.EPI_NONE,)), 1: ("axn_gemm_dgrad", (), ()),
                        2: ("axn_gemm_wgrad", (), (0, nv.BF16))}[op]
    dims = (M, N, K, a.shape[1], b.shape[1], rows[2][1])
    nv.call(name + "_ws", nv.ptr(a), nv.ptr(b), *none, nv.ptr(got), *none, nv.BF16, *dims, *last, nv.ptr(ws), 64,
            nv.current_stream())
    nv.call(name, nv.ptr(a), nv.ptr(b), *none, nv.ptr(want), *none, *dims, *last, nv.current_stream())
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K,none,bias,gelu", [(777, 14336, 1032, 256, 256, 128), (1591, 10752, 392, 256, 128, 128),
                                                  (2001, 4104, 2056, 256, 256, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_the_tile_of_a_ragged_forward_follows_its_epilogue(M, N, K, none, bias, gelu, dtype):
    """Whole numbers: the product, its sum with the bias and the saved pre-activation are exact on either tile,
    GELU as above."""
    gen = torch.Generator(device="cuda").manual_seed(M)
    X, W = (numbers(r, K, dtype, gen, 16) for r in (M, N))
    b = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
    product = X.double() @ W.double().t()
    sfx = "" if dtype == torch.bfloat16 else "_f16"
    for epi, tile, pre in ((nv.EPI_NONE, none, product), (nv.EPI_BIAS, bias, product + b),
                           (nv.EPI_BIAS_GELU, gelu, product + b)):
        fy, y = canvas(M, N, dtype)
        fz, z = canvas(M, N, dtype)
        call = lambda: nv.call(   # noqa: E731
            "axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(W), nv.ptr(b) if epi else None, nv.ptr(y),
            nv.ptr(z) if epi == nv.EPI_BIAS_GELU else None, M, N, K, X.stride(0), W.stride(0), y.stride(0), epi,
            nv.current_stream())
        name = launches(call)[0][0]
        assert "gemm_edge_kernel" in name and ("%d, %d" % (tile, tile) in name or "Li%dELi%dE" % (tile, tile) in name), name
        if epi == nv.EPI_BIAS_GELU:
            want = torch.nn.functional.gelu(pre)
            eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
            assert bool(((y.double() - want).abs() <= eps * want.abs() + 2e-7 * pre.abs().clamp(min=1)).all())
            check(fz, z, pre)
        else:
            check(fy, y, pre)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols,kc", [(3968, 3968, 1024), (1920, 4096, 1920), (640, 2176, 4096), (3200, 3200, 192)])
def test_outputs_of_whole_small_tiles_only(rows, cols, kc, dtype):
    """Multiples of 128 that are none of 256 take the tile with bounds that is estimated to be faster, or the
    small one: every product against 64 bits (one rounding to 16 bits of an fp32 sum)."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(rows + kc)
    draw = lambda *shape: torch.randn(*shape, generator=g, device="cuda").to(dtype)   # noqa: E731
    a, b = draw(rows, kc), draw(cols, kc)
    at, bt = a.t().contiguous(), b.t().contiguous()
    want = a.double() @ b.double().t()
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got in (ops.gemm_fwd(a, b)[0], ops.gemm_dgrad(a, bt), ops.gemm_wgrad(at, bt)):
        assert bool(((got.double() - want).abs() <= ulp * want.abs() + 1e-5 * want.abs().max()).all())
    y, z = ops.gemm_fwd(a * 0.05, b, bias=torch.ones(cols, device="cuda"), activation="gelu", save_z=True)
    pre = (a * 0.05).double() @ b.double().t() + 1
    assert bool(((z.double() - pre).abs() <= ulp * pre.abs() + 1e-5 * pre.abs().max()).all())
    gelu = torch.nn.functional.gelu(pre)
    assert bool(((y.double() - gelu).abs() <= ulp * gelu.abs() + 1e-5 * gelu.abs().max()).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,beta,dw_f32", [
    (649, 4032, 2176, 1, False), (2466, 4800, 1216, 0, False),      # longer tiles of dX, of dW first
    (2400, 4803, 1216, 1, True), (777, 6144, 4096, 0, True),        # any N; an fp32 dW
    (193, 9920, 5120, 0, False), (974, 50257, 768, 1, False),       # the fewest rows; ten parts
])
def test_both_gradients_in_one_launch_with_the_contraction_in_parts(M, N, K, beta, dw_f32, dtype):
    """Against the two calls, bit for bit, the operands in buffers of NaN, the outputs in canvases, the workspace
    exactly as large as it has to be."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(N)
    need = nv.load().axn_gemm_bwd_workspace_bytes(M, N, K, beta)
    assert need > 0
    dY = torch.full((M + 3, N + (-N) % 8 + 8), float("nan"), dtype=dtype, device="cuda")[:M]
    dY[:, N:N + (-N) % 8] = 0
    dY = dY[:, :N]
    dY.copy_(torch.randn(M, N, generator=g, device="cuda"))
    W, X = numbers(N, K, dtype, g, 8), numbers(M, K, dtype, g, 16)
    W.copy_(torch.randn(N, K, generator=g, device="cuda") * 0.1)
    dw_dtype = torch.float32 if dw_f32 else dtype
    fx, dx = canvas(M, K, dtype)
    fw, dw = canvas(N, K, dw_dtype)
    start = torch.ones(N, K, dtype=dw_dtype, device="cuda")
    if beta:
        dw.copy_(start)
    ws = torch.full((need // 4 + 64,), float("nan"), device="cuda")
    nv.call("axn_gemm_bwd_ws", nv.ptr(dY), nv.ptr(W), nv.ptr(X), nv.ptr(dx), nv.ptr(dw), nv.dtype_code(dtype), M, N, K,
            dY.stride(0), W.stride(0), X.stride(0), dx.stride(0), dw.stride(0), beta, nv.dtype_code(dw_dtype),
            nv.ptr(ws), need, nv.current_stream())
    assert bool(torch.isnan(ws[need // 4:]).all()), "written behind the workspace"
    want_dx = ops.gemm_dgrad(dY, W)
    want_dw = ops.gemm_wgrad(dY, X, out=start if beta else None, accumulate=bool(beta), out_dtype=dw_dtype)
    both = ops.gemm_bwd(dY, W, X, out_dtype=dw_dtype)
    assert torch.equal(both[0], want_dx)
    check(fx, dx, want_dx)
    check(fw, dw, want_dw)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,beta,dw_f32", [(256, 14336, 4096, 0, False), (768, 4864, 1792, 1, True),
                                               (1024, 6144, 4096, 0, False), (640, 6016, 3200, 0, True)])
def test_both_gradients_in_one_launch_of_whole_tiles(M, N, K, beta, dw_f32, dtype):
    """Against the kernels without bounds that the two calls take here."""
    test_both_gradients_in_one_launch_with_the_contraction_in_parts(M, N, K, beta, dw_f32, dtype)


@pytest.mark.parametrize("op,rows,cols,kc,beta,edge", [
    (2, 7040, 6528, 640, 1, False), (2, 3584, 4224, 384, 1, False), (2, 7040, 6528, 640, 0, False),
    (1, 6272, 7936, 1408, 0, False), (0, 7040, 4736, 3712, 0, False), (2, 2944, 2688, 768, 0, False),
    (0, 896, 14336, 4096, 0, True), (0, 8192, 5504, 2048, 0, True), (2, 2048, 5504, 8192, 0, True),
    (2, 2048, 5504, 8192, 1, False),
])
def test_the_tile_of_outputs_of_whole_small_tiles(op, rows, cols, kc, beta, edge):
    """Larger tiles with bounds where they are measured faster: clearly estimated so, and never to add to dW."""
    from launches import launches

    M, N, K = {0: (rows, cols, kc), 1: (rows, kc, cols), 2: (kc, rows, cols)}[op]
    a, b = {0: ((M, K), (N, K)), 1: ((M, N), (N, K)), 2: ((M, N), (M, K))}[op]
    a, b = torch.zeros(a, device="cuda").bfloat16(), torch.zeros(b, device="cuda").bfloat16()
    c = torch.zeros(rows, cols, device="cuda").bfloat16()
    call = lambda: nv.call("axn_gemm_any_n", op, nv.ptr(a), nv.ptr(b), None, nv.ptr(c), None, nv.BF16, M, N, K,   # noqa: E731
                           a.shape[1], b.shape[1], cols, nv.EPI_NONE, beta, nv.BF16, None, 0, nv.current_stream())
    assert ["edge" in name for name, _ in launches(call)][0] == edge
