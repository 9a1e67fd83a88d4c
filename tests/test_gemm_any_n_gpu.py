"""16-bit products with a number of output features that is no multiple of 8: every element against 64
bits, and nothing written behind the outputs."""

import pytest
import torch

from axonn_amd import _native as nv
from launches import launches

pytestmark = pytest.mark.gpu


def close(got, want, dtype):
    """One rounding to the result's type on top of fp32 sums (16-bit products are exact in fp32)."""
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -22}[dtype]
    scale = want.abs().max()
    return bool(((got.double() - want).abs() <= ulp * want.abs() + 1e-5 * scale).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 8), (3, 9, 72), (16, 1003, 512), (40, 4099, 1024),        # streamed forward
    (129, 257, 64), (256, 511, 2048), (300, 1001, 4096),             # contractions in parts
    (512, 20001, 768), (2048, 16391, 256),                           # full rounds and a rest
])
def test_products_against_64_bits(M, N, K, dtype):
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    X = torch.randn(M, K, generator=g, device="cuda").to(dtype)
    W = (torch.randn(N, K, generator=g, device="cuda") * 0.1).to(dtype)
    dY = torch.randn(M, N, generator=g, device="cuda").to(dtype)
    b = torch.randn(N, generator=g, device="cuda")
    X64, W64, dY64 = X.double(), W.double(), dY.double()
    pre = X64 @ W64.t()
    assert close(ops.gemm_fwd(X, W)[0], pre, dtype)
    y, z = ops.gemm_fwd(X, W, bias=b, activation="gelu", save_z=True)
    assert y.is_contiguous() and close(z, pre + b.double(), dtype)
    assert close(y, torch.nn.functional.gelu(pre + b.double()), dtype)
    assert close(ops.gemm_fwd(X, W, bias=b, out_f32=True)[0], pre + b.double(), torch.float32)
    wide = torch.full((M, N + 5), float("nan"), dtype=dtype, device="cuda")
    wide[:, 2:N + 2] = dY                                   # rows of an odd stride and offset
    dx, dw = ops.gemm_bwd(wide[:, 2:N + 2], W, X)
    assert close(dx, dY64 @ W64, dtype) and close(dw, dY64.t() @ X64, dtype)
    assert torch.equal(dx, ops.gemm_dgrad(dY, W)) and torch.equal(dw, ops.gemm_wgrad(dY, X))
    acc = torch.ones(N * K + 1, device="cuda")[1:]           # a flat buffer's view at an odd offset
    ops.gemm_wgrad(dY, X, out=acc, accumulate=True)
    assert close(acc.view(N, K), 1 + dY64.t() @ X64, torch.float32)
    before = dw.double()                                     # rounded once already
    ops.gemm_wgrad(dY, X, out=dw, accumulate=True)
    assert close(dw, before + dY64.t() @ X64, dtype)


def test_forward_leaves_the_neighbours_alone():
    """Y at an odd row stride inside a larger buffer: the elements between its rows stay."""
    M, N, K, ld = 300, 1003, 128, 1007
    X, W = (torch.randn(n, K, device="cuda").bfloat16() for n in (M, N))
    buf = torch.full((M * ld + 64,), 7.0, device="cuda").bfloat16()
    nv.call("axn_gemm_any_n", 0, nv.ptr(X), nv.ptr(W), None, nv.ptr(buf), None, nv.BF16, M, N, K, K, K, ld,
            nv.EPI_NONE, 0, nv.BF16, None, 0, nv.current_stream())
    assert close(buf[:M * ld].view(M, ld)[:, :N], X.double() @ W.double().t(), torch.bfloat16)
    assert bool((buf[:M * ld].view(M, ld)[:, N:] == 7).all()) and bool((buf[M * ld:] == 7).all())


@pytest.mark.parametrize("M,N,K", [(16, 1024, 64), (128, 128, 64), (512, 1024, 128), (2304, 2048, 64),
                                   (3072, 2048, 64), (4096, 4096, 64), (4352, 4096, 64), (256, 512, 4096)])
@pytest.mark.parametrize("out_f32", [False, True])
def test_forward_of_whole_tiles_at_odd_row_strides(M, N, K, out_f32):
    """Rows of Y that start anywhere are stored by kernels that do not take them for 16-byte aligned, whatever
    the shape: streamed, each tile size, full rounds and a rest, a contraction in parts.  Exact whole numbers."""
    g = torch.Generator(device="cuda").manual_seed(M)
    X, W = (torch.randint(-2, 3, (n, K), generator=g, device="cuda").bfloat16() for n in (M, N))
    b = torch.randint(-3, 4, (N,), generator=g, device="cuda").float()
    want = X.double() @ W.double().t() + b
    nbytes = nv.load().axn_gemm_workspace_bytes(0, M, N, K)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device="cuda")
    dtype = torch.float32 if out_f32 else torch.bfloat16
    for ld in (N + 1, N + 3, N + 8):
        buf = torch.full((M * ld + 64,), 7.0, device="cuda", dtype=dtype)

        def forward():
            nv.call("axn_gemm_any_n", 0, nv.ptr(X), nv.ptr(W), nv.ptr(b), nv.ptr(buf), None, nv.BF16, M, N, K, K, K,
                    ld, nv.EPI_BIAS, 0, nv.dtype_code(dtype), nv.ptr(ws), nbytes, nv.current_stream())

        names = [name for name, _ in launches(forward)]
        last = names[-1]   # of parts: the pass that adds them, with element-aligned rows
        if ld % 8:
            assert "edge_kernel" in last or "stream_kernel" in last or last.endswith("Lb1EEEvPKfNS_8GemmArgsE"), names
        assert torch.equal(buf[:M * ld].view(M, ld)[:, :N].double(), want.to(dtype).double())
        assert bool((buf[:M * ld].view(M, ld)[:, N:] == 7).all()) and bool((buf[M * ld:] == 7).all())


@pytest.mark.parametrize("M,N,K", [(256, 512, 4096), (129, 392, 4104), (300, 1001, 4096), (64, 520, 8192)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("narrow", [False, True])
def test_fp32_results_of_a_contraction_in_parts(M, N, K, dtype, narrow):
    """The pass that adds the parts with an fp32 result: bias (fp32 or of the operands' type), GELU with the
    pre-activation kept.  Whole numbers: sums are exact, GELU within the erf's 1.5e-7."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    X, W = (torch.randint(-2, 3, (n, K), generator=g, device="cuda").to(dtype) for n in (M, N))
    b = torch.randint(-3, 4, (N,), generator=g, device="cuda").to(dtype if narrow else torch.float32)
    nbytes = nv.load().axn_gemm_workspace_bytes(0, M, N, K)
    assert nbytes > 0, "this shape is meant to be split"
    ws = torch.full((nbytes // 4 + 8,), float("nan"), device="cuda")
    y, z = torch.empty(M, N, device="cuda"), torch.empty(M, N, dtype=dtype, device="cuda")
    pre = X.double() @ W.double().t() + b.double()
    for epi in (nv.EPI_BIAS, nv.EPI_BIAS_GELU):
        def forward():
            nv.call("axn_gemm_any_n", 0, nv.ptr(X), nv.ptr(W), nv.ptr(b), nv.ptr(y), nv.ptr(z), nv.dtype_code(dtype), M,
                    N, K, K, K, N, epi | (nv.BIAS_16BIT if narrow else 0), 0, nv.F32, nv.ptr(ws), nbytes,
                    nv.current_stream())

        assert "splitk_reduce_kernel" in launches(forward)[-1][0]
        if epi == nv.EPI_BIAS:
            assert torch.equal(y.double(), pre)
        else:
            want = torch.nn.functional.gelu(pre)
            assert bool(((y.double() - want).abs() <= 2.0 ** -23 * want.abs() + 2e-7 * pre.abs().clamp(min=1)).all())
            assert torch.equal(z, pre.to(dtype))
    assert bool(torch.isnan(ws[nbytes // 4:]).all()), "written behind the workspace"


@pytest.mark.parametrize("M,N,ld", [(1, 1, 1), (3, 17, 17), (5, 24, 31), (70, 1003, 1005)])
def test_pad_rows(M, N, ld):
    from axonn_amd import ops

    src = torch.randn(M, ld, device="cuda").half()[:, :N]
    out = ops._pad_rows(src)
    assert out.shape == (M, N + (-N) % 8)
    assert torch.equal(out[:, :N], src) and not out[:, N:].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(5, 1003, 64), (40, 72, 512), (256, 512, 256), (130, 264, 4096),
                                   (129, 1001, 64), (2304, 4096, 128)])
def test_bias_of_the_operands_type_equals_its_fp32_copy(M, N, K, dtype):
    """Streamed, whole, ragged and split products; a bias at an odd offset is widened beforehand."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(N)
    X, W = (torch.randn(n, K, generator=g, device="cuda").to(dtype) for n in (M, N))
    b = torch.randn(N + 1, generator=g, device="cuda").to(dtype)
    for bias in (b[:N], b[1:]):
        for act in (None, "gelu"):
            got = ops.gemm_fwd(X, W, bias=bias, activation=act, save_z=True)
            want = ops.gemm_fwd(X, W, bias=bias.float(), activation=act, save_z=True)
            assert torch.equal(got[0], want[0])
            assert act is None or torch.equal(got[1], want[1])
    pre = X.double() @ W.double().t() + b[:N].double()
    assert close(ops.gemm_fwd(X, W, bias=b[:N])[0], pre, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(65, 1, 64), (65, 7, 64), (129, 127, 64), (300, 129, 128), (257, 255, 72),
                                   (700, 1016, 64), (2100, 4093, 64), (3000, 7003, 64), (2048, 16385, 64)])
def test_odd_rows_hold_what_even_rows_hold(M, N, K, dtype):
    """The forward's output at odd row strides, on every tile and with every number of columns behind the last
    whole vector: the bits of the same product at an even stride, and nothing between the rows is touched."""
    g = torch.Generator(device="cuda").manual_seed(N)
    X, W = (torch.randn(n, K, generator=g, device="cuda").to(dtype) for n in (M, N))

    def product(ld):
        buf = torch.full((M * ld + 64,), 7.0, device="cuda", dtype=dtype)
        nv.call("axn_gemm_any_n", 0, nv.ptr(X), nv.ptr(W), None, nv.ptr(buf), None, nv.dtype_code(dtype), M, N, K, K,
                K, ld, nv.EPI_NONE, 0, nv.dtype_code(dtype), None, 0, nv.current_stream())
        assert bool((buf[M * ld:] == 7).all())
        rows = buf[:M * ld].view(M, ld)
        assert bool((rows[:, N:] == 7).all())
        return rows[:, :N]

    even = product(N + N % 2)
    assert close(even, X.double() @ W.double().t(), dtype)
    assert torch.equal(product(N + 1 - N % 2), even)
    assert torch.equal(product(N + 5 - N % 2), even)


@pytest.mark.parametrize("M,N,ld", [(3, 4097, 4103), (70, 5000, 5000), (300, 4159, 4160), (9, 4160, 4161)])
def test_wide_rows_are_padded_to_whole_lines(M, N, ld):
    """Rows of 4096 elements and more start on 128-byte lines, with zeros up to the next row."""
    from axonn_amd import ops

    src = torch.randn(M, ld, device="cuda").bfloat16()[:, :N]
    out = ops._pad_rows(src)
    assert out.shape == (M, N + (-N) % 8) and out.stride(0) == N + (-N) % 64
    assert torch.equal(out[:, :N], src)
    assert not out.as_strided((M, out.stride(0)), (out.stride(0), 1))[:, N:].any()
    w, x = torch.randn(N, 64, device="cuda").bfloat16(), torch.randn(M, 64, device="cuda").bfloat16()
    dx, dw = ops.gemm_bwd(src, w, x) if N % 8 else (ops._dgrad_any_n(out, w, N),
                                                   ops._wgrad_any_n(out, x, N, None, False, src.dtype))
    for got, want in ((dx, src.double() @ w.double()), (dw, src.double().t() @ x.double())):
        # bf16 rounding of the result and fp32 sums
        assert float((got.double() - want).norm() / want.norm()) < 2.0 ** -8


@pytest.mark.parametrize("M,N,K,odd", [(70, 689, 1192, False), (80, 1013, 448, False), (81, 1013, 448, True),
                                       (300, 50257, 64, True)])
def test_rows_from_which_odd_strides_take_the_exchange(M, N, K, odd):
    from launches import launches

    X, W = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(N, K, device="cuda").bfloat16()
    out, even = torch.empty(M, N, device="cuda").bfloat16(), torch.empty(M, N + 1, device="cuda").bfloat16()

    def call(to):
        nv.call("axn_gemm_any_n", 0, nv.ptr(X), nv.ptr(W), None, nv.ptr(to), None, nv.BF16, M, N, K, K, K, to.shape[1],
                nv.EPI_NONE, 0, nv.BF16, None, 0, nv.current_stream())

    def kernels(to):
        return [name for name, _ in launches(lambda: call(to))]

    assert (kernels(out) != kernels(even)) == odd
    call(out)
    call(even)
    assert torch.equal(out, even[:, :N])
