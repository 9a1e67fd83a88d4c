"""The forward kernel of a few tokens at the sizes where it can go wrong: one token to the last
it takes, outputs around its 16-, 32- and 64-row workgroups, contractions shorter than a line,
ending inside one, and with fewer lines than a workgroup has waves.

Operands are small whole numbers (every sum is exact in fp32) inside buffers of NaN, so the
expected result is the float64 product rounded once and anything read outside shows."""

import pytest
import torch

from axonn_amd import _native as nv

pytestmark = pytest.mark.gpu

CANARY = 7.0


@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(8, 8), (24, 64), (1000, 72), (4096, 328), (4104, 1024), (8200, 264), (16392, 200),
                                 (72, 8200)])   # a longer contraction than it is picked for with a workspace
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_tokens_are_exact(M, N, K, dtype):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)

    def numbers(rows, cols):
        full = torch.full((rows + 1, cols + 8), float("nan"), dtype=dtype, device="cuda")
        full[:rows, :cols] = torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda").to(dtype)
        return full[:rows, :cols]

    X, W = numbers(M, K), numbers(N, K)
    bias = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
    product = X.double() @ W.double().t()
    sfx = "" if dtype == torch.bfloat16 else "_f16"
    stream = nv.current_stream()

    def canvas(t):
        full = torch.full((M + 1, N + 8), CANARY, dtype=t, device="cuda")
        return full, full[:M, :N]

    def check(full, view, want):
        assert torch.equal(view.double(), want.to(view.dtype).double())
        view.fill_(CANARY)
        assert torch.equal(full, torch.full_like(full, CANARY)), "written outside the output"

    full, y = canvas(dtype)
    for b, epi, want in ((None, nv.EPI_NONE, product), (bias, nv.EPI_BIAS, product + bias)):
        nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(W), nv.ptr(b), nv.ptr(y), None, M, N, K, X.stride(0),
                W.stride(0), y.stride(0), epi, stream)
        check(full, y, want)
    full32, y32 = canvas(torch.float32)
    nv.call("axn_gemm_fwd_f32out", nv.ptr(X), nv.ptr(W), nv.ptr(bias), nv.ptr(y32), None, nv.dtype_code(dtype), M, N,
            K, X.stride(0), W.stride(0), y32.stride(0), nv.EPI_BIAS, stream)
    check(full32, y32, product + bias)
    # GELU: the saved pre-activation is exact, Y within one rounding and the erf's 1.5e-7
    fz, z = canvas(dtype)
    nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(W), nv.ptr(bias), nv.ptr(y), nv.ptr(z), M, N, K, X.stride(0),
            W.stride(0), y.stride(0), nv.EPI_BIAS_GELU, stream)
    pre = product + bias
    want = torch.nn.functional.gelu(pre)
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert bool(((y.double() - want).abs() <= eps * want.abs() + 2e-7 * pre.abs().clamp(min=1)).all())
    check(fz, z, pre)


@pytest.mark.parametrize("M,N,K", [(32, 512, 28672), (16, 64, 14336), (64, 512, 5120)])
@pytest.mark.parametrize("nbytes,offset", [(16, 0), (1 << 24, 4)])
def test_a_workspace_too_small_or_misaligned_for_parts(M, N, K, nbytes, offset):
    """Streamed, as without one, bit for bit, and the workspace is left alone."""
    assert nv.load().axn_gemm_workspace_bytes(0, M, N, K) > 16
    gen = torch.Generator(device="cuda").manual_seed(K)
    X, W = (torch.randn(r, K, generator=gen, device="cuda").bfloat16() for r in (M, N))
    ws = torch.full((nbytes + 16,), 7, dtype=torch.uint8, device="cuda")
    got, want = (torch.empty(M, N, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    for out, where, size in ((got, ws.data_ptr() + offset, nbytes), (want, None, 0)):
        nv.call("axn_gemm_any_n", 0, nv.ptr(X), nv.ptr(W), None, nv.ptr(out), None, nv.BF16, M, N, K, K, K, N,
                nv.EPI_NONE, 0, nv.BF16, where, size, nv.current_stream())
    assert torch.equal(got, want) and bool((ws == 7).all())


@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(8, 8), (24, 64), (1000, 72), (4096, 328), (4104, 1024), (8192, 264), (8200, 264),
                                 (16392, 200), (72, 8200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_up_of_few_tokens(M, N, K, dtype):
    """Pre-activations of whole numbers are exact, the activation is the separate kernel's on them bit for bit,
    nothing is written outside the outputs, and random operands of up to 32 tokens give the two products' bits."""
    from axonn_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)

    def rows(n, fill):
        full = torch.full((n + 1, K + 8), float("nan"), dtype=dtype, device="cuda")
        full[:n, :K] = fill(n).to(dtype)
        return full[:n, :K]

    def whole(n):
        return torch.randint(-2, 3, (n, K), generator=gen, device="cuda")

    X, G, U = rows(M, whole), rows(N, whole), rows(N, whole)
    full = [torch.full((M + 1, N + 8), CANARY, dtype=dtype, device="cuda") for _ in range(3)]
    h, gate, up = (f[:M, :N] for f in full)
    nv.call("axn_gemm_swiglu_fwd_few", nv.ptr(X), nv.ptr(G), nv.ptr(U), nv.ptr(h), nv.ptr(gate), nv.ptr(up),
            nv.dtype_code(dtype), M, N, K, K + 8, K + 8, N + 8, nv.current_stream())
    assert torch.equal(gate.double(), (X.double() @ G.double().t()).to(dtype).double())
    assert torch.equal(up.double(), (X.double() @ U.double().t()).to(dtype).double())
    assert torch.equal(h, ops.swiglu_fwd(gate.contiguous(), up.contiguous()))
    for f, view in zip(full, (h, gate, up)):
        view.fill_(CANARY)
        assert torch.equal(f, torch.full_like(f, CANARY)), "written outside the output"

    def random(n):
        return torch.randn(n, K, generator=gen, device="cuda") * 0.1

    X, G, U = rows(M, random), rows(N, random), rows(N, random)
    h, none_g, none_u = ops.gemm_swiglu_fwd(X, G, U, save=False, few=True)
    assert none_g is None and none_u is None
    sfx = "" if dtype == torch.bfloat16 else "_f16"
    for w, out in ((G, gate), (U, up)):   # (without a workspace: always the stream)
        nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(w), None, nv.ptr(out), None, M, N, K, K + 8, K + 8, N + 8,
                nv.EPI_NONE, nv.current_stream())
    want = ops.swiglu_fwd(gate.contiguous(), up.contiguous())
    if M <= 32:
        assert torch.equal(h, want)
    else:   # other order of sums: a rounding of each factor and of the product
        eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        assert ((h.double() - want.double()).norm() / want.double().norm()) < 4 * eps


@pytest.mark.parametrize("M", [33, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(8200, 8), (8200, 264), (9000, 72), (11008, 1160), (16392, 200), (8256, 4096)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gate_up_of_33_to_64_tokens_gives_the_bits_of_the_two_products(M, N, K, dtype):
    """Over more than 8192 outputs, where a wave has one slot for the tokens: lines of the contraction on one to
    four waves, one to many a wave."""
    from axonn_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(M + N + K)
    X, G, U = (torch.randn(n, K, generator=gen, device="cuda").to(dtype) * s for n, s in ((M, 1), (N, 0.1), (N, 0.1)))
    h, gate, up = ops.gemm_swiglu_fwd(X, G, U, save=True, few=True)
    sfx = "" if dtype == torch.bfloat16 else "_f16"
    want = [torch.empty_like(h), torch.empty_like(h)]
    for w, out in zip((G, U), want):   # (without a workspace: always the stream)
        nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(w), None, nv.ptr(out), None, M, N, K, K, K, N, nv.EPI_NONE,
                nv.current_stream())
    assert torch.equal(gate, want[0]) and torch.equal(up, want[1])
    assert torch.equal(h, ops.swiglu_fwd(*want))
