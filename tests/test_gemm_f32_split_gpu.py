"""fp32 products formed from bf16 parts (2^32 multiply-adds and more), whole and ragged, with vector and
single-element accesses, with the contraction in one part and in several, against 64 bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def bound(K):
    """Norm-wise: the dropped products are under 3 * 2^-24 of a product, the accumulators round once
    per 32 contraction indices (at random), and the outputs once; twice that."""
    return 2.0 * 2.0 ** -24 * (4 + (K / 32) ** 0.5)


def err(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("M,N,K", [
    (2048, 4096, 1024), (2052, 4100, 1028), (2047, 4099, 1027),    # whole, ragged, no vector access
    (256, 4096, 4128), (260, 4100, 4100), (257, 4099, 4103),       # parts, the last one shorter
    (8192, 16384, 32), (8196, 16388, 36), (33, 16384, 8192),       # one stage, and a rest; few rows
])
def test_products_against_64_bits(M, N, K):
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    X, W, dY = (torch.randn(s, generator=g, device="cuda") for s in ((M, K), (N, K), (M, N)))
    b = torch.randn(N, generator=g, device="cuda")
    z64 = X.double() @ W.double().t() + b.double()
    y, z = ops.gemm_fwd(X, W, bias=b, activation="gelu", save_z=True)
    assert err(z, z64) < bound(K)
    assert err(y, torch.nn.functional.gelu(z64)) < bound(K)
    assert err(ops.gemm_fwd(X, W)[0], z64 - b.double()) < bound(K)
    assert err(ops.gemm_dgrad(dY, W), dY.double() @ W.double()) < bound(N)
    dw64 = dY.double().t() @ X.double()
    dw = ops.gemm_wgrad(dY, X)
    assert err(dw, dw64) < bound(M)
    ops.gemm_wgrad(dY, X, out=dw, accumulate=True)
    assert err(dw, 2 * dw64) < bound(M)


@pytest.mark.parametrize("M,N,K", [(2048, 4096, 512), (512, 2048, 4096)])
def test_infinities_and_nans_stay_where_they_belong(M, N, K):
    """An infinity has no bf16 remainder (inf - inf): results that hold one are those of plain
    fp32 arithmetic, the others are untouched; the largest floats round to a bf16 infinity."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(3)
    X, W = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    X[3, 5], X[70, 9], X[M - 1, K - 1] = float("inf"), float("nan"), -float("inf")
    W[11, 7] = float("inf")
    X[200, 8] = 3.4e38           # above the largest bf16
    W[:, 8] *= 2.0 ** -20
    want = X.double() @ W.double().t()
    got = ops.gemm_fwd(X, W)[0]
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()] > 0, want[want.isinf()] > 0)
    row = got[200].double()
    ok = row.isfinite()
    assert err(row[ok], want[200][ok]) < bound(K)
    plain = torch.ones(M, dtype=torch.bool, device="cuda")
    plain[[3, 70, 200, M - 1]] = False
    cols = torch.ones(N, dtype=torch.bool, device="cuda")
    cols[11] = False
    assert err(got[plain][:, cols], want[plain][:, cols]) < bound(K)


@pytest.mark.parametrize("exponent", [-120, -100, 60])
def test_magnitudes_beyond_the_parts_keep_full_precision(exponent):
    """A float of 2^-120 has its third part below bf16's range."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(4)
    X = torch.randn(2048, 1024, generator=g, device="cuda")
    W = torch.randn(2048, 1024, generator=g, device="cuda")
    want = X.double() @ W.double().t()
    got = ops.gemm_fwd(X * 2.0 ** exponent, W)[0]
    assert err(got.double() * 2.0 ** -exponent, want) < 1e-6


@pytest.mark.parametrize("M,N,K", [(2050, 2049, 1030), (2052, 2052, 1032)])
@pytest.mark.parametrize("exponent", [-132, -140, -145])
def test_subnormal_operands_are_not_taken_as_zero(M, N, K, exponent):
    """The bf16 instruction flushes them. Whole multiples of 2^exponent, sums below 2^(exponent + 20):
    every one is a multiple of 2^-149, so the exact results are floats."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(5)
    X = torch.randint(-2, 3, (M, K), generator=g, device="cuda").float()
    W = torch.randint(-2, 3, (N, K), generator=g, device="cuda").float()
    X[7], W[:, 9] = 0, 0
    tiny = (X.double() * 2.0 ** exponent).float()
    got = ops.gemm_fwd(tiny, W)[0]
    assert torch.equal(got.double() * 2.0 ** -exponent, X.double() @ W.double().t())
    mixed = X.clone()
    mixed[:, 1:] = 0              # one subnormal column among zeros, split over parts
    mixed[:, 0] = tiny[:, 0]
    assert torch.equal(ops.gemm_fwd(mixed, W)[0].double(), mixed.double() @ W.double().t())


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 1024), (2050, 2049, 1030), (260, 4100, 4100)])
@pytest.mark.parametrize("small,large", [(-118, 60), (-122, 70), (-130, 100), (-145, 120)])
def test_small_operands_times_large_ones_keep_full_precision(M, N, K, small, large):
    """Numbers around 2^small times ones around 2^large, in one operand or the other: results of ordinary
    magnitude, of numbers whose last bits lie below bf16's multiples of 2^-133."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(6)
    X, W, dY = (torch.randn(s, generator=g, device="cuda").double() for s in ((M, K), (N, K), (M, N)))
    low = lambda t: (t * 2.0 ** small).float()   # noqa: E731
    high = lambda t: (t * 2.0 ** large).float()   # noqa: E731
    for got, a, b in ((ops.gemm_fwd(low(X), high(W))[0], low(X), high(W).t()),
                      (ops.gemm_fwd(high(X), low(W))[0], high(X), low(W).t()),
                      (ops.gemm_dgrad(high(dY), low(W)), high(dY), low(W)),
                      (ops.gemm_wgrad(low(dY), high(X)), low(dY).t(), high(X))):
        assert err(got, a.double() @ b.double()) < bound(max(M, N, K))


def test_a_small_operand_beside_ordinary_ones():
    """One term of a sum is a subnormal times a large number, the others are ordinary: the result is neither
    small nor zero, and without the one term it is 1."""
    from axonn_amd import ops

    X, W = torch.zeros(2048, 1024, device="cuda"), torch.zeros(2048, 1024, device="cuda")
    X[:, 0], W[:, 0] = 1, 1
    X[:, 9], W[:, 9] = 2.0 ** -140, 2.0 ** 120
    W[1000:, 9] = 2.0 ** 126
    want = X.double() @ W.double().t()
    assert torch.equal(ops.gemm_fwd(X, W)[0], want.float())
    assert torch.equal(ops.gemm_fwd(W, X)[0], want.t().float())


def test_large_operands_beside_ordinary_ones():
    """Numbers of 2^16 and more, nothing small: whole multiples, exact either way."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(9)
    X, W = (torch.randint(-7, 8, (2050, 1030), generator=g, device="cuda").float() for _ in range(2))
    X *= 2.0 ** 17
    assert torch.equal(ops.gemm_fwd(X, W)[0].double(), X.double() @ W.double().t())


def test_products_of_two_small_operands():
    """2^-70 times 2^-70: whole multiples of 2^-140, exact in subnormal floats."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(7)
    X, W = (torch.randint(-2, 3, s, generator=g, device="cuda").float() for s in ((2050, 1030), (2049, 1030)))
    got = ops.gemm_fwd(X * 2.0 ** -70, W * 2.0 ** -70)[0]
    assert torch.equal(got.double() * 2.0 ** 140, X.double() @ W.double().t())


def test_a_result_of_one_product():
    """Rows with one non-zero element: the dropped products are under 2^-24 of the product, the sum of the two
    accumulators rounds once."""
    from axonn_amd import ops

    g = torch.Generator(device="cuda").manual_seed(8)
    X, W = torch.zeros(2048, 1024, device="cuda"), torch.randn(2048, 1024, generator=g, device="cuda")
    X[torch.arange(2048), torch.randint(0, 1024, (2048,), generator=g, device="cuda").cpu()] = \
        torch.randn(2048, generator=g, device="cuda")
    want = X.double() @ W.double().t()
    got = ops.gemm_fwd(X, W)[0]
    assert bool(((got.double() - want).abs() <= 2.0 * 2.0 ** -24 * want.abs()).all())


@pytest.mark.parametrize("M,N,K", [(128, 128, 1 << 18), (300, 2048, 8192), (8, 8192, 65536)])
def test_few_tiles_without_a_workspace_are_left_to_the_native_kernel(M, N, K):
    """A workgroup or a few would walk the whole contraction.  Half of the rows are below 2^32 multiply-adds:
    the same bits."""
    from axonn_amd import _native as nv

    g = torch.Generator(device="cuda").manual_seed(10)
    X, W = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")

    def forward(rows):
        y = torch.empty(rows, N, device="cuda")
        nv.call("axn_gemm_fwd_f32", nv.ptr(X), nv.ptr(W), None, nv.ptr(y), None, rows, N, K, nv.EPI_NONE,
                nv.current_stream())
        return y

    assert M // 2 * N * K < 2 ** 32
    assert torch.equal(forward(M)[:M // 2], forward(M // 2))
    # four waves share a tile, the native instruction rounds once per 4 indices (at random); twice that
    assert err(forward(M), X.double() @ W.double().t()) < 2.0 * 2.0 ** -24 * (4 + (K / 16) ** 0.5)
