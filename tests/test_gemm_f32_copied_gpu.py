"""The native fp32 products whose operands are copied to LDS ahead, against the kernel that loads them directly (which
takes operands that do not start on 16 bytes): the same order of sums, so the same bits."""

import pytest
import torch

from axonn_amd import ops

from launches import launches

pytestmark = pytest.mark.gpu


def _placed(t, shift):
    """`t` inside a buffer of NaN, `shift` elements behind a 16-byte boundary."""
    n = t.numel()
    buf = torch.full((n + 512,), float("nan"), device="cuda")
    view = buf[256 + shift:256 + shift + n].view(t.shape)
    view.copy_(t)
    return view


# tokens, input features, output features: 16, 32 and 64 square tiles, waves of a tile together (contractions of 256 and
# 2048 on) and apart, whole tiles and rests of 4 on, contractions that end in a chunk, a unit, a block and a piece
@pytest.mark.parametrize("M,K,N", [
    (64, 1024, 4096), (64, 4096, 1024), (1, 512, 512), (17, 772, 1028), (40, 1100, 260), (16, 1024, 1024),
    (256, 1024, 4096), (260, 996, 4100), (1000, 600, 1200), (1004, 2052, 1028), (33, 2212, 4100), (132, 260, 2052),
    (68, 5120, 4096), (2001, 900, 1000), (259, 388, 1032), (8, 16380, 4), (3236, 768, 192), (512, 68, 8192), (76, 296, 548),
])
def test_products_are_those_of_direct_loads(M, K, N):
    g = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, w, dy = (torch.randn(s, generator=g, device="cuda") for s in ((M, K), (N, K), (M, N)))
    b = torch.randn(N, generator=g, device="cuda")
    results = []
    for shift in (0, 1):
        X, W, B, dY = (_placed(t, shift) for t in (x, w, b, dy))
        y, z = ops.gemm_fwd(X, W, B, "gelu", save_z=True)
        dw = torch.ones(N, K, device="cuda")
        ops.gemm_wgrad(dY, X, out=dw, accumulate=True)
        results.append((y, z, ops.gemm_fwd(X, W)[0], ops.gemm_dgrad(dY, W), ops.gemm_wgrad(dY, X), dw))
    for a, c in zip(*results):
        assert torch.equal(a, c)
    # every product is rounded to 2^-24 of itself and added in steps of 4: the root of their number, twice
    z64 = x.double() @ w.double().t() + b.double()
    assert float((results[0][1] - z64).norm() / z64.norm()) < 2 * 2.0 ** -24 * (4 + (K / 4) ** 0.5)


@pytest.mark.parametrize("M,K,N,copied", [
    (64, 1024, 4096, (True, True, True)), (64, 4096, 1024, (True, True, True)), (1000, 600, 1200, (True, True, True)),
    (1001, 600, 1200, (True, True, True)), (64, 1022, 4096, (False, False, False)), (916, 164, 336, (False, True, False)), (24, 3712, 6080, (True, True, False)),
])
def test_the_kernel_that_is_picked(M, K, N, copied):
    x, w, dy = (torch.randn(s, device="cuda") for s in ((M, K), (N, K), (M, N)))
    calls = (lambda: ops.gemm_fwd(x, w), lambda: ops.gemm_dgrad(dy, w), lambda: ops.gemm_wgrad(dy, x))
    for call, want in zip(calls, copied):
        names = [name for name, _ in launches(call)]
        assert any("gemm_f32_copied_kernel" in n for n in names) == want, names


def test_infinities_and_nans_stay_where_they_belong():
    x, w = torch.randn(64, 1028, device="cuda"), torch.randn(512, 1028, device="cuda")
    x[3, 1027], x[63, 0], w[511, 1027], w[5, 17] = float("inf"), float("nan"), -float("inf"), float("nan")
    want, got = x.double() @ w.double().t(), ops.gemm_fwd(x, w)[0]
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    back, want = ops.gemm_dgrad(want.float().nan_to_num(1, 2, 3), w), want.float().nan_to_num(1, 2, 3).double() @ w.double()
    assert torch.equal(back.isnan(), want.isnan()) and torch.equal(back.isinf(), want.isinf())


@pytest.mark.parametrize("tokens,out_features,in_features,copied", [
    (22, 128, 128, False), (30, 1088, 128, False), (32, 64, 320, False), (21, 2240, 224, False), (24, 320, 1472, False),   # one unit a wave
    (32, 512, 1408, True), (18, 240, 3840, True), (64, 1024, 1024, True),
])
def test_few_small_weight_gradients_are_loaded_directly(tokens, out_features, in_features, copied):
    dy, x = torch.randn(tokens, out_features, device="cuda"), torch.randn(tokens, in_features, device="cuda")
    out = torch.randn(out_features, in_features, device="cuda")
    want = out.double() + dy.double().t() @ x.double()
    dw = out.clone()
    assert any("gemm_f32_copied_kernel" in n for n, _ in launches(lambda: ops.gemm_wgrad(dy, x, out=dw, accumulate=True))) == copied
    got = ops.gemm_wgrad(dy, x, out=out, accumulate=True)
    assert float((got.double() - want).norm() / want.norm()) < 2 * 2.0 ** -24 * (5 + (tokens / 4) ** 0.5)
