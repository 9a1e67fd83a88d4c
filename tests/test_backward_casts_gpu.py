"""What the backward of a layer with fp32 parameters under autocast, and of one with 16-bit bias, writes in the type it is
wanted in: bit for bit what a cast before or behind the same kernels gives."""

import pytest
import torch

from axonn_amd import _native as nv
from axonn_amd import ops
from launches import launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N", [(1, 8), (5, 136), (127, 1000), (129, 128), (300, 2056), (3001, 520)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gelu", [False, True])
def test_an_fp32_gradient_is_rounded_on_the_way(M, N, dtype, gelu):
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    dy = torch.randn(M, N, generator=gen, device="cuda") * 100
    dy[0, 0], dy[-1, -1] = 1e6, -1e-9   # infinite and subnormal (or zero) in fp16
    z = torch.randn(M, N, generator=gen, device="cuda").to(dtype) if gelu else None
    dz, db = ops.dgelu_dbias(dy, z, dtype=dtype, dbias_dtype=torch.float32)
    want_dz, want_db = ops.dgelu_dbias(dy.to(dtype), z)
    assert dz.dtype == dtype and torch.equal(dz, want_dz) and torch.equal(db, want_db)
    alone, none = ops.dgelu_dbias(dy, z, want_dbias=False, dtype=dtype)
    assert none is None and torch.equal(alone, want_dz)
    strided = torch.full((M, N + 8), float("nan"), device="cuda")
    strided[:, :N] = dy
    assert torch.equal(ops.dgelu_dbias(strided[:, :N], z, dtype=dtype)[0], want_dz)
    # the bias gradient in the operands' type
    for g in (dy, dy.to(dtype)):
        dz, db16 = ops.dgelu_dbias(g, z, dtype=dtype, dbias_dtype=dtype)
        assert db16.dtype == dtype and torch.equal(db16, want_db.to(dtype)) and torch.equal(dz, want_dz)


def test_combinations_that_are_refused():
    a, ws = torch.zeros(64, 64, device="cuda"), torch.zeros(64 * 64, device="cuda")
    call = lambda dz, code, db, beta: nv.call(   # noqa: E731
        "axn_dgelu_dbias", nv.ptr(a), None, nv.ptr(dz), code, nv.ptr(db), 64, 64, 64, beta, nv.ptr(ws), 64 * 64 * 4,
        nv.current_stream())
    for dz, code, db, beta in ((None, nv.F16 | nv.DY_F32, a, 0), (a, nv.F32 | nv.DY_F32, a, 0), (a, nv.F16, a, 0),
                               (None, nv.F32 | nv.DBIAS_16BIT, a, 0), (None, nv.F16 | nv.DBIAS_16BIT, a, 1)):
        with pytest.raises(nv.AxnError):
            call(dz, code, db, beta)
    w = torch.zeros(64, 64, device="cuda").half()
    with pytest.raises(nv.AxnError, match="needs the workspace"):
        nv.call("axn_gemm_any_n", 1, nv.ptr(w), nv.ptr(w), None, nv.ptr(a), None, nv.F16, 64, 64, 64, 64, 64, 64, 0, 0,
                nv.F32 | nv.ROUNDED, None, 0, nv.current_stream())


@pytest.mark.parametrize("M,N,K", [(300, 8200, 2568), (3001, 2560, 640), (454, 1600, 2048), (512, 8192, 3584), (70, 1001, 520)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_an_input_gradient_rounded_and_stored_as_fp32(M, N, K, dtype):
    gen = torch.Generator(device="cuda").manual_seed(N)
    dy, w = (torch.randn(s, generator=gen, device="cuda").to(dtype) for s in ((M, N), (N, K)))
    got, want = ops.gemm_dgrad(dy, w, widen=True), ops.gemm_dgrad(dy, w)
    assert torch.equal(got.float(), want.float())
    if N % 8 == 0 and nv.load().axn_gemm_workspace_bytes(1, M, N, K):
        assert got.dtype == torch.float32
        names = [name for name, _ in launches(lambda: ops.gemm_dgrad(dy, w, widen=True))]
        assert len(names) == 2 and ("splitk_reduce" in names[1] or "widen_kernel" in names[1]), names


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("gelu", [None, "gelu"])
@pytest.mark.parametrize("grad_dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_gradients_of_an_autocast_layer_have_the_types_of_what_they_belong_to(bias, gelu, grad_dtype):
    from axonn_amd.intra_layer import Linear

    gen = torch.Generator(device="cuda").manual_seed(7)
    layer = Linear(1600, 2048, bias=bias, fused_activation=gelu).cuda()
    x = torch.randn(3, 151, 1600, generator=gen, device="cuda").requires_grad_()
    with torch.autocast("cuda", dtype=torch.float16):
        y = layer(x)
    y = y.to(grad_dtype)
    dy = torch.randn(y.shape, generator=gen, device="cuda").to(grad_dtype)
    y.backward(dy)
    x2 = x.detach().half().double().requires_grad_()
    w = layer.weight.detach().half().double().view(2048, 1600).requires_grad_()
    y2 = x2 @ w.t()
    y2 = torch.nn.functional.gelu(y2) if gelu else y2
    y2.backward(dy.double())
    assert x.grad.dtype == layer.weight.grad.dtype == torch.float32
    assert float((x.grad.double() - x2.grad).norm() / x2.grad.norm()) < 2e-3
    assert float((layer.weight.grad.double().view(2048, 1600) - w.grad).norm() / w.grad.norm()) < 2e-3
    if bias:
        assert layer.bias.grad.dtype == torch.float32
