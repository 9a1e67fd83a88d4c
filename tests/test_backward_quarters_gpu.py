"""Both gradients in one launch whose last tiles are four workgroups each: of dX, of dW, fresh and added to."""

import pytest
import torch

from axonn_amd import _native as nv
from launches import launches
from test_gemm_edge_gpu import canvas, check, numbers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,quartered", [(1536, 2816, 4096, 16), (2816, 1536, 4096, 16), (4096, 2560, 2560, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("out,beta", [(None, 0), (None, 1), (torch.float32, 0), (torch.float32, 1)])
def test_the_last_tiles_of_a_joint_backward(M, N, K, quartered, dtype, out, beta):
    out = out or dtype
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    dY, W, X = (numbers(r, c, dtype, gen, 16) for r, c in ((M, N), (N, K), (M, K)))
    (fx, dx), (fw, dw) = canvas(M, K, dtype), canvas(N, K, out)
    dw.fill_(3.0)
    call = lambda: nv.call(   # noqa: E731
        "axn_gemm_bwd", nv.ptr(dY), nv.ptr(W), nv.ptr(X), nv.ptr(dx), nv.ptr(dw), nv.dtype_code(dtype), M, N, K,
        dY.stride(0), W.stride(0), X.stride(0), dx.stride(0), dw.stride(0), beta, nv.dtype_code(out), nv.current_stream())
    tiles = (M // 256 + N // 256) * (K // 256)
    (name, workgroups), = launches(call)
    assert "gemm_backward_kernel" in name and workgroups == tiles + 3 * quartered, (name, workgroups)
    dw.fill_(3.0)
    call()
    check(fx, dx, dY.double() @ W.double())
    check(fw, dw, dY.double().t() @ X.double() + 3.0 * beta)
