"""Products of operands whose rows lie 2^22 elements and more apart: views such as the last token of
every sequence, and rows that long themselves.  Whole numbers, so results are exact; NaN around
the views."""

import pytest
import torch

from axonn_amd import _native as nv

pytestmark = pytest.mark.gpu


def far(rows, cols, ld, dtype, gen):
    full = torch.full(((rows - 1) * ld + cols + 8,), float("nan"), dtype=dtype, device="cuda")
    view = full.as_strided((rows, cols), (ld, 1))
    view.copy_(torch.randint(-2, 3, (rows, cols), generator=gen, device="cuda"))
    return view


@pytest.mark.parametrize("ld", [(1 << 22), (1 << 23) - 8, 1 << 23, (1 << 24) + 8])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (33, 40, 72), (70, 24, 200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_the_library_takes_any_row_stride(M, N, K, ld, dtype):
    gen = torch.Generator(device="cuda").manual_seed(M + ld % 1000)
    X, W, dY = (far(r, c, ld, dtype, gen) for r, c in ((M, K), (N, K), (M, N)))
    b = torch.randint(-3, 4, (N,), generator=gen, device="cuda").float()
    code, stream, sfx = nv.dtype_code(dtype), nv.current_stream(), "" if dtype == torch.bfloat16 else "_f16"
    y = torch.full((M + 1, N), 7.0, dtype=dtype, device="cuda")
    nv.call("axn_gemm_fwd" + sfx, nv.ptr(X), nv.ptr(W), nv.ptr(b), nv.ptr(y), None, M, N, K, ld, ld, N, nv.EPI_BIAS,
            stream)
    assert torch.equal(y[:M].double(), (X.double() @ W.double().t() + b).to(dtype).double())
    assert (y[M] == 7).all()
    dx = torch.full((M + 1, K), 7.0, dtype=dtype, device="cuda")
    nv.call("axn_gemm_dgrad" + sfx, nv.ptr(dY), nv.ptr(W), nv.ptr(dx), M, N, K, ld, ld, K, stream)
    assert torch.equal(dx[:M].double(), (dY.double() @ W.double()).to(dtype).double())
    assert (dx[M] == 7).all()
    dw = torch.full((N + 1, K), 3.0, device="cuda")
    nv.call("axn_gemm_wgrad" + sfx, nv.ptr(dY), nv.ptr(X), nv.ptr(dw), M, N, K, ld, ld, K, 1, nv.F32, stream)
    assert torch.equal(dw[:N].double(), dY.double().t() @ X.double() + 3)
    assert (dw[N] == 3).all()


@pytest.mark.parametrize("batch,length,K", [(8, 4096, 4096), (40, 2048, 4096), (70, 1024, 8192)])
def test_last_token_of_every_sequence(batch, length, K):
    from axonn_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(batch)
    X = far(batch, K, length * K, torch.bfloat16, gen)
    W = torch.randint(-2, 3, (264, K), generator=gen, device="cuda").bfloat16()
    dY = torch.randint(-2, 3, (batch, 264), generator=gen, device="cuda").bfloat16()
    assert torch.equal(ops.gemm_fwd(X, W)[0].double(), (X.double() @ W.double().t()).bfloat16().double())
    dx, dw = ops.gemm_bwd(dY, W, X)
    assert torch.equal(dx.double(), (dY.double() @ W.double()).bfloat16().double())
    assert torch.equal(dw.double(), (dY.double().t() @ X.double()).bfloat16().double())
