"""The gate/up forward in one launch at sizes that are not made of whole tiles: every tile at its edges, whole-number
operands in buffers of NaN, outputs in canvases; and the patched MLP that takes it, against its separate calls."""

import re

import pytest
import torch

from axonn_amd import _native as nv
from axonn_amd import ops
from launches import launches
from test_gemm_edge_gpu import CANARY, canvas, check, numbers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,tile", [
    (65, 8, 8, "128, 128"), (70, 136, 72, "64, 128"), (129, 1000, 136, "64, 128"),   # one to three stages
    (89, 10568, 328, "96, 128"), (150, 8184, 328, "96, 128"), (250, 8184, 328, "128, 128"),
    (573, 11000, 200, "128, 256"), (1001, 4088, 200, "192, 256"), (430, 5024, 136, "128, 256"),
    (397, 12360, 136, "224, 256"), (777, 14328, 136, "224, 256"), (689, 8288, 136, "256, 256"), (2047, 8184, 200, "256, 256"),
    (256, 2048, 512, "64, 128"), (256, 8192, 512, "128, 128"), (512, 8192, 512, "128, 256"), (768, 8192, 512, "192, 256"),   # whole tiles, too few large ones
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("save", [True, False])
def test_gate_up_of_any_size(M, N, K, tile, dtype, save):
    gen = torch.Generator(device="cuda").manual_seed(M + 3 * N + 7 * K)
    X, G, U = (numbers(r, K, dtype, gen, 16) for r in (M, N, N))
    (fh, h), (fg, gate), (fu, up) = (canvas(M, N, dtype) for _ in range(3))
    whole = ops.gemm_swiglu_supported(M, N, K, dtype)
    call = lambda: nv.call(   # noqa: E731
        "axn_gemm_swiglu_fwd", nv.ptr(X), nv.ptr(G), nv.ptr(U), nv.ptr(h), nv.ptr(gate) if save else None,
        nv.ptr(up) if save else None, nv.dtype_code(dtype) | (0 if whole else nv.ANY_SIZES), M, N, K, X.stride(0),
        G.stride(0), h.stride(0), nv.current_stream())
    (name, _), = launches(call)
    m = re.search(r"gemm_gate_up_edge_kernel(?:<|ILi)(\d+)(?:, |ELi)(\d+)", name)
    assert m and "%s, %s" % m.groups() == tile, name
    want_g, want_u = (X.double() @ W.double().t() for W in (G, U))
    assert torch.equal(h, ops.swiglu_fwd(want_g.to(dtype), want_u.to(dtype)))
    h.fill_(CANARY)
    assert torch.equal(fh, torch.full_like(fh, CANARY)), "written outside the output"
    if save:
        check(fg, gate, want_g)
        check(fu, up, want_u)


def test_sizes_that_stay_refused_without_the_flag():
    x, w = torch.zeros(300, 64, device="cuda").bfloat16(), torch.zeros(128, 64, device="cuda").bfloat16()
    with pytest.raises(nv.AxnError, match="M % 256 == 0"):
        ops.gemm_swiglu_fwd(x, w, w)
    h, _, _ = ops.gemm_swiglu_fwd(x, w, w, any_sizes=True)
    assert h.shape == (300, 128) and not h.any()


@pytest.mark.parametrize("tokens,hidden,ffn,grad", [(777, 512, 1408, False), (301, 1024, 2752, True)])
def test_the_patched_mlp_of_any_number_of_tokens(tokens, hidden, ffn, grad, monkeypatch):
    """Bars: both paths round the pre-activations, the activation and each product to bfloat16 (2^-9 each)."""
    from transformers import LlamaConfig
    from transformers.models.llama.modeling_llama import LlamaMLP

    import axonn_amd.axonn as ax
    from axonn_amd.models.transformers import modify_llama, parallelize

    ax.init(1, 1, 1, 1)
    cfg = LlamaConfig(hidden_size=hidden, intermediate_size=ffn, num_attention_heads=4, num_key_value_heads=2,
                      num_hidden_layers=1, vocab_size=32)
    with parallelize(cfg):
        mlp = LlamaMLP(cfg)
    mlp.forward = modify_llama.modified_mlp_forward.__get__(mlp)
    mlp = mlp.cuda().bfloat16()
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn(1, tokens, hidden, generator=gen, device="cuda").bfloat16().requires_grad_(grad)
    dy = torch.randn(1, tokens, hidden, generator=gen, device="cuda").bfloat16()

    def step():
        mlp.zero_grad(set_to_none=True)
        x.grad = None
        with torch.set_grad_enabled(grad):
            y = mlp(x)
        if not grad:
            return [y]
        y.backward(dy)
        return [y.detach(), x.grad] + [p.grad for p in mlp.parameters()]

    assert modify_llama._one_launch_gate_up(mlp, x)
    fused = step()
    monkeypatch.setattr(modify_llama, "_one_launch_gate_up", lambda mlp, x: False)
    for a, b in zip(fused, step()):
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 1e-2


@pytest.mark.parametrize("tokens,hidden,ffn", [(301, 1024, 2752), (777, 512, 1408)])
@pytest.mark.parametrize("x_dtype,dtype", [(torch.float32, torch.bfloat16), (torch.float32, torch.float16),
                                           (torch.bfloat16, torch.float16), (torch.bfloat16, torch.bfloat16)])
def test_input_gradients_are_added_in_the_inputs_type(tokens, hidden, ffn, x_dtype, dtype):
    """Each rounded to the products' type, converted to the input's and then added, as autograd adds those of two
    projections: an fp32 input under autocast has the fp32 sum of the two."""
    from axonn_amd.models.transformers.modify_llama import GateUpSwiGLU

    gen = torch.Generator(device="cuda").manual_seed(tokens)
    x = torch.randn(1, tokens, hidden, generator=gen, device="cuda").to(x_dtype).requires_grad_(True)
    wg, wu = (torch.randn(ffn, hidden, generator=gen, device="cuda").mul_(0.02).to(dtype).requires_grad_(True) for _ in range(2))
    dh = torch.randn(1, tokens, ffn, generator=gen, device="cuda").mul_(0.1).to(dtype)
    with torch.autocast("cuda", dtype):
        h = GateUpSwiGLU.apply(x, wg.view(-1), wu.view(-1), (ffn, hidden), True)
    h.backward(dh)
    x2 = x.detach()[0].to(dtype)
    _, gate, up = ops.gemm_swiglu_fwd(x2, wg.detach(), wu.detach(), any_sizes=True)
    (a, dwg), (b, dwu) = (ops.gemm_bwd(d, w.detach(), x2) for d, w in zip(ops.swiglu_bwd(dh[0], gate, up), (wg, wu)))
    assert a.dtype == b.dtype == dtype and x.grad.dtype == x_dtype
    assert torch.equal(x.grad[0], a.to(x_dtype) + b.to(x_dtype))
    assert torch.equal(wg.grad, dwg) and torch.equal(wu.grad, dwu)
