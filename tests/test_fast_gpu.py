"""The native host side of the usual Linear calls (csrc/fast.cpp) against the general one: the same kernels with the same
arguments, so the same bits; and the calls that it has to leave to the general way."""

import ctypes

import pytest
import torch

from axonn_amd import _native as nv
from axonn_amd import ops
from axonn_amd.intra_layer import Linear, optimize_communication

pytestmark = pytest.mark.gpu
nv.load()
FAST = nv.fast


def _both(monkeypatch, run):
    """run() with the native side and without, and how often the native side answered."""
    answers = []

    class Counted:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(FAST, name)(*args)
                answers.append((name, out is not None))
                return out
            return call

    monkeypatch.setattr(nv, "fast", Counted())
    got = run()
    monkeypatch.setattr(nv, "fast", None)
    want = run()
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
            assert a.requires_grad == b.requires_grad and torch.equal(a, b)
    return answers


def test_it_is_built():
    assert FAST is not None and FAST.ABI_VERSION == nv.ABI_VERSION


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("bias", [None, "own", "fp32"])
@pytest.mark.parametrize("act", [None, "gelu"])
@pytest.mark.parametrize("shape,features", [((1, 8), 8), ((8, 1024), 1024), ((3, 5, 264), 520), ((777, 64), 24), ((256,), 40),
                                            ((7, 72), 13), ((64, 4096), 64)])
def test_layer_calls_are_the_same(dtype, bias, act, shape, features, monkeypatch):
    torch.manual_seed(1)
    layer = Linear(shape[-1], features, bias=bias is not None, fused_activation=act).cuda().to(dtype)
    if bias is not None:
        layer.bias.data = torch.randn(features, device="cuda").to(torch.float32 if bias == "fp32" else dtype)
    x = torch.randn(shape, device="cuda").to(dtype)

    def infer():
        with torch.no_grad():
            return [layer(x)]

    answers = _both(monkeypatch, infer)
    assert answers.count(("linear", True)) == (bias is not None or act is not None)

    def train(out=None):
        layer.weight.grad = out
        if layer.bias is not None:
            layer.bias.grad = None
        leaf = x.clone().requires_grad_(True)
        y = layer(leaf)
        y.backward(torch.cos(torch.arange(y.numel(), device="cuda").view(y.shape)).to(y.dtype))
        return [y.detach(), leaf.grad, layer.weight.grad, None if layer.bias is None else layer.bias.grad]

    answers = _both(monkeypatch, train)
    assert ("gemm_fwd", True) in answers
    assert (("backward", True) in answers) == (features % 8 == 0)

    def accumulate():
        with optimize_communication(overlap_reduce_scatter=True):
            return train(torch.ones(layer.weight.numel(), device="cuda", dtype=dtype))

    answers = _both(monkeypatch, accumulate)
    assert len(shape) == 1 or (("backward", True) in answers) == (features % 8 == 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_autocast_is_the_same(dtype, act, monkeypatch):
    torch.manual_seed(2)
    layer = Linear(512, 256, fused_activation=act).cuda()
    x = torch.randn(300, 512, device="cuda")

    def run():
        layer.weight.grad = layer.bias.grad = None
        leaf = x.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype):
            y = layer(leaf)
            with torch.no_grad():
                y2 = layer(x)
        y.backward(torch.cos(y.detach()))
        return [y.detach(), y2, leaf.grad, layer.weight.grad, layer.bias.grad]

    answers = _both(monkeypatch, run)
    assert ("linear", True) not in answers and ("backward", True) in answers


@pytest.mark.parametrize("needs", [(True, False, False), (False, True, False), (False, False, True), (True, False, True),
                                   (False, True, True)])
def test_parts_of_the_backward(needs, monkeypatch):
    torch.manual_seed(3)
    layer = Linear(256, 384, fused_activation="gelu").cuda().bfloat16()
    x = torch.randn(96, 256, device="cuda").bfloat16()

    def run():
        layer.weight.grad = layer.bias.grad = None
        leaf = x.clone().requires_grad_(needs[0])
        layer.weight.requires_grad_(needs[1])
        layer.bias.requires_grad_(needs[2])
        layer(leaf).sum().backward()   # (an expanded gradient)
        y = layer(leaf)
        y.backward(torch.ones_like(y))
        return [leaf.grad, layer.weight.grad, layer.bias.grad]

    assert ("backward", True) in _both(monkeypatch, run)


def _watched():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    return {"functions": Functions, "dispatch": Dispatch}


class _Sub(torch.Tensor):
    pass


def test_what_is_left_to_the_general_way():
    lin = FAST.linear
    x = torch.randn(16, 64, device="cuda").bfloat16()
    w, b = torch.randn(48 * 64, device="cuda").bfloat16(), torch.randn(48, device="cuda").bfloat16()
    assert lin(x, w, b, 48, 64, False) is None                      # gradients are recorded
    with torch.no_grad():
        assert lin(x, w, b, 48, 64, False) is not None
        wide = torch.randn(16, 72, device="cuda").bfloat16()
        odd = torch.randn(16 * 64 + 1, device="cuda").bfloat16()[1:].view(16, 64)
        for args in [(x.cpu(), w, b), (x, w.cpu(), b), (x, w, b.cpu()), (x.half(), w, b), (x, w.half(), b), (x, w, b.half()),
                     (wide[:, :64], w, b), (odd, w, b), (x[:0], w, b), (x, w[:-64], b), (x, w, b[:-8]), (x, w, b.repeat(2)[::2]),
                     (x.t(), w, b), (x.as_subclass(_Sub), w, b), (x, w.as_subclass(_Sub), b), (x.double(), w.double(), b),
                     (x.to_sparse(), w, b), (x[0, 0], w, b)]:
            assert lin(*args, 48, 64, False) is None
        assert lin(x, w, b, 64, 48, False) is None and lin(x, w, b, 0, 64, False) is None
        for mode in _watched().values():
            with mode():
                assert lin(x, w, b, 48, 64, False) is None
        with torch.autocast("cuda", torch.bfloat16):
            assert lin(x, w, b, 48, 64, False) is None
        with torch.autograd.forward_ad.dual_level():
            assert lin(torch.autograd.forward_ad.make_dual(x, x), w, b, 48, 64, False) is None
        seen = []
        torch.vmap(lambda t: (seen.append(lin(t, w, b, 48, 64, False)), t)[1])(x.view(2, 8, 64))
        assert seen == [None]
    seen = []
    torch.func.grad(lambda t: (seen.append(FAST.gemm_fwd(t, w.view(48, 64), None, False, False, False)), t.float().sum())[1])(x)
    assert seen == [None]
    with torch.inference_mode():
        assert lin(x, w, b, 48, 64, False).is_inference()
    for args in [(), (x,), (x, w, b), (1, 2, 3, 4, 5, 6), (None,) * 6]:
        assert lin(*args) is None and FAST.gemm_fwd(*args) is None and FAST.backward(*args) is None
    assert FAST.backward(*(None,) * 11) is None
    back = lambda dy, z, out, dw: FAST.backward(dy, z, w.view(48, 64), x, out, True, True, True, nv.BF16, dw, False)
    dy = torch.randn(16, 48, device="cuda").bfloat16()
    assert back(dy, None, None, nv.BF16) is not None
    flat = torch.zeros(48 * 64 + 8, device="cuda")
    for args in [(dy[:8], None, None, 0), (dy.half(), None, None, 0), (dy, dy[:8], None, 0), (dy, dy.half(), None, 0),
                 (dy, None, flat[8:], 0), (dy, None, flat, 2), (dy, None, flat[1:-7], 2), (dy, None, None, 1),
                 (dy, None, None, -1), (dy.cpu(), None, None, 0), (dy[:, :1].expand(16, 48), None, None, 0)]:
        assert back(*args) is None


@pytest.mark.parametrize("dual", ["x", "weight", "bias"])
def test_a_tangent_is_refused_as_the_general_way_refuses_it(dual):
    """Of any operand, also where no gradients are recorded (forward mode goes on there): it is not dropped."""
    layer = Linear(64, 48).cuda().bfloat16()
    x = torch.randn(16, 64, device="cuda").bfloat16()
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        at = {"x": x, "weight": layer.weight, "bias": layer.bias}
        made = torch.autograd.forward_ad.make_dual(at[dual].detach(), torch.ones_like(at[dual]))
        if dual == "x":
            x = made
        with pytest.raises(NotImplementedError, match="jvp"):
            torch.func.functional_call(layer, {} if dual == "x" else {dual: made}, (x,))


def test_arguments_are_asked_with_the_interpreters_lock():
    x, w, b = (torch.randn(s, device="cuda").bfloat16() for s in ((16, 64), (48 * 64,), (48,)))

    class Asked:
        def __init__(self, answer):
            self.answer = answer

        def __bool__(self):
            return {"yes": True, "no": False}[self.answer]

    with torch.no_grad():
        for answer, plain in (("yes", True), ("no", False)):
            assert torch.equal(FAST.linear(x, w, b, 48, 64, Asked(answer)), FAST.linear(x, w, b, 48, 64, plain))
        with pytest.raises(KeyError):
            FAST.linear(x, w, b, 48, 64, Asked("neither"))
        with pytest.raises(TypeError):
            FAST.linear(x, w, b, "48", 64, False)


def test_errors_are_those_of_the_general_way():
    layer = Linear(64, 48).cuda().bfloat16()
    with torch.no_grad():
        with pytest.raises(TypeError, match="operand dtypes differ"):
            layer(torch.zeros(4, 64, device="cuda"))
        with pytest.raises(RuntimeError, match="GPU only"):
            layer(torch.zeros(4, 64).bfloat16())
        with pytest.raises(ValueError):
            layer(torch.zeros(4, 56, device="cuda").bfloat16())
        a = torch.zeros(8, 64, device="cuda").bfloat16()
        with pytest.raises(ValueError, match="needs `out`"):
            ops.gemm_bwd(a, a.new_zeros(64, 64), a, accumulate=True)
        stale = torch.ones(64, 64, device="cuda")
        assert not ops.gemm_bwd(a, a.new_zeros(64, 64), a, out=stale)[1].any()   # written, not added to
        assert ops.gemm_fwd(a, a.new_zeros(64, 64), None, "gelu", save_z=1)[1] is not None
        assert layer(torch.zeros(0, 64, device="cuda").bfloat16()).shape == (0, 48)
        assert ops.gemm_fwd(torch.zeros(4, 64, device="cuda"), torch.zeros(48, 64, device="cuda"))[0].shape == (4, 48)


# (each a different entry point: one launch, one in parts, two launches, full precision)
@pytest.mark.parametrize("dtype,M,N,K", [(torch.bfloat16, 64, 128, 64), (torch.bfloat16, 777, 6144, 4096),
                                         (torch.float16, 512, 8192, 3584), (torch.float32, 64, 128, 256)])
def test_an_error_behind_a_launch_is_raised_and_adds_once(dtype, M, N, K):
    """A launch that has been made and then reports an error (HIP reports one that an earlier call left behind): the
    weight gradient has been added, and is not added again by another way."""
    lib, calls = nv.load(), []

    def reports_an_error(name):
        def entry(*args):
            assert getattr(lib, name)(*args) == nv.AXN_OK
            calls.append(name)
            return nv.AXN_EHIP
        return ctypes.CFUNCTYPE(*[nv.SYMBOLS[name][0], *nv.SYMBOLS[name][1]])(entry)

    table = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in FAST.entry_points()}
    table["check"] = nv.check
    adding = [name for name in table if name.startswith(("axn_gemm_bwd", "axn_gemm_wgrad")) and not name.endswith("_bytes")]
    entries = {name: reports_an_error(name) for name in adding}
    dy, w, x = (torch.randint(-2, 3, s, device="cuda").to(dtype) for s in ((M, N), (N, K), (M, K)))
    grad = torch.full((N, K), 3.0, device="cuda")
    once = ops.gemm_wgrad(dy, x, out=grad.clone(), accumulate=True)
    FAST.bind(dict(table, **{name: ctypes.cast(e, ctypes.c_void_p).value for name, e in entries.items()}))
    try:
        with pytest.raises(nv.AxnError) as raised:
            ops.gemm_bwd(dy, w, x, out=grad, accumulate=True)
    finally:
        FAST.bind(table)
    assert raised.value.code == nv.AXN_EHIP and len(calls) == 1
    assert torch.equal(grad, once)


def test_streams_and_graphs():
    """On the current stream, and in a captured graph, replayed with other work between."""
    torch.manual_seed(4)
    layer = Linear(512, 512).cuda().bfloat16()
    x = torch.randn(32, 512, device="cuda").bfloat16()
    stream = torch.cuda.Stream()
    with torch.no_grad():
        want = layer(x).clone()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            busy = torch.randn(4096, 4096, device="cuda")
            for _ in range(4):
                busy = busy @ busy * 1e-2
            late = x + 0 * busy[:32, :512].nan_to_num(0, 0, 0).bfloat16()   # ready when the stream's work is done
            got = layer(late)
        stream.synchronize()
        assert torch.equal(got, want)
        graph, held = torch.cuda.CUDAGraph(), x.clone()
        with torch.cuda.graph(graph):
            y = layer(held)
        for seed in range(3):
            torch.manual_seed(seed)
            held.copy_(torch.randn(32, 512, device="cuda"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, layer(held))


def test_the_entry_points_it_binds_are_the_librarys():
    lib = nv.load()
    for name in FAST.entry_points():
        assert name in nv.SYMBOLS and ctypes.cast(getattr(lib, name), ctypes.c_void_p).value
