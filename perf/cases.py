"""The work that a training or inference program has this package do, as cases to time.

A case is one call pattern of such a program through the package's public entry points:

  linear     one `intra_layer.Linear`: forward, or forward and backward, alone or over several
             micro-batches whose weight gradients accumulate
  layer      the projections of one decoder layer: fused q/k/v, the attention's output and the
             patched Hugging Face gated MLP (the attention itself is not this package's)
  mlp        a whole training step of a two-layer perceptron: forward, loss, backward, optimizer
  embedding  token lookup and the table's gradient
  adam       the mixed-precision optimizer step over flat buffers

`listed()` names twelve of them, `draw()` gives others of the same ranges.  The floating-point
inputs are normal with the scales of a network in training, the token ids fall off like those of
a text (the n-th most frequent id with a share of 1 / n).
"""

import contextlib
import functools
import math
import types

import torch
import torch.nn.functional as F

from axonn_amd.inter_layer import LossScaler
from axonn_amd.intra_layer import Embedding, Linear, optimize_communication
from axonn_amd.models.transformers import modify_llama
from axonn_amd.optim import CPUAdam

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
LOSS_SCALE = 65536.0


def _linear(name, tokens, in_features, out_features, dtype="bf16", bias=True, gelu=False,
            autocast=False, train=True, micro=1):
    return {"name": name, "kind": "linear", "tokens": tokens, "in": in_features,
            "out": out_features, "dtype": dtype, "bias": bias, "gelu": gelu, "autocast": autocast,
            "train": train, "micro": micro}


def _layer(name, tokens, hidden, kv, ffn, dtype="bf16", train=True):
    return {"name": name, "kind": "layer", "tokens": tokens, "hidden": hidden, "kv": kv,
            "ffn": ffn, "dtype": dtype, "train": train}


def listed():
    return [
        # The smallest call: one layer of a small network answering a handful of requests.
        _linear("linear_8x1024", 8, 1024, 1024, train=False),
        # A small full-precision network trained step by step (the reference's own test model):
        # a dozen short launches, so latency and host work count.
        {"name": "mlp_fp32_step", "kind": "mlp", "batch": 64, "width": 1024, "hidden": 4096,
         "dtype": "fp32"},
        # Generation: 16 sequences, one token each, through a decoder layer; the weights stream by.
        _layer("layer_decode_16", 16, 4096, 2048, 14336, train=False),
        # A prompt of a length that no tile divides, through the same layer.
        _layer("layer_prefill_777", 777, 4096, 2048, 14336, train=False),
        # Training of that layer on two sequences of 2048 tokens.
        _layer("layer_train_4096", 4096, 4096, 2048, 14336),
        # One GPU's shard of a large MLP, bias and GELU fused, gradients of four micro-batches
        # accumulated in place.
        _linear("linear_gelu_shard_x4", 8192, 2560, 5120, gelu=True, micro=4),
        # A shard of a down projection on a short batch, where reading the weights is as long as
        # the arithmetic.
        _linear("linear_skinny_512", 512, 3584, 8192, bias=False),
        # Mixed precision as the reference sets it by default: fp32 parameters under fp16
        # autocast, on sequences packed to an odd number of tokens.
        _linear("linear_autocast_3001", 3001, 2560, 10240, dtype="fp16", autocast=True),
        # The head over a vocabulary of odd size.
        _linear("head_50257", 2048, 2048, 50257, bias=False),
        # A full-precision layer with real work in it.
        _linear("linear_fp32_2048", 2048, 1024, 4096, dtype="fp32", gelu=True),
        # Token lookup and its gradient over a large vocabulary.
        {"name": "embedding_128256", "kind": "embedding", "tokens": 16384, "vocab": 128256,
         "width": 2048, "dtype": "fp32"},
        # The optimizer step of a 1.3e9-parameter model in bf16 with gradient clipping.
        {"name": "adam_1p3e9", "kind": "adam", "elements": 1300000000, "tensors": 64,
         "dtype": "bf16", "clip": True},
    ]


# ------------------------------------------------------------------ draws ----
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _features(rng, lo, hi):
    """A feature count: mostly a multiple of 64, as models have them, sometimes of 8."""
    step = rng.choice((64, 64, 64, 256, 8))
    return max(step, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("forward", "train", "train", "autocast", "head", "fp32", "layer", "layer",
                       "mlp", "embedding", "adam"))
    if kind == "forward":
        c = _linear("", _log(rng, 1, 2048), _features(rng, 512, 8192), _features(rng, 512, 14336),
                    rng.choice(("bf16", "fp16")), rng.random() < 0.5, rng.random() < 0.3, train=False)
    elif kind == "train":
        c = _linear("", _log(rng, 64, 8192), _features(rng, 1024, 8192), _features(rng, 1024, 14336),
                    rng.choice(("bf16", "bf16", "fp16")), rng.random() < 0.5, rng.random() < 0.3,
                    micro=rng.choice((1, 1, 2, 4)))
    elif kind == "autocast":
        c = _linear("", _log(rng, 256, 4096), _features(rng, 1024, 5120), _features(rng, 1024, 10240),
                    rng.choice(("bf16", "fp16")), rng.random() < 0.7, autocast=True)
    elif kind == "head":
        c = _linear("", _log(rng, 256, 2048), _features(rng, 768, 2048),
                    rng.choice((rng.randrange(1000, 20000), 32000, 50257)), bias=False)
    elif kind == "fp32":
        c = _linear("", _log(rng, 16, 4096), _features(rng, 128, 2048), _features(rng, 128, 4096),
                    "fp32", rng.random() < 0.7, rng.random() < 0.5, train=rng.random() < 0.7)
    elif kind == "layer":
        hidden = 256 * rng.randrange(4, 17)
        c = _layer("", _log(rng, 1, 4096), hidden, 128 * rng.choice((2, 4, 8, 16)),
                   256 * round(hidden * rng.choice((2.6875, 3.5, 4.0)) / 256),
                   rng.choice(("bf16", "bf16", "fp16")), train=rng.random() < 0.4)
    elif kind == "mlp":
        c = {"kind": "mlp", "batch": _log(rng, 16, 2048), "width": _features(rng, 256, 2048),
             "hidden": _features(rng, 512, 4096), "dtype": rng.choice(("fp32", "bf16"))}
    elif kind == "embedding":
        c = {"kind": "embedding", "tokens": _log(rng, 16, 16384), "vocab": _log(rng, 1000, 128256),
             "width": _features(rng, 256, 2048), "dtype": rng.choice(("fp32", "bf16"))}
    else:
        c = {"kind": "adam", "elements": _log(rng, 100000, 1000000000), "tensors": _log(rng, 4, 300),
             "dtype": rng.choice(("bf16", "fp16", "fp32")), "clip": rng.random() < 0.7}
    c.pop("name", None)
    # the largest listed training cases bound what is drawn; a full-precision product takes
    # about ten times as long as a 16-bit one
    most = 2e11 if c.get("dtype") == "fp32" else 2.5e12
    while work(c)["flops"] > most:
        for size in ("tokens", "batch"):
            if size in c:
                c[size] = max(1, c[size] // 2 + c[size] % 2)
    return c


# ---------------------------------------------------------------- prepare ----
def _normal(gen, *shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _make_linear(in_features, out_features, bias, gen, dtype, **kwargs):
    layer = Linear(in_features, out_features, bias=bias,
                   init_method=lambda w: w.normal_(0.0, 0.02, generator=gen), **kwargs)
    layer = layer.to(device="cuda", dtype=dtype)
    if bias:
        with torch.no_grad():
            layer.bias.normal_(0.0, 0.02, generator=gen)
    return layer


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.no_grad():
        return {"linear": _prepare_linear, "layer": _prepare_layer, "mlp": _prepare_mlp,
                "embedding": _prepare_embedding, "adam": _prepare_adam}[case["kind"]](case, gen)


def _prepare_linear(case, gen):
    dtype = DTYPES[case["dtype"]]
    own = torch.float32 if case["autocast"] else dtype   # type of parameters and activations
    layer = _make_linear(case["in"], case["out"], case["bias"], gen, own,
                         fused_activation="gelu" if case["gelu"] else None)
    # an fp32 bias promotes the 16-bit product of an autocast region
    result = torch.float32 if case["autocast"] and case["bias"] else dtype
    std = 1e-3 * (LOSS_SCALE / 256 if dtype == torch.float16 else 1.0)
    xs, dys = [], []
    for _ in range(case["micro"]):
        x = _normal(gen, case["tokens"], case["in"], dtype=own)
        xs.append(x.requires_grad_(case["train"]))
        if case["train"]:
            dys.append(_normal(gen, case["tokens"], case["out"], std=std, dtype=result))
    return {"case": case, "layer": layer, "xs": xs, "dys": dys}


@functools.lru_cache(maxsize=None)
def _patched_mlp_class():
    modify_llama.monkey_patch_llama_with_axonn()   # once, for the life of the program
    return modify_llama.LlamaMLP


def _prepare_layer(case, gen):
    dtype, h = DTYPES[case["dtype"]], case["hidden"]
    qkv = _make_linear(h, h + case["kv"], False, gen, dtype)
    out = _make_linear(h, h, False, gen, dtype, transpose=True)
    mlp = _patched_mlp_class()(types.SimpleNamespace(
        hidden_size=h, intermediate_size=case["ffn"], hidden_act="silu", mlp_bias=False))
    mlp = mlp.to(device="cuda", dtype=dtype)
    for p in mlp.parameters():
        p.normal_(0.0, 0.02, generator=gen)
    state = {"case": case, "qkv": qkv, "out": out, "mlp": mlp}
    std = 1e-3 * (LOSS_SCALE / 256 if dtype == torch.float16 else 1.0)
    for name in ("x", "attended", "normed"):
        state[name] = _normal(gen, 1, case["tokens"], h, dtype=dtype).requires_grad_(case["train"])
    if case["train"]:
        state["dys"] = [_normal(gen, 1, case["tokens"], n, std=std, dtype=dtype)
                        for n in (h + case["kv"], h, h)]
    return state


def _prepare_mlp(case, gen):
    dtype = DTYPES[case["dtype"]]
    fc1 = _make_linear(case["width"], case["hidden"], True, gen, dtype, fused_activation="gelu")
    fc2 = _make_linear(case["hidden"], case["width"], True, gen, dtype)
    with torch.enable_grad():
        opt = CPUAdam(list(fc1.parameters()) + list(fc2.parameters()), lr=1e-3)
    return {"case": case, "fc1": fc1, "fc2": fc2, "opt": opt,
            "x": _normal(gen, case["batch"], case["width"], dtype=dtype),
            "target": _normal(gen, case["batch"], case["width"], dtype=dtype)}


def _prepare_embedding(case, gen):
    dtype = DTYPES[case["dtype"]]
    layer = Embedding(case["vocab"], case["width"],
                      init_method=lambda w: w.normal_(0.0, 0.02, generator=gen))
    layer = layer.to(device="cuda", dtype=dtype)
    u = torch.rand(1, case["tokens"], generator=gen, device="cuda", dtype=torch.float64)
    ids = (torch.exp(u * math.log(case["vocab"] + 1)) - 1).long().clamp_(0, case["vocab"] - 1)
    return {"case": case, "layer": layer, "ids": ids,
            "dy": _normal(gen, 1, case["tokens"], case["width"], std=1e-3, dtype=dtype)}


def _tensor_sizes(total, count, gen):
    """`count` odd and even sizes between a fraction and a few times their mean."""
    w = torch.rand(count, generator=gen, device="cuda", dtype=torch.float64).cpu()
    w = torch.exp(w * math.log(100.0))
    sizes = [max(1, int(v)) for v in (w / w.sum() * total).tolist()]
    sizes[-1] = max(1, sizes[-1] + total - sum(sizes))
    return sizes


def _prepare_adam(case, gen):
    dtype = DTYPES[case["dtype"]]
    sizes = _tensor_sizes(case["elements"], case["tensors"], gen)
    with torch.enable_grad():
        params = [torch.nn.Parameter(_normal(gen, n, std=0.02, dtype=dtype)) for n in sizes]
        scaler = LossScaler(loss_scale=LOSS_SCALE) if dtype != torch.float32 else None
        opt = CPUAdam(params, lr=1e-3, max_grad_norm=1.0 if case["clip"] else None,
                      loss_scaler=scaler)
    scale = LOSS_SCALE if dtype != torch.float32 else 1.0
    # fp16: gradients small enough that the sum of a whole tensor stays in range (the overflow
    # test is on that sum)
    opt.model_grads_fp16.normal_(0.0, (1e-6 if dtype == torch.float16 else 1e-3) * scale, generator=gen)
    return {"case": case, "opt": opt, "params": params}


# -------------------------------------------------------------------- run ----
def run(state):
    return {"linear": _run_linear, "layer": _run_layer, "mlp": _run_mlp,
            "embedding": _run_embedding, "adam": _run_adam}[state["case"]["kind"]](state)


def _run_linear(state):
    case, layer = state["case"], state["layer"]
    context = contextlib.nullcontext()
    if case["autocast"]:
        context = torch.autocast("cuda", dtype=DTYPES[case["dtype"]])
    if not case["train"]:
        with torch.no_grad(), context:
            return layer(state["xs"][0])
    layer.zero_grad(set_to_none=True)
    outputs, gradients = [], []
    accumulating = (optimize_communication(overlap_reduce_scatter=True) if case["micro"] > 1
                    else contextlib.nullcontext())
    with accumulating:
        for x, dy in zip(state["xs"], state["dys"]):
            x.grad = None
            with context:
                y = layer(x)
            y.backward(dy)
            outputs.append(y.detach())
            gradients.append(x.grad)
    return outputs, gradients, [p.grad for p in layer.parameters()]


def _run_layer(state):
    train, mlp = state["case"]["train"], state["mlp"]
    if not train:
        with torch.no_grad():
            return (state["qkv"](state["x"]), state["out"](state["attended"]),
                    mlp(state["normed"]))
    inputs = [state[name] for name in ("x", "attended", "normed")]
    for x in inputs:
        x.grad = None
    for module in (state["qkv"], state["out"], mlp):
        module.zero_grad(set_to_none=True)
    outputs = (state["qkv"](state["x"]), state["out"](state["attended"]),
               mlp(state["normed"]))
    torch.autograd.backward(outputs, state["dys"])
    weights = [p for module in (state["qkv"], state["out"], mlp) for p in module.parameters()]
    return [y.detach() for y in outputs], [x.grad for x in inputs], [p.grad for p in weights]


def _run_mlp(state):
    opt = state["opt"]
    opt.zero_grad()
    y = state["fc2"](state["fc1"](state["x"]))
    loss = F.mse_loss(y, state["target"])
    loss.backward()
    opt.step()
    return y.detach(), loss.detach(), opt.model_grads_fp16, opt.model_params_fp32, opt.exp_avg, opt.exp_avg_sq


def _run_embedding(state):
    layer = state["layer"]
    layer.zero_grad(set_to_none=True)
    rows = layer(state["ids"])
    rows.backward(state["dy"])
    return rows.detach(), layer.weight.grad


def _run_adam(state):
    opt = state["opt"]
    opt.step()
    return opt.model_params_fp32, opt.exp_avg, opt.exp_avg_sq, opt.model_params_fp16


# ------------------------------------------------------------ work, limits ---
def _product(tokens, n_in, n_out, train):
    """(elements moved, FLOPs) of one projection: X, W and Y; backward dY, W, X, dX and dW."""
    elements = tokens * n_in + n_in * n_out + tokens * n_out
    return (3 * elements if train else elements), (6 if train else 2) * tokens * n_in * n_out


def work(case):
    kind = case["kind"]
    size = 4 if case["dtype"] == "fp32" else 2
    if kind == "linear":
        elements, flops = _product(case["tokens"], case["in"], case["out"], case["train"])
        nbytes = elements * size
        if case["autocast"]:   # parameters, input and their gradients are fp32
            nbytes += 2 * (2 * case["tokens"] * case["in"] + 2 * case["in"] * case["out"])
        return {"bytes": case["micro"] * nbytes, "flops": case["micro"] * flops}
    if kind == "layer":
        h, t, train = case["hidden"], case["tokens"], case["train"]
        parts = [_product(t, a, b, train) for a, b in
                 ((h, h + case["kv"]), (h, h), (h, case["ffn"]), (h, case["ffn"]), (case["ffn"], h))]
        return {"bytes": size * sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if kind == "mlp":
        b, w, h = case["batch"], case["width"], case["hidden"]
        # the input takes no gradient; the update moves 28 bytes an element
        elements = 3 * _product(b, w, h, False)[0] + 3 * _product(b, h, w, False)[0] - b * w
        return {"bytes": elements * size + 28 * 2 * w * h, "flops": 10 * b * w * h}
    if kind == "embedding":
        t, v, w = case["tokens"], case["vocab"], case["width"]
        return {"bytes": size * (3 * t * w + v * w) + 16 * t, "flops": t * w}
    # gradient, parameter and two moments read; parameter, moments and a 16-bit copy written;
    # the norm or the overflow test has to read every gradient before the first update
    scanned = case["clip"] or case["dtype"] == "fp16"
    per = (size if scanned else 0) + size + 24 + (2 if size == 2 else 0)
    return {"bytes": per * case["elements"], "flops": 12 * case["elements"]}


def tolerance(case):
    """About four times (bf16 products: two and a half times) the largest relative difference
    seen between this path, the same computed in 64 bits, and the same in torch's own kernels at
    the same precision: 4.1e-3, 5.2e-4 and 1.3e-6 for products of bf16, fp16 and fp32; 6.1e-3
    (bf16) and 1.5e-6 (fp32) for the training step, whose second moment squares a gradient;
    1.5e-3 and 2.1e-7 for the table's gradient; 3.4e-7 for optimizer state and 2.3e-6 for the
    16-bit copy, where a weight on a rounding boundary may go either way."""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "mlp":
        return {"rel": {"bf16": 2.4e-2, "fp32": 6e-6}[dtype]}
    if kind == "embedding":
        return {"rel": {"bf16": 6e-3, "fp32": 1e-6}[dtype]}
    if kind == "adam":
        return {"rel": 1.5e-6 if dtype == "fp32" else 1e-5}
    return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 5e-6}[dtype]}
