"""Weight gradients over few tokens, by workgroups that take several tiles: tiles in whole and broken rounds, tokens that
end inside a stage, outputs that end inside a tile, strided operands."""

import re

import pytest
import torch

from axonn_amd import ops
from launches import launches

pytestmark = pytest.mark.gpu

SHAPES = [   # and the tile that covers the gradient in fewer of them
    (265, 8200, 2056, "256, 128"),     # the fewest tokens, a broken stage, rows and columns past the edges, 2 to 3 tiles each
    (320, 16384, 3584, "128, 256"),    # whole tiles, 7 rounds
    (448, 12288, 2048, "128, 256"),    # whole tiles, 3 whole rounds
    (447, 3336, 5128, "128, 256"),     # the last of a CU's is another tile column
    (799, 6016, 2880, "256, 128"),     # nearly the most tokens
    (300, 33000, 520, "256, 128"),     # tall
]


def tile_in_rounds(call):
    """The tile of gemm_fed_rounds_kernel if call() launches that, with 256 workgroups, and nothing else; or None."""
    found = launches(call)
    m = re.search(r"gemm_fed_rounds_kernel(?:<|ILi)(\d+)(?:, |ELi)(\d+)", found[0][0])
    assert m is None or (len(found) == 1 and found[0][1] == 256), found
    return "%s, %s" % m.groups() if m else None


@pytest.mark.parametrize("tokens, out_features, in_features, add, dtype", [
    (264, 8200, 2056, False, None), (801, 6016, 2880, False, None),          # fewer tokens, more
    (320, 8192, 2048, False, None),                                          # two rounds
    (449, 16384, 4096, False, None), (512, 8192, 3584, False, None),         # as many half rounds as large tiles take
    (440, 8288, 3736, False, None), (708, 8192, 2304, False, None), (787, 34048, 1024, False, None),   # measured slower in rounds
    (320, 16384, 3584, True, None), (320, 16384, 3584, False, torch.float32),   # bound by the output
])
def test_what_the_rule_leaves_to_others(tokens, out_features, in_features, add, dtype):
    dy = torch.zeros(tokens, out_features, device="cuda", dtype=torch.bfloat16)
    x = torch.zeros(tokens, in_features, device="cuda", dtype=torch.bfloat16)
    out = torch.zeros(out_features * in_features, device="cuda", dtype=dtype or torch.bfloat16)
    assert tile_in_rounds(lambda: ops.gemm_wgrad(dy, x, out=out, accumulate=add)) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens, out_features, in_features, tile", SHAPES)
def test_equals_the_gradient_in_pieces(tokens, out_features, in_features, tile, dtype):
    gen = torch.Generator(device="cuda").manual_seed(7)
    dy = torch.randn(tokens, out_features, generator=gen, device="cuda").to(dtype)
    x = torch.randn(tokens, in_features, generator=gen, device="cuda").to(dtype)
    assert tile_in_rounds(lambda: ops.gemm_wgrad(dy, x)) == tile
    dw = ops.gemm_wgrad(dy, x).reshape(out_features, in_features)
    # pieces of 1024 rows are less than two rounds, each with a workgroup a tile: the same sums in the same order
    piece = dy[:, :1024].contiguous()
    assert tile_in_rounds(lambda: ops.gemm_wgrad(piece, x)) is None
    for first in range(0, out_features, 1024):
        piece = ops.gemm_wgrad(dy[:, first:first + 1024].contiguous(), x).reshape(-1, in_features)
        assert torch.equal(dw[first:first + 1024], piece), first
    rows = torch.randint(0, out_features, (64,), generator=gen, device="cuda")
    exact = dy[:, rows].double().t().contiguous() @ x.double()
    # one rounding to 16 bits (2^-9 or 2^-12 of a value) and fp32 sums of `tokens` products (tokens 2^-24, normwise)
    bound = (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12) + tokens * 2.0 ** -24
    assert float((dw[rows].double() - exact).norm() / exact.norm()) <= bound


def test_leaves_what_lies_beside_the_output():
    """An output inside a larger buffer, operands whose rows are part of longer ones."""
    tokens, out_features, in_features = 300, 8200, 2056
    gen = torch.Generator(device="cuda").manual_seed(8)
    dy = torch.randn(tokens, out_features + 24, generator=gen, device="cuda").bfloat16()[:, 8:8 + out_features]
    x = torch.randn(tokens, in_features + 40, generator=gen, device="cuda").bfloat16()[:, 16:16 + in_features]
    buffer = torch.full((64 + out_features * in_features + 64,), 3.0, device="cuda", dtype=torch.bfloat16)
    out = buffer[64:64 + out_features * in_features]
    assert tile_in_rounds(lambda: ops.gemm_wgrad(dy, x, out=out)) == "256, 128"
    ops.gemm_wgrad(dy, x, out=out)
    assert torch.equal(out, ops.gemm_wgrad(dy.contiguous(), x.contiguous()).reshape(-1))
    assert bool((buffer[:64] == 3).all()) and bool((buffer[-64:] == 3).all())
