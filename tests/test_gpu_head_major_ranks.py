"""Head-major dy at the kernel ranks whose backward runs as passes of ranks: every gradient is bitwise
that of the [B, T, D] layout, also where dx comes from launches of its own (one head to a 128-channel
chunk, two, and heads across chunks; rows that end inside a tile, several runs)."""

import math

import pytest
import torch

from helpers import gen, randn
from dynconv import lowrank as lr_mod

pytestmark = pytest.mark.gpu
bf16, fp16 = torch.bfloat16, torch.float16

SHAPES = [(35, True, 3, bf16), (63, True, 4, bf16), (64, False, 5, fp16), (40, False, 8, bf16), (63, True, 7, bf16),
          (95, True, 5, bf16), (127, True, 2, fp16), (100, False, 4, bf16), (50, True, 12, bf16), (130, False, 2, bf16)]
CASES = [(2, T, D, hd, *s) for s in SHAPES for T, D, hd in ((45, 384, 192), (70, 384, 64), (33, 512, 128), (7, 320, 64))]
CASES += [(1, 35000, 128, 64, *s) for s in SHAPES[1:4]]


@pytest.mark.parametrize("case", CASES, ids=[f"T{c[1]}D{c[2]}h{c[3]}R{c[4]}W{c[6]}" for c in CASES])
def test_head_major_is_bitwise(case):
    B, T, D, hd, R, static, W, dtype = case
    g = gen(T + D + hd + R + W)
    x, z = randn(g, B, T, D).to(dtype).cuda(), randn(g, B, T, R).to(dtype).cuda()
    U = randn(g, R, W * D, scale=1 / math.sqrt((R + 1) * W)).to(dtype).cuda()
    sw = randn(g, W, D, scale=1 / math.sqrt(W)).to(dtype).cuda() if static else None
    dy = randn(g, B, T, D).to(dtype).cuda()

    def grads(h, dyl):  # any rank (the public function asserts a power of two)
        ps = [t.detach().requires_grad_() for t in (x, z, U, *([sw] if static else []))]
        ys = lr_mod._GroupedLowrankDynamicConvolutionFn.apply(ps[0], True, 1, static, h, *ps[1:])
        return torch.autograd.grad(ys, ps, [dyl])

    ref = grads(0, dy)
    got = grads(hd, dy.view(B, T, D // hd, hd).transpose(1, 2).contiguous())
    for a, b, n in zip(got, ref, ("dx", "dz", "dU", "dstatic_w")):
        assert torch.equal(a, b), n
