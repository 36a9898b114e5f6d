"""The lowrank backward's later passes (taps, or ranks over the fp32 accumulator), which add to the dx rows
of the earlier ones: rows taken with the tile, at its start and before its last tap, the open rows
of the tile before among them, at the edges of tiles and of runs, against the CPU oracle."""

import math

import pytest
import torch

from helpers import assert_ns, check_reductions, gen, randn, run_fwd_bwd, uniform
from dynconv import lowrank as lr_mod
from oracle.reference_cpu import lowrank_dynamic_convolution_ref as lr_ref

pytestmark = pytest.mark.gpu
bf16, fp16 = torch.bfloat16, torch.float16

# kernel rank, W: two rank chunks in passes of 3 + 2, 4 + 4, 4 + 3 + 3 taps and five of 4; one chunk in 6 + 6;
# more than two passes of ranks at W 1-4, and of ranks x taps
SHAPES = [(31, True, 5, bf16), (32, False, 8, bf16), (24, False, 10, fp16), (31, True, 20, bf16), (16, False, 12, bf16),
          (160, False, 1, bf16), (130, True, 2, fp16), (160, False, 3, bf16), (140, False, 4, bf16), (95, True, 6, bf16),
          (127, True, 8, fp16), (50, False, 18, bf16)]
# one row, a tile and one row, rows up to a tile's open ones, several runs of one and of two tiles
CASES = [(B, T, D, *s) for s in SHAPES for B, T, D in ((1, 1, 8), (1, 33, 40), (2, 61, 264))]
CASES += [(1, 16500, 64, *s) for s in SHAPES[::2]] + [(3, 5000, 72, *s) for s in SHAPES[1::2]]


@pytest.mark.parametrize("case", CASES, ids=[f"B{c[0]}T{c[1]}D{c[2]}R{c[3]}W{c[5]}{'s' if c[4] else ''}" for c in CASES])
def test_backward_passes(case):
    B, T, D, R, static, W, dtype = case
    g = gen(T * 1009 + D * 7 + R + W)
    x, dy, z = randn(g, B, T, D), randn(g, B, T, D), randn(g, B, T, R)
    U = randn(g, R, W * D, scale=1 / math.sqrt((R + 1) * W))
    sw = uniform(g, W, D, lo=-1 / math.sqrt(W), hi=1 / math.sqrt(W)) if static else None

    def kernel(a, b, c, d, residual):  # any rank (the public function asserts a power of two)
        return lr_mod._LowrankDynamicConvolutionFn.apply(a, b, c, d, residual)

    q = [None if t is None else t.to(dtype).float() for t in (x, z, U, sw)]
    _, g_q = run_fwd_bwd(lr_ref, q, dy.to(dtype).float(), True)
    dev = [None if t is None else t.to(dtype).cuda() for t in q]
    _, g_k = run_fwd_bwd(kernel, dev, dy.to(dtype).cuda(), True)
    for a, b, n in zip(g_k, g_q, ["dx", "dz", "dU", "dstatic_w"]):
        if b is not None:
            assert_ns(a, b, dtype, n, elementwise=n == "dx")
    check_reductions("lr", q, dy.to(dtype).float(), g_k, dtype)
