"""The lowrank backward's 32-row x 32-channel tiles (lr_bwd_t32) where they can go wrong: sequence
lengths around a tile and a run of tiles, channels that end inside a 32-channel wavefront and a
256-channel workgroup, every width of one pass (the look-ahead sums reach W - 1 <= 7 rows into the
group above), ranks around a rank chunk, passes of taps and of ranks, against the CPU oracle."""

import math

import pytest
import torch

from helpers import assert_ns, check_reductions, gen, randn, run_fwd_bwd, uniform
from dynconv import lowrank as lr_mod
from oracle.reference_cpu import lowrank_dynamic_convolution_ref as lr_ref

pytestmark = pytest.mark.gpu
bf16, fp16 = torch.bfloat16, torch.float16

CASES = (
    # tile edges at one and two rank chunks: one row, a tile less one, one, one more, two tiles and one row
    [(1, T, 40, R, 4, st, bf16) for T in (1, 31, 32, 33, 65) for R, st in ((16, False), (31, True))]
    # every width of one pass at a short second tile (rows 32 .. 32 + W - 2 close the first tile's open rows)
    + [(2, 38, 264, 15, W, True, bf16) for W in range(1, 9)]
    # channels: one octet, an octet past a wavefront's 32 and past a workgroup's 256
    + [(1, 70, D, 16, 3, True, fp16) for D in (8, 40, 264)]
    # ranks around the chunks
    + [(2, 45, 64, R, 2, st, bf16) for R, st in ((1, False), (3, True), (15, True), (17, False), (32, False))]
    # passes of 32 ranks in one launch (dx in a launch of its own): the static rank in, and alone in, the last
    + [(2, 100, 72, R, W, st, bf16) for R, W, st in ((40, 3, True), (63, 4, True), (64, 4, True), (127, 2, True),
                                                        (63, 5, True), (40, 6, False), (63, 8, True), (80, 5, True),
                                                        (64, 8, False), (127, 4, True), (96, 1, False))]
    # dx in two launches of taps over an fp32 accumulator: sequences shorter than the second's
    # first tap, of whole tiles, and off them
    + [(2, T, D, R, W, st, bf16) for T, D, R, W, st in ((5, 40, 40, 12, False), (64, 136, 63, 9, True),
                                                          (33, 264, 64, 16, False), (100, 72, 50, 13, True))]
    + [(1, 35050, 136, 40, 10, True, fp16)]
    # its runs of tiles: the dx launch's carry over tiles, the tile after a run
    + [(1, 70100, 136, 63, 4, True, bf16), (1, 70100, 136, 40, 8, True, fp16)]
    # passes of taps (dx of the earlier passes added) at one and two rank chunks, rows 32 apart from the halo
    + [(1, 97, 64, 16, 12, False, bf16), (1, 97, 64, 31, 7, True, fp16), (1, 33, 64, 20, 20, True, bf16)]
    # several runs to a sequence: the tile after a run closes its last rows
    + [(1, 9000, 64, 15, 4, True, bf16), (3, 4500, 40, 31, 4, True, fp16), (1, 9000, 64, 16, 8, False, bf16)]
)


@pytest.mark.parametrize("case", CASES, ids=[f"B{c[0]}T{c[1]}D{c[2]}R{c[3]}W{c[4]}{'s' if c[5] else ''}" for c in CASES])
def test_backward_tiles(case):
    B, T, D, R, W, static, dtype = case
    g = gen(T * 1009 + D * 7 + R + W)
    x, dy, z = randn(g, B, T, D), randn(g, B, T, D), randn(g, B, T, R)
    U = randn(g, R, W * D, scale=1 / math.sqrt((R + 1) * W))
    sw = uniform(g, W, D, lo=-1 / math.sqrt(W), hi=1 / math.sqrt(W)) if static else None
    src = [x, z, U, sw]

    def kernel(a, b, c, d, residual):  # any rank (the public function asserts a power of two)
        return lr_mod._LowrankDynamicConvolutionFn.apply(a, b, c, d, residual)

    q = [None if t is None else t.to(dtype).float() for t in src]
    y_q, g_q = run_fwd_bwd(lr_ref, q, dy.to(dtype).float(), True)
    dev = [None if t is None else t.to(dtype).cuda() for t in src]
    y_k, g_k = run_fwd_bwd(kernel, dev, dy.to(dtype).cuda(), True)
    assert_ns(y_k, y_q, dtype, "y")
    for a, b, n in zip(g_k, g_q, ["dx", "dz", "dU", "dstatic_w"]):
        if b is not None:
            assert_ns(a, b, dtype, n, elementwise=n == "dx")
    check_reductions("lr", q, dy.to(dtype).float(), g_k, dtype)
