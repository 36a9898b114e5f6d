"""The fp32 lowrank kernels' runs of tiles: one tile to a run, two, several with a shorter last one,
more sequences than a round of workgroups (and than eight) holds, passes of taps and of ranks over
them, against the CPU oracle."""

import math

import pytest
import torch

from helpers import assert_ns, check_reductions, gen, randn, run_fwd_bwd, uniform
from dynconv import lowrank as lr_mod
from oracle.reference_cpu import lowrank_dynamic_convolution_ref as lr_ref

pytestmark = pytest.mark.gpu

CASES = [
    (2, 512, 256, 15, 4, True), (1, 17, 64, 16, 3, False), (3, 500, 136, 7, 2, True),  # one tile to a run
    (2, 1024, 512, 16, 4, False), (5, 1000, 256, 7, 3, True),  # two
    (1, 5005, 520, 15, 8, True), (2, 3000, 768, 15, 2, True),  # several, the last one shorter
    (1, 1000, 64, 15, 12, True), (2, 700, 264, 31, 4, True), (1, 400, 64, 63, 5, True),  # passes
    (300, 40, 64, 8, 2, False), (2100, 17, 8, 3, 2, True),  # rounds of sequences
]


@pytest.mark.parametrize("case", CASES, ids=[f"B{c[0]}T{c[1]}D{c[2]}R{c[3]}W{c[4]}{'s' if c[5] else ''}" for c in CASES])
def test_fp32_runs(case):
    B, T, D, R, W, static = case
    dtype = torch.float32
    g = gen(T * 1009 + D * 7 + R + W)
    x, dy, z = randn(g, B, T, D), randn(g, B, T, D), randn(g, B, T, R)
    U = randn(g, R, W * D, scale=1 / math.sqrt((R + 1) * W))
    sw = uniform(g, W, D, lo=-1 / math.sqrt(W), hi=1 / math.sqrt(W)) if static else None
    src = [x, z, U, sw]

    def kernel(a, b, c, d, residual):  # any rank (the public function asserts a power of two)
        return lr_mod._LowrankDynamicConvolutionFn.apply(a, b, c, d, residual)

    y_q, g_q = run_fwd_bwd(lr_ref, src, dy, True)
    y_k, g_k = run_fwd_bwd(kernel, [None if t is None else t.cuda() for t in src], dy.cuda(), True)
    assert_ns(y_k, y_q, dtype, "y")
    for a, b, n in zip(g_k, g_q, ["dx", "dz", "dU", "dstatic_w"]):
        if b is not None:
            assert_ns(a, b, dtype, n, elementwise=n == "dx")
    check_reductions("lr", src, dy, g_k, dtype)
