"""The headwise kernels' runs of rows where the plan stretches them to keep the launch within one
round of workgroups (the forward below W 6 by up to a quarter, else by at least one step), and where it does
not, against the CPU oracle."""

import math

import pytest
import torch

from helpers import assert_ns, check_reductions, gen, randn, run_fwd_bwd, uniform
from headwise import headwise_dynamic_convolution as hw
from oracle.reference_cpu import headwise_dynamic_convolution_ref as hw_ref

pytestmark = pytest.mark.gpu
bf16, fp32 = torch.bfloat16, torch.float32

# B, T, D, W, head size, static, dtype: the backward's runs one step longer than the forward's, ...
CASES = [(3, 1365, 112, 4, 1, True, fp32), (5, 2042, 64, 5, 8, True, bf16), (5, 1225, 120, 3, 4, False, bf16),
         (3, 455, 520, 2, 1, True, fp32), (5, 1633, 112, 8, 1, True, fp32),
         # ... and both longer by up to a quarter
         (3, 2045, 568, 3, 1, True, bf16), (5, 1633, 576, 4, 32, True, bf16), (5, 1225, 272, 3, 16, False, fp32)]


@pytest.mark.parametrize("case", CASES, ids=[f"B{c[0]}T{c[1]}D{c[2]}W{c[3]}h{c[4]}" for c in CASES])
def test_headwise_runs(case):
    B, T, D, W, hs, static, dtype = case
    g = gen(T * 1009 + D * 7 + W)
    x, dy = randn(g, B, T, D), randn(g, B, T, D)
    w = randn(g, B, T, D // hs, W, scale=1 / math.sqrt(W))
    sw = uniform(g, W, D, lo=-1 / math.sqrt(W), hi=1 / math.sqrt(W)) if static else None
    q = [None if t is None else t.to(dtype).float() for t in (x, w, sw)]
    y_q, g_q = run_fwd_bwd(hw_ref, q, dy.to(dtype).float(), True)
    y_k, g_k = run_fwd_bwd(hw, [None if t is None else t.to(dtype).cuda() for t in q], dy.to(dtype).cuda(), True)
    assert_ns(y_k, y_q, dtype, "y")
    for a, b, n in zip(g_k, g_q, ["dx", "dweight", "dstatic_w"]):
        if b is not None:
            assert_ns(a, b, dtype, n, elementwise=n != "dstatic_w")
    check_reductions("hw", q, dy.to(dtype).float(), g_k, dtype)
