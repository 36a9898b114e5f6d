"""The lowrank backward's 16-row tiles at one and two rank chunks, which take the problems that stream past
the last-level cache (x, dy and dx above 240 or 280 MB): rows that end inside a tile, sequences of
several runs with an odd number of them (two runs to a workgroup at one chunk), channels that end inside
a workgroup's 256, dy head-major, against float64 sums of the same rounded inputs on the device."""

import math

import pytest
import torch

from helpers import assert_ns_full, assert_sum
from dynconv import lowrank as lr_mod

pytestmark = pytest.mark.gpu
bf16, fp16 = torch.bfloat16, torch.float16

CASES = [(1, 640003, 64, 15, True, 4, bf16, None), (1, 630001, 64, 16, False, 1, fp16, None),
         (3, 42011, 320, 7, False, 2, bf16, None), (5, 26000, 320, 15, True, 3, bf16, None),
         (3, 210005, 64, 13, False, 4, fp16, None), (9, 2300, 1984, 3, True, 4, bf16, 64),
         (1, 126000, 320, 31, True, 1, bf16, None), (2, 74003, 320, 31, True, 4, bf16, None),
         (3, 49999, 320, 32, False, 4, fp16, 64), (2, 33000, 640, 20, False, 1, bf16, 128)]


@pytest.mark.parametrize("case", CASES, ids=[f"B{c[0]}T{c[1]}D{c[2]}R{c[3]}W{c[5]}{'h' if c[7] else ''}" for c in CASES])
def test_backward_streams(case):
    B, T, D, R, static, W, dtype, hd = case
    assert 6 * B * T * D > (240e6 if R + static <= 16 or W == 1 else 280e6)
    gen = torch.Generator(device="cuda").manual_seed(T + D + R + W)

    def randn(*s, scale=1.0):
        return (torch.randn(*s, generator=gen, device="cuda") * scale).to(dtype)

    x, dy, z = randn(B, T, D), randn(B, T, D), randn(B, T, R)
    U = randn(R, W * D, scale=1 / math.sqrt((R + 1) * W))
    sw = randn(W, D, scale=1 / math.sqrt(W)) if static else None
    dyk = dy.view(B, T, D // hd, hd).transpose(1, 2).contiguous() if hd else dy
    ps = [t.detach().requires_grad_() for t in (x, z, U, *([sw] if static else []))]
    y = lr_mod._GroupedLowrankDynamicConvolutionFn.apply(ps[0], True, 1, static, hd or 0, *ps[1:])
    got = [t.detach() for t in torch.autograd.grad(y, ps, [dyk])]

    xd, dyd, zf = x.double(), dy.double(), z.double().view(B * T, R)
    dx = dyd.clone()
    dz = [torch.zeros(B * T, R, device="cuda", dtype=torch.float64) for _ in range(3)]
    dU, ds = [[], [], []], [[], [], []]
    for k in range(W):
        Uk = U[:, k * D:(k + 1) * D].double().contiguous()
        K = (zf @ Uk).view(B, T, D)
        if static:
            K += sw[k].double()
        dx[:, :T - k] += dyd[:, k:] * K[:, k:]
        del K
        G = dyd.clone()
        G[:, :k] = 0
        G[:, k:] *= xd[:, :T - k]
        G = G.view(B * T, D)
        for i, f in enumerate((lambda t: t, torch.abs, torch.square)):
            fG = f(G)
            dU[i].append(f(zf).t().contiguous() @ fG)
            ds[i].append(fG.sum(0))
            dz[i] += fG @ f(Uk).t().contiguous()
            del fG
        del G
    assert_ns_full(got[0], dx, dtype, "dx")
    sub = 4 * 2.0**-25  # fp16: products in the subnormal range (helpers.SUM_TOL)
    ref = [torch.cat(p, 1) for p in dU]
    assert_sum(got[2], (ref[0].cpu(), ref[1].cpu(), ref[2].sqrt().cpu()), dtype, "dU",
               floor=(sub * math.sqrt(B * T) * zf.abs().amax(0)).view(R, 1).cpu())
    assert_sum(got[1], (dz[0].cpu(), dz[1].cpu(), dz[2].sqrt().cpu()), dtype, "dz",
               floor=(sub * math.sqrt(W * D) * U.double().abs().amax(1)).view(1, R).cpu())
    if static:
        ref = [torch.stack(p) for p in ds]
        assert_sum(got[3], (ref[0].cpu(), ref[1].cpu(), ref[2].sqrt().cpu()), dtype, "dstatic_w", floor=sub * math.sqrt(B * T))
