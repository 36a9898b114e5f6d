"""The lowrank forward's runs of tiles: a problem with enough tiles for the chip runs several of them
to a wavefront (rows pass from tile to tile), a smaller one a single one; the last run of a sequence
is shorter.  Against float64 sums of the same rounded inputs on the device."""

import math

import pytest
import torch

from helpers import assert_ns_full
from dynconv import lowrank as lr_mod

pytestmark = pytest.mark.gpu

# T x D in tiles of 16 x 128: 2048 wavefronts take one tile each up to 2048 tiles, then 2, .. 8
# ranks of 32 to a product: whole octets, octets and a static rank, R % 8 == 7; other ranks beside them
RANKS = [(24, True), (32, False), (23, True), (31, False), (63, True), (56, True), (64, False), (17, True), (50, False)]
CASES = [(2, T, 136, R, st, W) for T, W in ((1, 4), (31, 1), (33, 8), (70, 5)) for R, st in RANKS]
CASES += [(1, T, 264, R, st, W) for T in (10900, 11000, 40001) for R, st, W in ((15, True, 3), (31, True, 4), (16, False, 8),
                                                                             (40, False, 5), (15, True, 12))]


@pytest.mark.parametrize("B,T,D,R,static,W", CASES)
def test_forward_runs(B, T, D, R, static, W):
    g = torch.Generator(device="cuda").manual_seed(T + R + W)

    def n(*s, scale=1.0):
        return (torch.randn(*s, generator=g, device="cuda") * scale).to(torch.bfloat16)

    x, z = n(B, T, D), n(B, T, R)
    U = n(R, W * D, scale=1 / math.sqrt((R + 1) * W))
    sw = n(W, D, scale=1 / math.sqrt(W)) if static else None
    with torch.no_grad():
        y = lr_mod._LowrankDynamicConvolutionFn.apply(x, z, U, sw, True)
    ref = x.double()
    for k in range(W):
        K = (z.double().view(B * T, R) @ U[:, k * D:(k + 1) * D].double().contiguous()).view(B, T, D)
        if static:
            K += sw[k].double()
        ref[:, k:] += K[:, k:] * x[:, :T - k].double()
    assert_ns_full(y, ref, torch.bfloat16, "y")
