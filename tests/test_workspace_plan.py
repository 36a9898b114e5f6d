"""The lowrank backward's workspace against its launch plan, over the row strides that the size query does
not see.  A run's buffer resources hold fewer rows of a wider x or dx, so a strided call can have more
runs, each with a dU partial of its own, than the query's plan: it then runs in parts over the slots
there are.  On the CPU the plan's ends stay inside the queried bytes; on the GPU such calls give what
the contiguous one gives."""

import ctypes
import itertools
import math

import pytest
import torch

from helpers import check_reductions
from dynconv import _capi
from dynconv import lowrank as lr_mod

bf16, fp16, fp32 = torch.bfloat16, torch.float16, torch.float32


def _ranges(lib, B, T, D, R, W, dt, st, x_ld, dx_ld, hd, ws):
    fn = lib.dc_lowrank_strided_plan_ranges
    fn.restype = ctypes.c_int64
    fn.argtypes = [ctypes.c_int64] * 5 + [ctypes.c_int] * 3 + [ctypes.c_int64] * 4 + [ctypes.c_void_p, ctypes.c_int64]
    n = fn(B, T, D, R, W, dt, st, 1, x_ld, dx_ld, hd, ws, None, 0)
    assert n >= 0, n
    buf = (ctypes.c_int64 * (2 * max(n, 1)))()
    assert fn(B, T, D, R, W, dt, st, 1, x_ld, dx_ld, hd, ws, buf, n) == n
    return [(buf[2 * i], buf[2 * i + 1]) for i in range(n)]


def _check(lib, B, T, D, R, W, dt, st, x_ld, dx_ld, hd):
    ws = lib.dc_lowrank_bwd_ws_bytes(B, T, D, R, W, dt, st)
    assert ws > 0
    pairs = _ranges(lib, B, T, D, R, W, dt, st, x_ld, dx_ld, hd, ws)
    for i, (v, bound) in enumerate(pairs):
        assert 0 <= v <= bound, (dict(B=B, T=T, D=D, R=R, W=W, dt=dt, st=st, x_ld=x_ld, dx_ld=dx_ld, hd=hd), i, v, bound)
    return len(pairs)


def test_plan_fits_the_queried_workspace():
    lib = _capi.load()
    n = 0
    # runs of hundreds of tiles: a fused projection of four groups, a slice of a wide tensor
    for B, T, D in ((16, 8192, 4096), (16, 16384, 4096), (8, 16384, 4096), (1, 900, 32768), (1, 33, 65536), (64, 4096, 512)):
        for dt, (R, st), W in itertools.product((0, 1, 2), ((15, 1), (16, 0), (31, 1), (40, 0), (63, 1), (95, 1)),
                                                (1, 2, 4, 6, 8, 12, 20)):
            for x_ld, dx_ld in ((D, D), (3 * D, 3 * D), (4 * D, 4 * D), (34304, D), (D, 34304), (1 << 18, D), (1 << 19, 1 << 19)):
                for hd in (0, 128):
                    n += _check(lib, B, T, D, R, W, dt, st, max(x_ld, D), max(dx_ld, D), hd)
    assert n > 10000


# runs capped below the contiguous plan's: three runs on two slots, four on two, five on four; one and two
# rank chunks, passes of taps, three chunks on 16-row tiles, passes of ranks with dx apart, fp32
CASES = [(bf16, 1, 900, 32768, 7, True, 3, 1, 1 << 19, None), (fp16, 1, 1300, 32768, 24, False, 2, 1, 1 << 19, None),
         (bf16, 1, 900, 32768, 15, True, 9, 1, 1 << 19, None), (bf16, 1, 900, 32768, 40, False, 1, 1, 1 << 20, None),
         (bf16, 1, 900, 32768, 35, True, 3, 1, 1 << 19, None), (bf16, 1, 1700, 16384, 4, False, 2, 2, 1 << 19, 128),
         (fp32, 1, 900, 32768, 7, True, 3, 1, 1 << 18, None), (fp32, 1, 900, 32768, 20, False, 5, 1, 1 << 18, None)]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[f"{str(c[0])[6:]}T{c[2]}D{c[3]}R{c[4]}W{c[6]}G{c[7]}" for c in CASES])
def test_runs_in_parts(case):
    dtype, B, T, D, R, static, W, G, x_ld, hd = case
    lib = _capi.load()
    dt = _capi.DTYPE_CODES[dtype]
    # the plan has more parts than the contiguous one
    assert (_check(lib, B, T, D, R, W, dt, int(static), x_ld, G * D, hd or 0)
            > _check(lib, B, T, D, R, W, dt, int(static), G * D, G * D, hd or 0))
    gen = torch.Generator(device="cuda").manual_seed(T + R + W)

    def randn(*s, scale=1.0):
        return (torch.randn(*s, generator=gen, device="cuda") * scale).to(dtype)

    wide = torch.zeros(B, T, x_ld, device="cuda", dtype=dtype)
    wide[..., :G * D] = randn(B, T, G * D)
    x = wide[..., :G * D]
    z = [randn(B, T, R) for _ in range(G)]
    U = [randn(R, W * D, scale=1 / math.sqrt((R + 1) * W)) for _ in range(G)]
    sw = [randn(W, D, scale=1 / math.sqrt(W)) for _ in range(G)] if static else None
    dy = [randn(B, T, D) for _ in range(G)]
    if hd:
        dyk = [t.view(B, T, D // hd, hd).transpose(1, 2).contiguous() for t in dy]
    else:
        dyk = dy

    def grads(x):
        ps = [t.detach().requires_grad_() for t in (x, *z, *U, *(sw or []))]
        # any rank (the public function asserts a power of two)
        ys = lr_mod._GroupedLowrankDynamicConvolutionFn.apply(ps[0], True, G, static, hd or 0, *ps[1:])
        return torch.autograd.grad(ys, ps, dyk)

    got, ref = grads(x), grads(x.contiguous())
    assert torch.equal(got[0], ref[0])                     # dx and dz: row by row, whatever the runs
    for a, b in zip(got[1:1 + G], ref[1:1 + G]):
        assert torch.equal(a, b)
    for g in range(G):                                     # dU, dstatic_w: sums over the runs
        cpu = [t.float().cpu() for t in (x[..., g * D:(g + 1) * D], z[g], U[g])]
        cpu.append(sw[g].float().cpu() if static else None)
        check_reductions("lr", cpu, dy[g].float().cpu(),
                         [None, got[1 + g], got[1 + G + g], got[1 + 2 * G + g] if static else None], dtype)
