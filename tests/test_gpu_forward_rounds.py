"""Run lengths of the lowrank forward at two and four rank chunks.

The forward's tiles per run are chosen by a model of whole rounds of workgroups
(t32_fwd_run_tiles, csrc/lowrank_mfma_t32.h), so a batch and each of its sequences
run with different lengths.  A row of y and of the z_eff copy depends on its own
rows only: the batch's must be those of the sequences, bit for bit, and those of a
short call, whose runs are one tile, must be the oracle's (test_gpu_parity.py).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(3, 4788, 3712), (4, 4096, 2560), (5, 1003, 1416)]


@pytest.mark.parametrize("B,T,D", SHAPES)
@pytest.mark.parametrize("R,static,W", [(32, False, 4), (31, True, 3), (31, True, 8), (63, True, 4), (64, False, 6),
                                        (63, True, 8)])
def test_rows_do_not_depend_on_runs(B, T, D, R, static, W):
    from dynconv import _capi
    lib = _capi.load()
    g = torch.Generator(device="cuda").manual_seed(B * T + W)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(torch.bfloat16)
    x, z, U = rnd(B, T, D), rnd(B, T, R), rnd(R, W * D) * 0.1
    sw = rnd(W, D) if static else None

    def fwd(x, z):
        b, t = x.shape[:2]
        n = max(lib.dc_lowrank_zeff_bytes(b, t, D, R, W, 0, int(static)), 0)
        y = torch.full_like(x, float("nan"))
        ze = torch.zeros(max(n, 16), dtype=torch.uint8, device="cuda")
        st = lib.dc_lowrank_fwd(x.data_ptr(), z.data_ptr(), U.data_ptr(), sw.data_ptr() if static else None,
                                y.data_ptr(), ze.data_ptr() if n else None, n, b, t, D, R, W, 0, 1,
                                torch.cuda.current_stream().cuda_stream)
        assert st == 0, lib.dc_status_string(st) if hasattr(lib, "dc_status_string") else st
        return y, ze[:n]

    y, ze = fwd(x, z)
    assert not y.isnan().any()
    for b in range(B):
        yb, zb = fwd(x[b:b + 1].contiguous(), z[b:b + 1].contiguous())
        assert torch.equal(y[b:b + 1], yb)
        k = ze.numel() // B
        assert torch.equal(ze[b * k:(b + 1) * k], zb)
    # a short head of the last sequence: runs of one tile
    n = 200
    yh, _ = fwd(x[-1:, :n].contiguous(), z[-1:, :n].contiguous())
    assert torch.equal(y[-1:, :n], yh)
