"""proj_in over its sizes: the longest problems keep runs whose byte offsets fit (workspace query and
forward checks, on the CPU), and the backward's 16-row tiles, which take the smallest problems and the
large streams of few ranks, against the float64 sums of test_gpu_proj_in."""

import ctypes

import pytest
import torch

import helpers  # noqa: F401  (puts the package on sys.path)
from dynconv import _capi

P = 0x10000  # a fake, 256-byte aligned device pointer; never dereferenced (no device, or refused)
UNSUPPORTED, DEVICE = -4, -7


@pytest.mark.parametrize("G,M,K,R", [(3, 1048576, 8192, 31), (3, 4194304, 4096, 31), (3, 262144, 16384, 31),
                                     (1, 1048576, 8192, 15), (1, 1 << 24, 1024, 128), (1, (1 << 31) - 65, 8, 4),
                                     (4, 65536, 65536, 32)])
def test_long_problems_are_taken(G, M, K, R):
    lib = _capi.load()
    need = lib.dc_proj_in_bwd_ws_bytes(G, M, K, R, 0)
    assert need > 0 and need % (G * R * K * 4) == 0
    # runs of at most 2 GiB of rows each
    assert need // (G * R * K * 4) >= M * K * 2 / 2**31
    if not torch.cuda.is_available():
        z = (ctypes.c_void_p * G)(*[P] * G)
        assert lib.dc_proj_in_fwd(P, P, z, G, M, K, R, 0, None) == DEVICE
        assert lib.dc_proj_in_bwd(P, P, z, P, P, P, need, G, M, K, R, 0, None) == DEVICE
    assert lib.dc_proj_in_bwd_ws_bytes(G, M, 1 << 24, R, 0) == UNSUPPORTED


# M K N <= 20 Mi and past 64 MB of pre_z and dpre_z with N = G * R <= 64 (one to four 16-rank chunks, cut and
# whole; rows that end inside a tile, channels inside a wavefront's 64 and a workgroup's 256), past 400
# MB up to 96; and just past the smallest
CASES = [(1, 1, 8, 1, torch.bfloat16), (3, 17, 264, 21, torch.float16), (4, 512, 520, 16, torch.bfloat16),
         (1, 2048, 512, 20, torch.bfloat16), (1, 2049, 512, 20, torch.bfloat16), (1, 15999, 1032, 15, torch.bfloat16), (3, 16001, 1024, 15, torch.bfloat16), (4, 16016, 1000, 16, torch.float16),
         (1, 80010, 264, 1, torch.float16), (2, 8200, 2056, 31, torch.bfloat16), (1, 16385, 1024, 33, torch.bfloat16),
         (3, 100001, 1008, 31, torch.bfloat16), (1, 98307, 1024, 70, torch.float16)]


@pytest.mark.gpu
@pytest.mark.parametrize("G,M,K,R,dtype", CASES)
def test_line_tiles(G, M, K, R, dtype):
    import test_gpu_proj_in as base

    base.test_proj_in_against_float64(G, 1, M, K, R, dtype)
