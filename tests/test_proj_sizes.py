"""proj_in over its sizes: the longest problems keep runs whose byte offsets fit (workspace query and
forward checks, on the CPU)."""

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

