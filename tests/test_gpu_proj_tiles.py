"""proj_in's backward on 32-row tiles: rows around a tile, one to four groups, ranks that fill one to
four pairs per staging thread and end inside a 16- and a 32-rank chunk, channels that end inside a
wavefront's 32, against the float64 sums of test_gpu_proj_in."""

import pytest
import torch

import test_gpu_proj_in as base

pytestmark = pytest.mark.gpu

CASES = [(G, 1, M, K, R, dt)
         for (G, R, dt), (M, K) in zip(
             [(1, 128, torch.bfloat16), (1, 1, torch.float16), (1, 97, torch.bfloat16), (2, 64, torch.bfloat16),
              (2, 33, torch.float16), (3, 42, torch.bfloat16), (3, 5, torch.bfloat16), (4, 31, torch.float16),
              (4, 1, torch.bfloat16), (4, 32, torch.bfloat16), (1, 16, torch.bfloat16), (3, 16, torch.bfloat16)],
             [(65, 264), (1, 8), (31, 40), (32, 264), (33, 296), (64, 520), (4100, 264), (700, 1032), (97, 24),
              (2000, 72), (129, 248), (63, 256)])]


@pytest.mark.parametrize("G,B,T,K,R,dtype", CASES)
def test_proj_tiles(G, B, T, K, R, dtype):
    base.test_proj_in_against_float64(G, B, T, K, R, dtype)
