"""Host side of the native binding, without a GPU: what the module hands to it."""

import types

import pytest
import torch

import helpers  # noqa: F401  (puts the package on sys.path)
from dynconv import _capi
from dynconv.modules import GroupedLowRankDynamicShortConvolution


@pytest.mark.parametrize("head_dim", [None, 32, 32.0])
def test_module_head_dim(head_dim, monkeypatch):
    """A head dim that is a whole float reaches the binding as the int that the Python path makes of it."""
    seen = []
    fake = types.SimpleNamespace(grouped_module=lambda *a: seen.append(a[-1]) or "ys")
    monkeypatch.setattr(_capi, "binding", fake)
    m = GroupedLowRankDynamicShortConvolution(64, 7, 4, groups=2, head_dim=head_dim)
    assert m(torch.zeros(1, 3, 128), torch.zeros(1, 3, 64)) == "ys"
    assert seen == [None if head_dim is None else 32] and not isinstance(seen[0], float)
