"""The grouped module's native node with some of its inputs frozen: the gradients that are wanted are bitwise
those of the Python Functions, and a frozen projection (neither pre_z nor proj_in.weight wanted) has no
backward of its own: no gradient of pre_z is allocated."""

import pytest
import torch

import helpers  # noqa: F401  (puts the package on sys.path)
from dynconv import _capi
from dynconv.modules import GroupedLowRankDynamicShortConvolution

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _setup(D=256, G=3, R=15, W=4, B=2, T=75):
    g = torch.Generator(device="cuda").manual_seed(D + T)
    m = GroupedLowRankDynamicShortConvolution(D, R, W, groups=G).to("cuda", bf16)
    with torch.no_grad():
        m.proj_out.copy_(torch.randn(G, R, W * D, generator=g, device="cuda") * 0.1)
    x = torch.randn(B, T, G * D, generator=g, device="cuda").to(bf16)
    pre = torch.randn(B, T, D, generator=g, device="cuda").to(bf16)
    dys = [torch.randn(B, T, D, generator=g, device="cuda").to(bf16) for _ in range(G)]
    return m, x, pre, dys


WANTED = [("x",), ("pre",), ("w",), ("U",), ("b",), ("x", "U", "b"), ("pre", "w"), ("x", "w"), ("x", "pre", "w", "U", "b")]


@pytest.mark.parametrize("wanted", WANTED, ids="-".join)
def test_partly_frozen(wanted, monkeypatch):
    _capi.load()
    assert _capi.binding is not None
    m, x, pre, dys = _setup()
    inputs = {"x": x, "pre": pre, "w": m.proj_in.weight, "U": m.proj_out, "b": m.proj_out_bias}
    for n, t in inputs.items():
        t.requires_grad_(n in wanted)
    leaves = [inputs[n] for n in wanted]
    got = torch.autograd.grad(m(x, pre), leaves, dys)
    monkeypatch.setattr(_capi, "binding", None)
    for a, b in zip(got, torch.autograd.grad(m(x, pre), leaves, dys)):
        assert torch.equal(a, b)


def test_frozen_projection_allocates_no_gradient():
    m, x, pre, dys = _setup(D=1024, G=1, B=2, T=2048)
    x.requires_grad_()

    def peak(frozen):
        pre.requires_grad_(not frozen)
        m.proj_in.weight.requires_grad_(not frozen)
        leaves = [x] if frozen else [x, pre]
        y = m(x, pre)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        torch.autograd.grad(y, leaves, dys)
        torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - before

    # the caching allocator leaves a remainder of up to 1 MB in a block; the frozen pass has four large ones
    # (dx, dU with dstatic_w, dz, the workspace)
    assert peak(True) + pre.numel() * 2 - 4 * 2**20 <= peak(False)


def test_one_wanted_of_several_is_all_the_engine_asks(monkeypatch):
    """autograd.grad on x alone, the projection not frozen: its backward is not asked for either."""
    m, x, pre, dys = _setup()
    x.requires_grad_()
    pre.requires_grad_()
    got = torch.autograd.grad(m(x, pre), [x], dys)[0]
    monkeypatch.setattr(_capi, "binding", None)
    assert torch.equal(got, torch.autograd.grad(m(x, pre), [x], dys)[0])
