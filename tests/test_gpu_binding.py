"""The native autograd binding (csrc/torch_binding.cpp): bitwise the results of the Python Functions it
stands in for, the same behaviour under autograd's own machinery, and None (the Python path, with its
errors) for every call that it does not take."""

import math
import threading

import pytest
import torch

import helpers  # noqa: F401  (puts the package on sys.path)
from dynconv import _capi
from dynconv import headwise as hw_mod
from dynconv import lowrank as lr_mod
from dynconv.modules import GroupedLowRankDynamicShortConvolution

pytestmark = pytest.mark.gpu
bf16, fp16, fp32 = torch.bfloat16, torch.float16, torch.float32


def _rand(seed, *shape, dtype=bf16, scale=1.0, grad=True):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype).requires_grad_(grad)


def _hw(dtype=bf16, static=True, T=70):
    x, w = _rand(1, 2, T, 64, dtype=dtype), _rand(2, 2, T, 16, 4, dtype=dtype, scale=0.5)
    return x, w, (_rand(3, 4, 64, dtype=dtype, scale=0.5) if static else None)


def _lr(dtype=bf16, static=True, T=70):
    R = 15 if static else 16
    return (_rand(1, 2, T, 64, dtype=dtype), _rand(2, 2, T, R, dtype=dtype), _rand(3, R, 256, dtype=dtype, scale=0.1),
            _rand(4, 4, 64, dtype=dtype, scale=0.5) if static else None)


@pytest.fixture(autouse=True)
def _loaded():
    _capi.load()
    assert _capi.binding is not None, "dynconv/_binding.so is missing or built for another torch"


def _grads(y, args, dy):
    return torch.autograd.grad(y, [a for a in args if a is not None], dy)


@pytest.mark.parametrize("dtype", [bf16, fp16, fp32])
@pytest.mark.parametrize("static", [True, False])
@pytest.mark.parametrize("residual", [True, False])
def test_same_as_functions(dtype, static, residual):
    for make, native, fn in ((_hw, "headwise", hw_mod._HeadwiseDynamicConvolutionFn),
                             (_lr, "lowrank", lr_mod._LowrankDynamicConvolutionFn)):
        args = make(dtype, static)
        y = getattr(_capi.binding, native)(*args, residual)
        assert y is not None and y.grad_fn is not None
        r = fn.apply(*args, residual)
        dy = _rand(9, *y.shape, dtype=dtype, grad=False)
        assert torch.equal(y, r)
        for a, b in zip(_grads(y, args, dy), _grads(r, args, dy)):
            assert a.dtype == b.dtype and torch.equal(a, b)
        with torch.no_grad():
            n = getattr(_capi.binding, native)(*args, residual)
        assert n.grad_fn is None and torch.equal(n, r)
        with torch.inference_mode():
            assert torch.equal(getattr(_capi.binding, native)(*args, residual), r)


@pytest.mark.parametrize("head_dim", [None, 64])
@pytest.mark.parametrize("dtype,R", [(bf16, 15), (fp16, 31), (bf16, 7)])
def test_grouped_module(head_dim, dtype, R, monkeypatch):
    D, G, B, T = 128, 3, 2, 75
    m = GroupedLowRankDynamicShortConvolution(D, R, 4, groups=G, head_dim=head_dim).to("cuda", dtype)
    with torch.no_grad():
        m.proj_out.copy_(_rand(5, G, R, 4 * D, dtype=dtype, scale=0.1))
    wide = _rand(6, B, T, G * D + 8, dtype=dtype)  # rows further apart than G * D
    pre = _rand(7, B, T, D, dtype=dtype)
    leaves = [wide, pre, *m.parameters()]
    dys = [_rand(20 + g, B, *((T, D) if head_dim is None else (D // head_dim, T, head_dim)), dtype=dtype, grad=False)
           for g in range(G)]
    ys = m(wide[..., :G * D], pre)
    got = torch.autograd.grad(ys, leaves, dys)
    only = torch.autograd.grad(m(wide[..., :G * D], pre)[1], leaves, dys[1])  # the other outputs have no gradient
    monkeypatch.setattr(_capi, "binding", None)
    ref = m(wide[..., :G * D], pre)
    for a, b in zip(ys, ref):
        assert a.shape == b.shape and torch.equal(a, b)
    for a, b in zip(got, torch.autograd.grad(ref, leaves, dys)):
        assert torch.equal(a, b)
    for a, b in zip(only, torch.autograd.grad(m(wide[..., :G * D], pre)[1], leaves, dys[1])):
        assert torch.equal(a, b)


def test_declined_calls_take_the_python_path():
    x, w, sw = _hw()
    b = _capi.binding

    class Sub(torch.Tensor):
        pass

    assert b.headwise(x.detach().as_subclass(Sub), w, sw, True) is None
    assert b.headwise(x.cpu(), w.cpu(), sw.cpu(), True) is None
    assert b.headwise(x, w.float(), sw, True) is None                      # mixed dtypes
    assert b.headwise(x, w.transpose(2, 3).contiguous().transpose(2, 3), sw, True) is None  # non-contiguous weight
    assert b.headwise(x, w, sw.t().contiguous().t(), True) is None
    assert b.headwise(x[:, ::2], w, sw, True) is None
    assert b.headwise(x, None, sw, True) is None
    xl, z, U, s = _lr()
    assert b.lowrank(xl, z[..., :14].contiguous(), U[:14].contiguous(), s, True) is None  # rank + 1 no power of two
    assert b.lowrank(xl, z, U, s.float(), True) is None
    with pytest.raises(AssertionError):
        lr_mod.lowrank_dynamic_convolution(xl, z[..., :14].contiguous(), U[:14].contiguous(), s)
    with pytest.raises(AssertionError):
        hw_mod.headwise_dynamic_convolution(x[:, ::2], w, sw)
    # function transforms and forward-mode derivatives have no rule for the operators: still refused
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: hw_mod.headwise_dynamic_convolution(t, w.detach(), sw.detach()))(x.detach()[None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: hw_mod.headwise_dynamic_convolution(t, w.detach(), sw.detach()).sum())(x.detach())
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x))
        assert b.headwise(d, w, sw, True) is None
        with pytest.raises(Exception):
            hw_mod.headwise_dynamic_convolution(d, w, sw)


def test_autograd_machinery():
    args = _lr()
    dy = _rand(9, 2, 70, 64, grad=False)
    ref = _grads(lr_mod._LowrankDynamicConvolutionFn.apply(*args, True), args, dy)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(), lambda t: t.cuda()):
        y = lr_mod.lowrank_dynamic_convolution(*args, residual=True)
    assert len(packed) == 4
    for a, b in zip(_grads(y, args, dy), ref):
        assert torch.equal(a, b)
    y = lr_mod.lowrank_dynamic_convolution(*args, residual=True)
    first = torch.autograd.grad(y, args, dy, retain_graph=True)
    for a, b, c in zip(first, torch.autograd.grad(y, args, dy), ref):
        assert torch.equal(a, c) and torch.equal(b, c)
    with pytest.raises(RuntimeError):  # freed
        torch.autograd.grad(y, args, dy)
    y = lr_mod.lowrank_dynamic_convolution(*args, residual=True)
    with torch.no_grad():
        args[1].add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(y, args, dy)
    # one input alone requires a gradient, a strided output gradient of another dtype
    x, w, sw = (t.detach() for t in _hw())
    w.requires_grad_()
    g = _rand(10, 2, 64, 70, grad=False).transpose(1, 2)
    a = torch.autograd.grad(hw_mod.headwise_dynamic_convolution(x, w, sw), w, g)[0]
    b = torch.autograd.grad(hw_mod._HeadwiseDynamicConvolutionFn.apply(x, w, sw, False), w, g)[0]
    assert torch.equal(a, b)


def test_streams_and_threads():
    args = _hw(T=600)
    dy = _rand(9, 2, 600, 64, grad=False)
    ref = _grads(hw_mod._HeadwiseDynamicConvolutionFn.apply(*args, True), args, dy)
    torch.cuda.synchronize()
    out, errors = {}, []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(5):
                    out[k] = _grads(hw_mod.headwise_dynamic_convolution(*args, residual=True), args, dy)
                torch.cuda.current_stream().synchronize()
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors
    for k in range(4):
        for a, b in zip(out[k], ref):
            assert torch.equal(a, b)


def test_kernel_error_is_a_runtime_error():
    x = torch.zeros(1, 4, 8, device="cuda", dtype=bf16)
    w = torch.zeros(1, 4, 8, 1025, device="cuda", dtype=bf16)  # W past DC_MAX_W
    with pytest.raises(RuntimeError, match="dynconv headwise forward failed"):
        hw_mod.headwise_dynamic_convolution(x, w)
    assert math.isfinite(float(x.sum()))
