"""What autograd may do around the training functions that stand in for chains
of torch operations, on the CPU: their kernels are replaced by stand-ins of
the same contract, which read their operands by address as the kernels do."""
import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from src.model import kernels
from src.model.chassis import RMSNorm, RMSNormFunction
from src.model.linear import FewRowsLinear


def _floats(ptr, n):
    return torch.from_numpy(np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_float)), (n,)).copy())


def _bf16(ptr, n):
    raw = np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_int16)), (n,)).copy()
    return torch.from_numpy(raw).view(torch.bfloat16)


def _store(ptr, t):
    if ptr:
        ctypes.memmove(ptr, t.contiguous().data_ptr(), t.numel() * t.element_size())


class _Lib:
    def __getattr__(self, name):
        return lambda *a: 64


def _call(name, *a, **kw):
    """walsh_rmsnorm_fwd / _bwd on host memory, with their alignment checks."""
    x, w, M, C = (a[0], a[1], a[2], a[3]) if name == "walsh_rmsnorm_fwd" else (a[0], a[1], a[4], a[5])
    assert x % 8 == 0 and w % 16 == 0
    xf, wf = _bf16(x, M * C).view(M, C).float(), _floats(w, C) if w else None
    if name == "walsh_rmsnorm_fwd":
        r = torch.rsqrt(xf.pow(2).mean(-1) + a[4])
        _store(a[5], (xf * r[:, None]).bfloat16().float() * wf)
        _store(a[6], r)
        return
    assert name == "walsh_rmsnorm_bwd" and a[3] % 16 == 0 and a[6] % 8 == 0
    r, gy = _floats(a[2], M)[:, None], _floats(a[3], M * C).view(M, C)
    if a[6]:
        g = (gy * wf).bfloat16().float()
        _store(a[6], (g * r - xf * r.pow(3) * (g * xf).mean(-1, keepdim=True)).bfloat16())
    _store(a[7], (gy * (xf * r).bfloat16().float()).sum(0))


@pytest.fixture
def norm(monkeypatch):
    """(fused, plain) RMSNorm of one weight on bf16 rows of 8 columns."""
    monkeypatch.setattr(kernels._hip, "call", _call)
    monkeypatch.setattr(kernels._hip, "lib", lambda: _Lib())
    monkeypatch.setattr(kernels._hip, "stream", lambda d: 0)
    monkeypatch.setattr(kernels._hip, "require_device", lambda t, what="": None)
    torch.manual_seed(0)
    m = RMSNorm(8)
    with torch.no_grad():
        m.weight.uniform_(0.5, 1.5)
    return m, lambda x: RMSNormFunction.apply(x.clone(), m.weight, m.eps), lambda x: m(x)


def _close(a, b):
    for u, v in zip(a, b):
        u, v = u.detach().float(), v.detach().float()
        assert torch.allclose(u, v, rtol=2.0 ** -6, atol=2.0 ** -7 * float(v.abs().max()))


def _rows(n=5):
    return torch.randn(n, 8).bfloat16().requires_grad_(True)


@pytest.mark.parametrize("rows", [1, 5])
def test_rmsnorm_gradient_at_any_offset(norm, rows):
    """A gradient that arrives as a contiguous view 12 bytes past an aligned
    address (the norm's output flattened behind three other values)."""
    m, fused, plain = norm
    x, head, g = _rows(rows), torch.zeros(3), torch.randn(3 + rows * 8)
    close = [torch.autograd.grad(torch.cat([head, f(x).reshape(-1)]), (x, m.weight), g) for f in (fused, plain)]
    _close(*close)


def test_rmsnorm_saved_tensor_hooks(norm):
    """Hooks that give the saved rows back in another layout or off alignment."""
    m, fused, plain = norm
    x, g = _rows(), torch.randn(5, 8)
    ref = torch.autograd.grad(plain(x), (x, m.weight), g)

    def shifted(t):
        return torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)
    for pack, unpack in ((lambda t: t.t().contiguous() if t.dim() == 2 else t,
                          lambda t: t.t() if t.dim() == 2 else t), (lambda t: t, shifted)):
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = fused(x)
        _close(torch.autograd.grad(y, (x, m.weight), g), ref)


def _linear(w):
    return lambda x: FewRowsLinear.apply(x, w), lambda x: F.linear(x, w.to(x.dtype))


@pytest.fixture
def wgrad(monkeypatch):
    def call(name, g, x, M, N, K, dw, *rest, **kw):
        assert name == "walsh_linear_wgrad" and x % 16 == 0
        _store(dw, _bf16(g, M * N).view(M, N).float().t() @ _bf16(x, M * K).view(M, K).float())
    monkeypatch.setattr(kernels._hip, "call", call)
    monkeypatch.setattr(kernels._hip, "lib", lambda: _Lib())
    monkeypatch.setattr(kernels._hip, "stream", lambda d: 0)
    monkeypatch.setattr(kernels._hip, "require_device", lambda t, what="": None)
    torch.manual_seed(1)
    return torch.randn(6, 8).requires_grad_(True)


def test_few_rows_linear_weight_updated_before_backward(wgrad):
    """Two forwards before an optimizer step, or a step between a forward and
    its backward: the gradients belong to the weight of the forward."""
    w = wgrad
    x, g = _rows(), torch.randn(5, 6).bfloat16()
    got = []
    for f in _linear(w):
        y = f(x)
        before = w.detach().clone()
        with torch.no_grad():
            w.mul_(-3.0)
        got.append((y,) + torch.autograd.grad(y, (x, w), g))
        with torch.no_grad():
            w.copy_(before)
    _close(*got)
    second = []
    for f in _linear(w):
        gx, gw = torch.autograd.grad(f(x).float().square().sum(), (x, w), create_graph=True)
        second.append(torch.autograd.grad(gx.float().square().sum() + gw.square().sum(), (x, w)))
    _close(*second)


def test_few_rows_linear_saved_tensor_hooks(wgrad):
    x, g = _rows(), torch.randn(5, 6).bfloat16()
    f, plain = _linear(wgrad)
    ref = torch.autograd.grad(plain(x), (x, wgrad), g)
    for pack, unpack in ((lambda t: t.t().contiguous(), lambda t: t.t()),
                         (lambda t: t, lambda t: torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape))):
        with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
            y = f(x)
        _close(torch.autograd.grad(y, (x, wgrad), g), ref)


def test_rmsnorm_gain_updated_before_backward(norm):
    """Rows without a gradient: the gain's own gradient does not depend on it,
    and it may change between the forward and the backward."""
    m, fused, plain = norm
    x, g = _rows().detach(), torch.randn(5, 8)
    got = []
    for f in (fused, plain):
        y = f(x)
        with torch.no_grad():
            m.weight.mul_(2.0)
        got.append(torch.autograd.grad(y, (m.weight,), g))
    _close(*got)


@pytest.mark.parametrize("wrt", [(0, 1), (0,), (1,)])
def test_rmsnorm_differentiated_backward(norm, wrt):
    m, fused, plain = norm
    x = _rows()
    ins = [(x, m.weight)[i] for i in wrt]
    if 0 not in wrt:
        x = x.detach()
    got = []
    for f in (fused, plain):
        first = torch.autograd.grad(f(x).pow(3).sum(), ins, create_graph=True)
        got.append(first + torch.autograd.grad(sum(v.float().square().sum() for v in first), ins))
    _close(*got)


def _batched(y, ins, gs):
    return torch.autograd.grad(y, ins, gs, is_grads_batched=True)


def test_rmsnorm_batched_gradients(norm):
    m, fused, plain = norm
    x, gs = _rows(), torch.randn(3, 5, 8)
    _close(_batched(fused(x), (x, m.weight), gs), _batched(plain(x), (x, m.weight), gs))
    jac = [torch.autograd.functional.jacobian(f, x.detach(), vectorize=True) for f in (fused, plain)]
    _close(*([j] for j in jac))


def test_few_rows_linear_batched_gradients(wgrad):
    x, gs = _rows(), torch.randn(3, 5, 6).bfloat16()
    f, plain = _linear(wgrad)
    _close(_batched(f(x), (x, wgrad), gs), _batched(plain(x), (x, wgrad), gs))


def test_backward_under_a_dispatch_mode(norm):
    """A mode around the backward alone sees its operations, and a functional
    transform of a whole step keeps the plain form's values."""
    from torch.utils._python_dispatch import TorchDispatchMode
    m, fused, plain = norm
    x, g = _rows(), torch.randn(5, 8)

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    seen, y = [], fused(x)
    with Seen():
        got = torch.autograd.grad(y, (x, m.weight), g)
    assert len(seen) > 5
    _close(got, torch.autograd.grad(plain(x), (x, m.weight), g))
