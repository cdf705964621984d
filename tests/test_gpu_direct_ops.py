"""Ops called without the dispatcher (tsfast_amd/ops.py): everything a dispatched call would show or
handle still is, and the direct call gives the dispatched call's bits."""

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from tsfast_amd import ops, scan

pytestmark = pytest.mark.gpu


def _inputs(dev, cplx=True):
    g = torch.Generator().manual_seed(3)
    lam = torch.polar(torch.rand(6, generator=g) * 0.1 + 0.85, torch.rand(6, generator=g))
    v, gy = torch.randn(2, 50, 6, dtype=torch.complex64, generator=g), torch.randn(2, 50, 6, dtype=torch.complex64, generator=g)
    return (lam.to(dev), v.to(dev), gy.to(dev)) if cplx else (lam.real.contiguous().to(dev), v.real.contiguous().to(dev), gy.real.contiguous().to(dev))


def _pass(lam, v, gy):
    lam, v = lam.detach().requires_grad_(), v.detach().requires_grad_()
    y = scan.diagonal_recurrence(lam, v)
    return [y, *torch.autograd.grad(y, (lam, v), gy)]


class _Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


def test_direct_equals_dispatched_and_modes_see_the_ops(gpu):
    direct = _pass(*_inputs(gpu))
    with _Names() as mode:
        dispatched = _pass(*_inputs(gpu))
    assert any("scan_diagonal_shared." in n for n in mode.names) and any("shared_bwd" in n for n in mode.names)
    for a, b in zip(direct, dispatched):
        assert torch.equal(a, b)


def test_lazy_conjugates_are_resolved(gpu):
    lam, v, gy = _inputs(gpu)
    want = _pass(lam.conj().resolve_conj(), v.conj().resolve_conj(), gy.conj().resolve_conj())
    assert gy.conj().is_conj()
    for a, b in zip(_pass(lam.conj(), v.conj(), gy.conj()), want):
        assert torch.equal(a, b)
    lr, vr, gr = _inputs(gpu, cplx=False)
    neg = torch.complex(torch.zeros_like(vr), vr).conj().imag  # a lazily negated view of -v
    assert neg.is_neg()
    for a, b in zip(_pass(lr, neg, gr), _pass(lr, -vr, gr)):
        assert torch.equal(a, b)


def test_no_second_derivative_inference_and_saved_tensor_hooks(gpu):
    lam, v, gy = _inputs(gpu, cplx=False)
    lam.requires_grad_()
    y = scan.diagonal_recurrence(lam, v)
    (glam,) = torch.autograd.grad(y, lam, gy, create_graph=True)
    with pytest.raises(RuntimeError, match="no autograd|autograd formula"):
        glam.sum().backward()
    with torch.inference_mode():
        assert torch.equal(scan.diagonal_recurrence(lam.detach(), v), y)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        y = scan.diagonal_recurrence(lam, v)
    assert y.shape in packed
    y.backward(gy)
    y = scan.diagonal_recurrence(lam, v)
    y.add_(1.0)  # the backward's saved states changed in place
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


def test_transforms_take_the_registered_op(gpu, monkeypatch):
    lam, v, _ = _inputs(gpu, cplx=False)
    seen = []
    plain = ops._plain
    monkeypatch.setattr(ops, "_plain", lambda t: seen.append(1) or plain(t))
    try:
        torch.func.vmap(lambda a: scan.diagonal_recurrence(lam, a))(v)
    except RuntimeError:
        pass  # no batching rule: the registered op says so
    assert not seen
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        scan.diagonal_recurrence(lam, v)
    assert any(e.key.startswith("tsfast_hip::scan_diagonal") for e in prof.key_averages())


def test_a_first_call_in_inference_mode_leaves_later_calls_direct(gpu, monkeypatch):
    lam, v, gy = _inputs(gpu)
    monkeypatch.setattr(ops, "_plain_keys", set())
    with torch.inference_mode():
        scan.diagonal_recurrence(lam, v)
    dispatched = []
    monkeypatch.setattr(scan._scan_shared_op, "_op", lambda *a: dispatched.append(a))
    _pass(lam, v, gy)
    with torch.inference_mode():
        scan.diagonal_recurrence(lam, v.clone())
    assert not dispatched
