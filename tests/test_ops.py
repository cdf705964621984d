"""Ops called without the dispatcher (tsfast_amd/ops.py), on the CPU: which calls may go directly."""

import pytest
import torch

from tsfast_amd import ops


def _keys(t):
    return torch._C._dispatch_keys(t).raw_repr()


def test_plain_keys_do_not_depend_on_the_mode_of_the_first_call():
    ordinary = torch.zeros(2)
    with torch.inference_mode():
        inference = torch.zeros(2)
        first_in_inference = ops._keys_of_plain(torch.device("cpu"))
    assert _keys(ordinary) != _keys(inference)
    assert first_in_inference == ops._keys_of_plain(torch.device("cpu")) == {_keys(ordinary), _keys(inference)}


@pytest.fixture(scope="module")
def scaled():
    """An op of the package's kind, ``x * 2 (+ y)``."""

    @ops.custom_op("tsfast_hip_test::scaled")
    def scaled(x: torch.Tensor, y: torch.Tensor | None) -> torch.Tensor:
        return x * 2 if y is None else x * 2 + y

    scaled.register_fake(lambda x, y: torch.empty_like(x))
    return scaled


@pytest.fixture
def direct(monkeypatch):
    """CPU tensors stand in for GPU tensors: plain ones are called directly."""
    monkeypatch.setattr(ops, "_plain_keys", ops._keys_of_plain(torch.device("cpu")))


def test_tensor_likes_and_keywords_reach_the_registered_op(scaled, direct):
    x = torch.arange(3.0)

    class Recorder:
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            return func

    assert torch.equal(scaled(x, None), 2 * x)
    assert scaled(x, Recorder()) is torch.ops.tsfast_hip_test.scaled.default
    assert torch.equal(scaled(x, y=x), 3 * x)
    with pytest.raises(RuntimeError):
        scaled(x, "y")


def test_ops_offer_what_a_custom_op_offers(scaled, direct):
    scaled.register_vmap(lambda info, in_dims, x, y: (scaled(x, y), in_dims[0]))
    x = torch.randn(4, 3)
    assert torch.equal(torch.func.vmap(lambda t: scaled(t, None))(x), 2 * x)
    with pytest.raises(AttributeError):
        scaled.no_such_attribute


@pytest.mark.parametrize("how", ["kernel", "library", "autocast", "autograd"])
def test_registrations_from_elsewhere_are_not_passed_by(direct, monkeypatch, how):
    name = f"tsfast_hip_test::replaced_by_{how}"

    @ops.custom_op(name)
    def op(x: torch.Tensor) -> torch.Tensor:
        return x * 2

    op.register_autograd(lambda ctx, g: 2 * g, setup_context=lambda ctx, inputs, output: None)
    dispatched = []
    registered = op._op
    monkeypatch.setattr(op, "_op", lambda *a: dispatched.append(1) or registered(*a))
    x = torch.randn(3, requires_grad=True)
    op(x).sum().backward()
    assert not dispatched and torch.equal(x.grad, torch.full((3,), 2.0))
    if how == "kernel":
        torch.library.register_kernel(name, "cuda", lambda x: x * 3)
    elif how == "library":
        library = torch.library.Library("tsfast_hip_test", "IMPL")
        library.impl(name.split("::")[1], lambda x: x * 3, "CUDA")
    elif how == "autocast":
        torch.library.register_autocast(name, "cuda", torch.float32)
    else:
        torch.library.register_autograd(name, lambda ctx, g: 5 * g)
    x.grad = None
    op(x).sum().backward()
    assert dispatched
    assert torch.equal(x.grad, torch.full((3,), 5.0 if how == "autograd" else 2.0))
