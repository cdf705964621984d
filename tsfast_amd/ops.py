"""Custom ops that cost a plain eager call no dispatcher round trip.

``custom_op`` registers an op as ``torch.library.custom_op`` does. A call that nothing but the
kernels would see (dense GPU tensors, or None; no trace, transform, mode, forward-mode level or
profiler) runs the op's function directly, under an ``autograd.Function`` with the op's own rules
when a gradient is wanted. Every other call goes through the registered op, also under
``torch.set_default_device``, which is a mode, and where a program has registered a kernel, cast or
autograd rule of its own on the op (from Python). The dispatcher's Python layers bound small passes: a
truncated-BPTT chunk (8 x 4096 x 128, forward and backward) took 263 us through them and takes 192
us without, a Mamba window (64 x 512 x 128) 239 and 201 us, a forward call without gradients 49 and
44 us.
"""

from __future__ import annotations

__all__ = ["custom_op"]

import torch
from torch.autograd import forward_ad

# bound once: every call asks all of these (the lookups were 0.5 us of a call of four tensors)
_dispatch_keys = torch._C._dispatch_keys
_len_dispatch_modes = torch._C._len_torch_dispatch_stack
_function_mode = torch._C._is_torch_function_mode_enabled
_transform = torch._C._functorch.peek_interpreter_stack
_tracing_state = torch._C._get_tracing_state
_profiler = torch._C._autograd._profiler_enabled
_registered = torch.library._impls  # what Python code has registered on any op, as "namespace/op/key"
# dispatch keys of a plain dense GPU tensor (made in and outside inference mode); any other key
# (conjugate or negative views, subclasses, functional, sparse, nested, batched ..) needs the dispatcher
_plain_keys: set[int] = set()


def _keys_of_plain(device: torch.device) -> set[int]:
    """The keys of both, whatever mode the caller is in: a first call under inference mode (a model
    validated before it is trained) must not leave ordinary tensors to the dispatcher for good."""
    keys = set()
    for mode in (False, True):
        with torch.inference_mode(mode):
            keys.add(_dispatch_keys(torch.empty(0, device=device)).raw_repr())
    return keys


def _plain(t) -> bool:
    if type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter:
        return False
    if not _plain_keys and t.is_cuda:
        _plain_keys.update(_keys_of_plain(t.device))
    return _dispatch_keys(t).raw_repr() in _plain_keys


def _unobserved() -> bool:
    """No trace, transform, mode or profiler would see an op called now."""
    return (
        _len_dispatch_modes() == 0
        and not _function_mode()
        and _transform() is None
        and _tracing_state() is None
        and forward_ad._current_level < 0
        and not _profiler()
    )


class _Op:
    """A registered custom op and its direct form; see ``custom_op``."""

    def __init__(self, name: str, fn):
        self._fn = fn
        self._def = torch.library.custom_op(name, fn, mutates_args=())
        ns, op = name.split("::")
        self._op = getattr(getattr(torch.ops, ns), op).default
        self._function = self._backward = None
        # what a registration from elsewhere that a GPU call would meet is recorded under
        self._overrides = frozenset(
            f"{ns}/{op}{overload}/{key}" for overload in ("", ".default") for key in ("CUDA", "AutogradCUDA", "AutocastCUDA")
        )
        self.__doc__ = fn.__doc__

    def __getattr__(self, name):
        """Everything else a custom op offers (``register_kernel``, ``register_vmap`` ..)."""
        if name == "_def":  # not set yet
            raise AttributeError(name)
        return getattr(self._def, name)

    def register_autograd(self, backward, *, setup_context):
        self._def.register_autograd(backward, setup_context=setup_context)
        impl = self._fn

        class Direct(torch.autograd.Function):
            @staticmethod
            def forward(ctx, *args):
                out = impl(*args)
                setup_context(ctx, args, out)
                return out

            @staticmethod
            def backward(ctx, *grads):
                return backward(ctx, *grads)

        Direct.__name__ = Direct.__qualname__ = f"Direct_{impl.__name__}"
        self._function, self._backward = Direct, self._def._backward_fn

    def _overridden(self) -> bool:
        return not self._overrides.isdisjoint(_registered) or self._def._backward_fn is not self._backward

    def __call__(self, *args, **kwargs):
        if kwargs or torch.compiler.is_compiling() or not _unobserved() or self._overridden():
            return self._op(*args, **kwargs)
        wants_grad = False
        for t in args:
            if t is None:
                continue
            if not _plain(t):  # also what is no tensor: the dispatcher takes or refuses it (a proxy of a trace ..)
                return self._op(*args)
            wants_grad = wants_grad or t.requires_grad
        if wants_grad and torch.is_grad_enabled():
            # an op without rules (a backward's) says so itself when it is differentiated
            return self._op(*args) if self._function is None else self._function.apply(*args)
        return self._fn(*args)


def custom_op(name: str):
    """Decorator: register ``fn`` as the custom op ``name`` (no argument mutated) and return it in
    the form described above, with ``register_fake`` and ``register_autograd``."""
    return lambda fn: _Op(name, fn)
