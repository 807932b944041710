"""What lets a layer replace the forward of its submodules by its own kernels: only modules that would do exactly that
mathematics, and only on ordinary tensors.  (No device needed.)"""
import pytest
import torch

from fsa_hip import ops


def _linear():
    return torch.nn.Linear(8, 8, bias=False)


def test_plain_linear():
    assert ops.is_plain_linear(_linear())
    assert not ops.is_plain_linear(torch.nn.Linear(8, 8))
    assert not ops.is_plain_linear(type("Scaled", (torch.nn.Linear,), {})(8, 8, bias=False))


def test_patched_forward_is_not_replaced():
    m = _linear()
    plain = m.forward
    m.forward = lambda x: 2 * plain(x)
    assert not ops.is_plain_linear(m)
    del m.forward
    assert ops.is_plain_linear(m)
    s = torch.nn.Sigmoid()
    s.forward = lambda x: x
    assert not ops.is_plain(s, torch.nn.Sigmoid)


def test_patched_class_is_not_replaced(monkeypatch):
    monkeypatch.setattr(torch.nn.Linear, "forward", lambda self, x: x)
    assert not ops.is_plain_linear(_linear())


@pytest.mark.parametrize("register", ["register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook",
                                      "register_full_backward_pre_hook"])
def test_hooks_are_run(register):
    m = _linear()
    handle = getattr(m, register)(lambda *a: None)
    assert not ops.is_plain_linear(m)
    handle.remove()
    assert ops.is_plain_linear(m)


@pytest.mark.parametrize("register", ["register_module_forward_hook", "register_module_forward_pre_hook",
                                      "register_module_full_backward_hook", "register_module_full_backward_pre_hook"])
def test_global_hooks_are_run(register):
    handle = getattr(torch.nn.modules.module, register)(lambda *a: None)
    try:
        assert not ops.is_plain_linear(_linear())
        assert not ops.is_plain(torch.nn.Sigmoid(), torch.nn.Sigmoid)
    finally:
        handle.remove()
    assert ops.is_plain_linear(_linear())


class Wrapped(torch.Tensor):
    """A tensor whose values live elsewhere (as those of quantised or sharded weights do)."""

    @staticmethod
    def __new__(cls, inner):
        return torch.Tensor._make_wrapper_subclass(cls, inner.shape, dtype=inner.dtype, device=inner.device)

    def __init__(self, inner):
        self.inner = inner

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        y = func(*[a.inner if isinstance(a, cls) else a for a in args], **(kwargs or {}))
        return cls(y) if func is torch.ops.aten.detach.default else y


def test_tensor_subclasses_go_through_torch():
    w = _linear()
    w.weight = torch.nn.Parameter(Wrapped(torch.randn(8, 8)), requires_grad=False)
    assert not ops.is_plain_linear(w)
    assert ops.are_plain_tensors(torch.zeros(1), torch.nn.Parameter(torch.zeros(1)))
    assert not ops.are_plain_tensors(torch.zeros(1), w.weight)
