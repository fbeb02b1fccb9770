"""The question whether a kernel may stand in for torch operators reads states that
torch keeps under private names: a torch without one of them gets the operators,
not an error. (No GPU work: no tensors are asked about.)"""

import sys

import pytest
import torch

from late_interaction_kernels import _lib


def test_plain_without_anything_active():
    assert _lib.plain_op()


@pytest.mark.parametrize("owner,name", [("torch.autograd.forward_ad", "_current_level"),
                                        ("torch._C._functorch", "maybe_current_level"),
                                        ("torch._C", "_len_torch_dispatch_stack"),
                                        ("torch._C", "_len_torch_function_stack"),
                                        ("torch.jit", "is_tracing"), ("torch.compiler", "is_compiling")])
def test_a_missing_probe_means_operators(monkeypatch, owner, name):
    mod = torch
    for part in owner.split(".")[1:]:
        mod = getattr(mod, part)
    monkeypatch.delattr(mod, name)
    assert _lib.plain_op() is False


@pytest.mark.parametrize("name", ["_cuda_getCurrentRawStream", "_cuda_getDevice"])
def test_package_imports_without_the_private_handles(monkeypatch, name):
    import importlib.util

    monkeypatch.delattr(torch._C, name, raising=False)
    spec = importlib.util.spec_from_file_location("_lib_copy", _lib.__file__)
    mod = importlib.util.module_from_spec(spec)
    monkeypatch.setitem(sys.modules, "_lib_copy", mod)
    spec.loader.exec_module(mod)
    assert callable(mod._raw_stream) and callable(mod._current_device)
    if name == "_cuda_getDevice":
        assert mod._current_device is torch.cuda.current_device


def test_function_mode_means_operators():
    from torch.overrides import TorchFunctionMode

    class Mode(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not _lib.plain_op()
    with torch.autograd.forward_ad.dual_level():
        assert not _lib.plain_op()
