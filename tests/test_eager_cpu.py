"""The direct route of eager calls (``eager.plain``) reads torch's state through names that torch
may move: where one is missing, every call takes the general route instead of raising."""
from __future__ import annotations

import importlib.util
import os

import pytest
import torch

from conftest import PKG_NAME, ROOT, dpa_mod

dpa_mod("eager")        # (the package, for the copies' relative imports)


def _copy(name):
    """A fresh import of a module of the package, beside the one in use."""
    path = os.path.join(ROOT, PKG_NAME, name + ".py")
    spec = importlib.util.spec_from_file_location(f"{PKG_NAME}.{name}_copy", path)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


class _Double(torch.autograd.Function):
    direct = None

    @staticmethod
    def forward(ctx, x):
        _Double.direct = type(ctx).__name__ == "NoGraph"
        return x * 2


@pytest.mark.parametrize("owner,name", [
    (torch._C, "_dispatch_keys"), (torch._C, "_dispatch_tls_local_include_set"),
    (torch._C, "_len_torch_function_stack"), (torch._C, "DispatchKeySet"),
    (torch.autograd, "_profiler_enabled"), (torch.autograd.forward_ad, "_current_level"),
], ids=lambda v: v if isinstance(v, str) else v.__name__)
def test_a_missing_name_of_torch_means_the_general_route(monkeypatch, owner, name):
    with torch.no_grad():
        eager = _copy("eager")
        assert eager.plain(1, None)         # nothing is active, no tensor to look at
        monkeypatch.delattr(owner, name)
        eager = _copy("eager")
        monkeypatch.undo()
        assert not eager.plain(1, None)
        x = torch.ones(3)
        assert torch.equal(eager.apply(_Double, x), x * 2) and _Double.direct is False


def test_a_missing_stream_handle_means_the_stream_object(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    lib = _copy("_lib")
    monkeypatch.undo()

    class _Stream:
        cuda_stream = 77

    class _Gpu:
        is_cuda, device = True, "cuda:0"
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: _Stream())
    assert lib.current_stream(_Gpu()) == 77
