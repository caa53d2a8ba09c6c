"""What the FP8 layers and the ops under them refuse before they launch anything: operands on
different GPUs. Fake tensors have a device and a shape but no memory, so no GPU is needed."""
from __future__ import annotations

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from conftest import dpa_mod

K = dpa_mod("fp8_kernels")
CL = torch.channels_last


@pytest.fixture
def no_launch(monkeypatch):
    """A call into the library is a failure, whatever it would have said."""
    def refuse(name, *args):
        pytest.fail(f"{name} was called")
    monkeypatch.setattr(K._lib, "call", refuse)


def _bf16(*shape, device="cuda:0"):
    t = torch.empty(shape, device=device, dtype=torch.bfloat16)
    return t.contiguous(memory_format=CL) if len(shape) == 4 else t


@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("call", [
    lambda x, w: K.conv2d_fp8(x, w, 1, 1),
    lambda x, w: K.conv2d_fp8(x, w, 2, 1),
    lambda x, w: K.triton_conv2d_fp8(x, w),
    lambda x, w: K.linear_fp8_autograd(x[:, :, 0, 0], w[:, :, 0, 0]),
    lambda x, w: K._quantize_with_weight_impl(x, w, False),
    lambda x, w: K._quantize_with_weight_impl(x, w, True),
], ids=["conv", "conv_s2", "registry_conv", "linear", "op", "op_frag"])
def test_a_weight_on_another_gpu_is_refused(no_launch, call, wdtype):
    with FakeTensorMode():
        x, w = _bf16(2, 128, 32, 32), _bf16(128, 128, 3, 3, device="cuda:1").to(wdtype)
        with pytest.raises(AssertionError):
            call(x, w)
        with pytest.raises(AssertionError):
            call(x.to("cuda:1"), w.to("cuda:0"))
        with pytest.raises(AssertionError):
            call(x, w.cpu())
