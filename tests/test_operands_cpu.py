"""What the FP8 layers and the ops under them refuse before they launch anything: operands on
different GPUs, and operands whose dtype, scale or shape their kernels do not check. Fake tensors have a device and a shape but no memory, so no GPU is needed."""
from __future__ import annotations

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from conftest import dpa_mod

K = dpa_mod("fp8_kernels")
OPS = dpa_mod("ops")
BODY = dpa_mod("eager")._BODY
CL = torch.channels_last
E4M3 = torch.float8_e4m3fn


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


def _e4m3(*shape, device="cuda:0"):
    return _bf16(*shape, device=device).to(E4M3)


def _scale(device="cuda:0", dtype=torch.float32, n=1):
    return torch.empty((n,) if n > 1 else (), device=device, dtype=dtype)


def _args(op):
    """A call of an op's body that it takes, by argument name."""
    w9 = 9 * 256 * 128
    return {
        "quantize_with_weight": lambda: dict(x=_bf16(2, 128, 8, 8), weight=_bf16(256, 128, 3, 3).float(),
                                             frag=True),
        "conv_fwd_prepared": lambda: dict(
            x=_e4m3(2, 128, 6, 10), weight=_e4m3(256, 128, 3, 3), x_scale=_scale(),
            weight_scale=_scale(), cout=256, stride=2, padding=1),
        "conv_fwd_frag": lambda: dict(
            x=_e4m3(2, 128, 8, 8), weight=torch.empty(w9, device="cuda:0", dtype=torch.uint8),
            x_scale=_scale(), weight_scale=_scale(), cout=256, stride=1, padding=1),
        "conv_dgrad_prepared": lambda: dict(
            dy=_e4m3(2, 256, 3, 5), weight_t=torch.empty((128, 3, 3, 256), device="cuda:0", dtype=E4M3),
            dy_scale=_scale(), weight_scale=_scale(), cin=128, height=6, width=10, k=3, stride=2,
            padding=1),
        "conv_dgrad_frag": lambda: dict(
            dy=_e4m3(2, 256, 8, 8), weight_t=torch.empty(w9, device="cuda:0", dtype=torch.uint8),
            dy_scale=_scale(), weight_scale=_scale(), cin=128, height=8, width=8, k=3, stride=1,
            padding=1),
        "gemm_dgrad_wt": lambda: dict(dy=_e4m3(64, 256), weight_t=_e4m3(128, 256),
                                      dy_scale=_scale(), weight_scale=_scale()),
    }[op]()


def _wrong_scales(*names):
    return [dict([(n, f)]) for n in names for f in (
        lambda: _scale("cuda:1"), lambda: _scale(dtype=torch.float64), lambda: _scale(n=2))]


WRONG = {
    "quantize_with_weight": [
        dict(x=lambda: _bf16(2, 128, 8, 8).float()), dict(x=lambda: _bf16(2, 128, 8, 8).to(torch.float16)),
        dict(weight=lambda: _bf16(256, 128, 3, 3, device="cuda:1")),
        dict(weight=lambda: _bf16(256, 128))],                         # fragments of a linear's
    "conv_fwd_prepared": _wrong_scales("x_scale", "weight_scale") + [
        dict(weight=lambda: _e4m3(256, 128, 3, 3, device="cuda:1")), dict(cout=lambda: 384),
        dict(weight=lambda: _bf16(256, 128, 3, 3)), dict(x=lambda: _bf16(2, 128, 6, 10))],
    "conv_fwd_frag": _wrong_scales("x_scale", "weight_scale") + [
        dict(weight=lambda: torch.empty(9 * 256 * 128, device="cuda:1", dtype=torch.uint8)),
        dict(stride=lambda: 2), dict(padding=lambda: 0), dict(cout=lambda: 384),
        dict(x=lambda: _e4m3(2, 128, 6, 6)), dict(x=lambda: _bf16(2, 128, 8, 8))],
    "conv_dgrad_prepared": _wrong_scales("dy_scale", "weight_scale") + [
        dict(height=lambda: 8), dict(stride=lambda: 1), dict(k=lambda: 1), dict(cin=lambda: 256),
        dict(weight_t=lambda: torch.empty((128, 3, 3, 256), device="cuda:1", dtype=E4M3)),
        dict(weight_t=lambda: torch.empty((128, 3, 3, 128), device="cuda:0", dtype=E4M3))],
    "conv_dgrad_frag": _wrong_scales("dy_scale", "weight_scale") + [
        dict(weight_t=lambda: torch.empty(9 * 256 * 128, device="cuda:1", dtype=torch.uint8)),
        dict(stride=lambda: 2), dict(k=lambda: 1), dict(height=lambda: 16), dict(cin=lambda: 256)],
    "gemm_dgrad_wt": _wrong_scales("dy_scale", "weight_scale") + [
        dict(dy=lambda: _bf16(64, 256)), dict(weight_t=lambda: _bf16(128, 256)),
        dict(weight_t=lambda: _e4m3(128, 384)), dict(weight_t=lambda: _e4m3(128, 128)),
        dict(weight_t=lambda: _e4m3(128, 256, device="cuda:1"))],
}


@pytest.mark.parametrize("op,i", [(op, i) for op, w in WRONG.items() for i in range(len(w))], ids=str)
def test_bodies_of_ops_refuse_operands_that_their_kernels_would_misread(no_launch, op, i):
    body = BODY[getattr(OPS, op.replace("_frag", "_prepared"))]
    with FakeTensorMode():
        args = _args(op)
        args.update({k: f() for k, f in WRONG[op][i].items()})
        with pytest.raises(AssertionError):
            body(**args)


def test_a_strided_gradient_of_the_linear_is_made_dense(monkeypatch):
    """gemm_dgrad_wt reads dense rows: a strided dy or weight reaches the library as a copy."""
    seen = []
    monkeypatch.setattr(K, "_stream", lambda t: 0)
    monkeypatch.setattr(K._lib, "call", lambda name, *a: seen.append(a[:2]))
    wide, tall = torch.empty(64, 512, dtype=E4M3), torch.empty(256, 128, dtype=E4M3)
    one = torch.ones(())

    class _Cuda(torch.Tensor):
        is_cuda = True
    dy, wt = wide[:, :256].as_subclass(_Cuda), tall.t().as_subclass(_Cuda)
    K._linear_dgrad_wt(dy, wt, one, one)
    assert len(seen) == 1 and seen[0][0] != wide.data_ptr() and seen[0][1] != tall.data_ptr()


@pytest.mark.parametrize("frag", [True, False])
def test_forwards_that_record_nothing_leave_the_data_gradient_copy_out(monkeypatch, frag):
    """A forward called by ``eager.apply`` has no backward: the weight's second copy is neither
    allocated nor written, while a recorded forward asks for it."""
    class _Asked(Exception):
        pass

    def asked(ctx, op, *args):
        raise _Asked(args[-1])
    monkeypatch.setattr(K, "run_in", asked)
    no_graph, recorded = dpa_mod("eager").NoGraph(), object()
    with FakeTensorMode():
        x, w = _bf16(2, 128, 8, 8), _bf16(128, 128, 3, 3)
        for ctx, want in ((no_graph, False), (recorded, True)):
            with pytest.raises(_Asked, match=str(want)):
                K._conv_current_fwd(ctx, x, w, 1, 1)
        with pytest.raises(_Asked, match="False"):
            K.LinearFP8Function.forward(no_graph, x[:, :, 0, 0], w[:, :, 0, 0])

    calls = []
    monkeypatch.setattr(K, "_stream", lambda t: 0)
    monkeypatch.setattr(K._lib, "call", lambda name, *a: calls.append(a))

    class _Cuda(torch.Tensor):
        is_cuda = True
    x = torch.empty(16, 128, dtype=torch.bfloat16).as_subclass(_Cuda)
    w = torch.empty((128, 128, 3, 3) if frag else (256, 128)).as_subclass(_Cuda)
    for copy in (True, False):
        wt = K._quantize_with_weight_impl(x, w, frag, copy)[3]
        assert (wt.numel() == w.numel()) if copy else (wt.numel() == 0)
        assert (calls[-1][10] is None) == (not copy)
