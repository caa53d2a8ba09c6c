"""Eager calls that go straight to an op's body or a Function's forward (``eager.plain``): the
same bits as the general route, and the general route wherever something records, traces,
transforms or profiles the call."""
import pytest
import torch
import torch.autograd.forward_ad as fwd_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from conftest import dpa_mod

pytestmark = pytest.mark.gpu

E = dpa_mod("eager")
K = dpa_mod("fp8_kernels")
GN = dpa_mod("gn_silu")
R = dpa_mod("residual")
OPS = dpa_mod("ops")
CL = torch.channels_last


def _x(shape=(2, 128, 8, 8), dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(3)
    return torch.randn(shape, generator=g).to(dtype).cuda().contiguous(memory_format=CL)


class _Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Function(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Sub(torch.Tensor):
    pass


def test_plain_calls_only():
    x = _x()
    assert E.plain(x, torch.nn.Parameter(x.float(), requires_grad=False), 1, None, 2.0)
    leaf = x.float().requires_grad_()
    assert not E.plain(leaf)
    with torch.no_grad():
        assert E.plain(leaf)
    with torch.inference_mode():
        assert E.plain(x, x + 1)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert E.plain(x)
    assert not E.plain(x.cpu()) and not E.plain(x.as_subclass(_Sub))
    assert not E.plain(torch._neg_view(x)) and not E.plain(x.to_sparse())
    for mode in (_Dispatch(), _Function(), torch.profiler.profile()):
        with mode:
            assert not E.plain(x), type(mode)
    seen = []

    def probe(t):
        seen.append(E.plain(t))
        return t * 2
    torch.func.vmap(probe)(x)
    torch.func.grad(lambda t: probe(t).sum())(x.float())
    torch.func.functionalize(probe)(x)
    torch.jit.trace(probe, x, check_trace=False)
    assert not any(seen) and len(seen) == 4


def test_forwards_alone_equal_apply():
    """Both routes of each kind of call: outputs, their views and their refusals."""
    x, w = _x(), _x((128, 128, 3, 3)) * 0.05
    gamma, beta = torch.ones(128, device="cuda"), torch.zeros(128, device="cuda")
    for op, args in ((OPS.quantize, (x,)), (OPS.quantize_with_weight, (x, w.float(), False))):
        for a, b in zip(E.run(op, *args), op(*args)):
            assert a.dtype == b.dtype and a.stride() == b.stride()
            assert torch.equal(a.view(torch.uint8) if a.element_size() == 1 else a,
                               b.view(torch.uint8) if b.element_size() == 1 else b)
    calls = ((K.Conv2dFP8General, (x, w, 1, 1)), (K.Conv2dFP8Specialized, (_x((2, 256, 8, 8)),
             _x((256, 256, 3, 3)), None, None, False)),
             (K.LinearFP8Function, (x.permute(0, 2, 3, 1).reshape(-1, 128), w[:, :, 0, 0], None)),
             (GN.GroupNormSiLU, (x, gamma, beta, 32, 1e-5)),
             (GN.GroupNormSiLUTee, (x, gamma, beta, 32, 1e-5, True, None)),
             (R.ResidualScale, (x, x)), (R.Downsample2Tee, (x,)))
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        for fn, args in calls:
            a, b = E.apply(fn, *args), fn.apply(*args)
            for u, v in zip(*((a, b) if isinstance(a, tuple) else ((a,), (b,)))):
                assert torch.equal(u, v) and u.stride() == v.stride(), fn
                assert (u._base is None) == (v._base is None) and u is not args[0], fn
        with fwd_ad.dual_level():
            dual = fwd_ad.make_dual(x, torch.ones_like(x))
            with pytest.raises(Exception):
                R.ResidualScale.apply(dual, dual)
            with pytest.raises(Exception):
                R.residual_join(dual, dual)
    with pytest.raises(NotImplementedError):
        E.run(OPS.quantize, x.cpu())
    y = K.conv2d_fp8(x.detach().requires_grad_(), w, 1, 1)
    assert y.requires_grad and type(y.grad_fn).__name__ == "Conv2dFP8GeneralBackward"


def test_launches_follow_the_current_stream():
    """Work on a side stream is ordered with that stream's own; a CPU tensor is refused."""
    lib, s = dpa_mod("_lib"), torch.cuda.Stream()
    x = _x()
    assert lib.current_stream(x) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(s):
        assert lib.current_stream(x) == s.cuda_stream
    with pytest.raises(ValueError):
        lib.current_stream(x.cpu())
