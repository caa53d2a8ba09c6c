"""GPU parity of the fused GroupNorm(+FiLM)+SiLU forward/backward against the float64 oracle.

The reference runs GroupNorm and SiLU in float32 under autocast (diffusion/unet.py:151,
:157-159) and the FP8 conv then rounds the result to bf16 (diffusion/fp8_kernels.py:835). The
fused kernel emits that bf16 directly. Against the float64 oracle, a float32 evaluation may
land on the other side of a bf16 rounding boundary, so the forward bar is one bf16 ulp, with
almost every element bit-identical. Gradients are float32 reductions: normwise 1e-4 for the
parameter gradients and the conv tolerance (one bf16 ulp + noise) for dx.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from conftest import assert_bf16_close, dpa_mod, dropout_band, nhwc_bits, randn_bf16
from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu

GROUPS = 32


@pytest.fixture(scope="module")
def G():
    return dpa_mod("gn_silu")


def cl(t):
    return t.cuda().contiguous(memory_format=torch.channels_last)


def params(c, n, seed, film):
    g = torch.Generator().manual_seed(seed)
    gamma = 1.0 + 0.1 * torch.randn(c, generator=g)
    beta = 0.1 * torch.randn(c, generator=g)
    fs = fb = None
    if film:
        fs = 1.0 + 0.2 * torch.randn(n, c, generator=g)   # the reference's (w + 1)
        fb = 0.2 * torch.randn(n, c, generator=g)
    return gamma, beta, fs, fb


def assert_fwd_close(got_bits, ref_bits, what):
    g = O.bf16_bits_to_f32(got_bits).astype(np.float64)
    r = O.bf16_bits_to_f32(ref_bits).astype(np.float64)
    assert np.isfinite(g).all(), what
    # one bf16 ulp of the reference (at most 2^-7 |r|) plus float32 noise near zero
    bad = np.abs(g - r) > 2.0**-7 * np.abs(r) + 1e-6
    assert not bad.any(), f"{what}: {int(bad.sum())} elements beyond 1 bf16 ulp"
    exact = float(np.mean(got_bits == ref_bits))
    assert exact > 0.995, f"{what}: only {exact:.4f} bit-identical"


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)


CASES = [
    # (n, c, h, w, film): the reference U-Net's GroupNorm sites at reduced batch
    (2, 128, 32, 32, False),
    (2, 256, 16, 16, True),
    (2, 512, 8, 8, False),
    (3, 256, 4, 4, True),
    (2, 256, 7, 9, True),    # ragged pixel count
    (2, 128, 17, 19, True),  # chunked form with a ragged last chunk (323 = 128 + 128 + 67)
    (1, 128, 5, 3, False),
]


@pytest.mark.parametrize("n,c,h,w,film", CASES, ids=lambda v: str(v))
def test_gn_silu_fwd_bwd_vs_oracle(G, n, c, h, w, film):
    if not G.supported(c, GROUPS):
        pytest.skip(f"C={c}, G={GROUPS} outside the fused kernel's shapes")
    seed = n * 1000 + c + h
    x = randn_bf16((n, c, h, w), seed=seed, std=2.0)
    x = (x.float() + 0.5).to(torch.bfloat16)      # non-zero group means
    dout = randn_bf16((n, c, h, w), seed=seed + 1, std=1e-2)
    gamma, beta, fs, fb = params(c, n, seed + 2, film)
    fs_d = None if fs is None else fs.cuda()[:, :, None, None]
    fb_d = None if fb is None else fb.cuda()[:, :, None, None]

    out, mean, rstd = G.gn_silu_fwd(cl(x), gamma.cuda(), beta.cuda(), GROUPS, 1e-5, fs_d, fb_d)
    dx, dgamma, dbeta, dfs, dfb = G.gn_silu_bwd(
        cl(x), cl(dout), gamma.cuda(), beta.cuda(), mean, rstd, GROUPS, fs_d, fb_d)
    torch.cuda.synchronize()

    xb = nhwc_bits(x)
    npf = None if fs is None else fs.numpy()
    npb = None if fb is None else fb.numpy()
    ref = O.gn_silu_fwd(xb, gamma.numpy(), beta.numpy(), GROUPS, 1e-5, npf, npb)
    assert out.is_contiguous(memory_format=torch.channels_last) and out.dtype == torch.bfloat16
    assert_fwd_close(nhwc_bits(out.cpu()), ref, f"fwd {(n, c, h, w, film)}")

    # group statistics
    xg = O.bf16_bits_to_f32(xb).astype(np.float64).reshape(n, h * w, GROUPS, c // GROUPS)
    m_ref = xg.mean(axis=(1, 3))
    v_ref = xg.var(axis=(1, 3))
    assert rel(mean.cpu().numpy().reshape(n, GROUPS), m_ref) < 1e-5
    assert rel(rstd.cpu().numpy().reshape(n, GROUPS), 1 / np.sqrt(v_ref + 1e-5)) < 1e-5

    rdx, rdg, rdb, rdfs, rdfb = O.gn_silu_bwd(xb, nhwc_bits(dout), gamma.numpy(), beta.numpy(),
                                             GROUPS, 1e-5, npf, npb)
    assert_bf16_close(nhwc_bits(dx.cpu()), O.f32_to_bf16_bits(rdx.astype(np.float32)),
                      f"dx {(n, c, h, w, film)}")
    assert rel(dgamma.cpu().numpy(), rdg) < 1e-4
    assert rel(dbeta.cpu().numpy(), rdb) < 1e-4
    if film:
        assert rel(dfs.cpu().numpy(), rdfs) < 1e-4
        assert rel(dfb.cpu().numpy(), rdfb) < 1e-4
    else:
        assert dfs is None and dfb is None


def test_gn_silu_cfg4_full_size_vs_torch_fp32(G):
    """cfg4's norm2 site at full size ([128,256,16,16] with FiLM) through the autograd
    Function, against torch float32 GroupNorm+SiLU on the GPU."""
    n, c, h, w = 128, 256, 16, 16
    x = cl(randn_bf16((n, c, h, w), seed=0))
    gamma, beta, fs, fb = params(c, n, 3, True)
    gamma, beta = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    fs = fs.cuda()[:, :, None, None].requires_grad_()
    fb = fb.cuda()[:, :, None, None].requires_grad_()
    dout = cl(randn_bf16((n, c, h, w), seed=1, std=1e-2))

    xa = x.clone().requires_grad_()
    out = G.group_norm_silu(xa, gamma, beta, GROUPS, 1e-5, fs, fb)
    out.backward(dout)

    xr = x.float().clone().requires_grad_()
    gr, br = gamma.detach().clone().requires_grad_(), beta.detach().clone().requires_grad_()
    fsr, fbr = fs.detach().clone().requires_grad_(), fb.detach().clone().requires_grad_()
    ref = F.silu(fsr * F.group_norm(xr, GROUPS, gr, br, 1e-5) + fbr)
    ref.backward(dout.float())
    torch.cuda.synchronize()

    def nerr(a, b):
        a, b = a.detach().float(), b.detach().float()
        return float((a - b).norm() / b.norm())

    assert out.dtype == torch.bfloat16
    assert nerr(out, ref) < 2**-8
    assert nerr(xa.grad, xr.grad) < 1e-2
    assert xa.grad.dtype == torch.bfloat16
    for got, want in ((gamma.grad, gr.grad), (beta.grad, br.grad), (fs.grad, fsr.grad),
                      (fb.grad, fbr.grad)):
        assert got.shape == want.shape
        assert nerr(got, want) < 1e-3


@pytest.mark.parametrize("n,c,h,w", [(3, 256, 16, 16), (2, 128, 32, 32), (2, 512, 8, 8)])
def test_gn_silu_film_from_time_projection_matches_split_form(G, n, c, h, w):
    """GroupNormSiLUFilm (the kernel reads wb = [w | b] in bf16 and forms bf16(w + 1)) equals
    GroupNormSiLU on the reference's w + 1 and b (diffusion/unet.py:157-159) bit for bit:
    output, dx, dgamma, dbeta, and d(wb) = [d(w + 1) | d(b)] in bf16."""
    g = torch.Generator().manual_seed(n + c)
    x = (torch.randn((n, c, h, w), generator=g) * 2 + 0.5).to(torch.bfloat16)
    gamma, beta, _, _ = params(c, n, c + 1, False)
    wb = (0.3 * torch.randn((n, 2 * c, 1, 1), generator=g)).to(torch.bfloat16).cuda()
    dout = randn_bf16((n, c, h, w), seed=c + 7)

    xa = cl(x).requires_grad_()
    ga, ba = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    wba = wb.clone().requires_grad_()
    ya = G.group_norm_silu_film(xa, ga, ba, GROUPS, 1e-5, wba)
    ya.backward(cl(dout))

    xb = cl(x).requires_grad_()
    gb, bb = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    wbb = wb.clone().requires_grad_()
    wpart, bpart = torch.chunk(wbb, 2, dim=1)
    yb = G.group_norm_silu(xb, gb, bb, GROUPS, 1e-5, wpart + 1, bpart)
    yb.backward(cl(dout))
    torch.cuda.synchronize()
    for got, ref, what in ((ya, yb, "out"), (xa.grad, xb.grad, "dx"), (ga.grad, gb.grad, "dgamma"),
                           (ba.grad, bb.grad, "dbeta"), (wba.grad, wbb.grad, "dwb")):
        assert got.dtype == ref.dtype and got.shape == ref.shape, what
        assert torch.equal(got.detach(), ref.detach()), what


@pytest.mark.parametrize("n,c,h,w,film", [(2, 128, 40, 40, True), (1, 256, 36, 36, False)])
def test_one_launch_and_chunked_forms_agree(G, n, c, h, w, film):
    """Images above 1024 pixels (beyond the resident form) run the chunked kernels when given
    the full workspace; the one-launch kernels (no forward workspace, a backward workspace of
    only the per-image partials) compute the same quantities with another summation order."""
    L = dpa_mod("_lib")
    x = cl(randn_bf16((n, c, h, w), seed=n + c, std=2.0))
    dout = cl(randn_bf16((n, c, h, w), seed=n + c + 1, std=1e-2))
    gamma, beta, fs, fb = params(c, n, c, film)
    gamma, beta = gamma.cuda(), beta.cuda()
    fs = None if fs is None else fs.cuda().contiguous()
    fb = None if fb is None else fb.cuda().contiguous()
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    s = torch.cuda.current_stream().cuda_stream
    hw = h * w
    assert L.query("dpa_gn_silu_fwd_workspace_bytes", n, hw, c, GROUPS) > 0
    res = {}
    for form in ("chunked", "one"):
        out = torch.empty_like(x)
        mean = torch.empty(n * GROUPS, device="cuda")
        rstd = torch.empty(n * GROUPS, device="cuda")
        if form == "chunked":
            wsb = L.query("dpa_gn_silu_fwd_workspace_bytes", n, hw, c, GROUPS)
            ws = torch.empty(wsb, device="cuda", dtype=torch.uint8)
            L.call("dpa_gn_silu_fwd_ws_bf16", x.data_ptr(), gamma.data_ptr(), beta.data_ptr(),
                   p(fs), p(fb), None, out.data_ptr(), mean.data_ptr(), rstd.data_ptr(),
                   ws.data_ptr(), wsb, n, hw, c, GROUPS, 1e-5, s)
            bws = L.query("dpa_gn_silu_bwd_workspace_bytes", n, hw, c, GROUPS)
        else:
            L.call("dpa_gn_silu_fwd_bf16", x.data_ptr(), gamma.data_ptr(), beta.data_ptr(),
                   p(fs), p(fb), out.data_ptr(), mean.data_ptr(), rstd.data_ptr(), n, hw, c,
                   GROUPS, 1e-5, s)
            bws = 2 * n * c * 4
        dx = torch.empty_like(x)
        dg = torch.empty(c, device="cuda")
        db = torch.empty(c, device="cuda")
        dfs = torch.empty((n, c), device="cuda") if film else None
        dfb = torch.empty((n, c), device="cuda") if film else None
        ws = torch.empty(bws, device="cuda", dtype=torch.uint8)
        L.call("dpa_gn_silu_bwd_bf16", x.data_ptr(), dout.data_ptr(), gamma.data_ptr(),
               beta.data_ptr(), p(fs), p(fb), mean.data_ptr(), rstd.data_ptr(), dx.data_ptr(),
               dg.data_ptr(), db.data_ptr(), p(dfs), p(dfb), ws.data_ptr(), bws, n, hw, c,
               GROUPS, s)
        torch.cuda.synchronize()
        res[form] = [t.cpu() for t in (out, mean, rstd, dx, dg, db)] + (
            [dfs.cpu(), dfb.cpu()] if film else [])
    a, b = res["chunked"], res["one"]
    assert_fwd_close(nhwc_bits(a[0]), nhwc_bits(b[0]), "out")
    assert rel(a[1].numpy(), b[1].numpy()) < 1e-5 and rel(a[2].numpy(), b[2].numpy()) < 1e-5
    assert_bf16_close(nhwc_bits(a[3]), nhwc_bits(b[3]), "dx")
    for k in range(4, len(a)):
        assert rel(a[k].numpy(), b[k].numpy()) < 1e-4, k


F32_CASES = [
    # fp32 inputs (the fp32 residual stream / decoder concatenations): resident, chunked and
    # small forms; 1024 pixels without FiLM (the decoder's first GroupNorm) is resident
    (2, 128, 32, 32, False),
    (2, 512, 32, 32, False),
    (2, 128, 32, 32, True),  # 1024 pixels with FiLM: chunked
    (2, 256, 16, 16, True),
    (2, 512, 8, 8, False),
    (3, 256, 4, 4, True),
    (2, 128, 17, 19, True),  # chunked, ragged last chunk
]


@pytest.mark.parametrize("n,c,h,w,film", F32_CASES, ids=lambda v: str(v))
def test_gn_silu_fp32_input_vs_oracle(G, n, c, h, w, film):
    """An fp32 x is normalised as it is (autocast's float32 GroupNorm, diffusion/unet.py:151,
    :157) and dx comes back in fp32: forward within one bf16 ulp of the float64 oracle on the
    fp32 values, dx normwise 2e-5 of the oracle's float64 gradient."""
    seed = n * 1000 + c + h + 7
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((n, c, h, w), generator=g) * 2.0 + 0.5     # fp32, not bf16-representable
    dout = randn_bf16((n, c, h, w), seed=seed + 1, std=1e-2)
    gamma, beta, fs, fb = params(c, n, seed + 2, film)
    fs_d = None if fs is None else fs.cuda()[:, :, None, None]
    fb_d = None if fb is None else fb.cuda()[:, :, None, None]
    xd = cl(x)
    assert G.f32_input_ok(xd)
    out, mean, rstd = G.gn_silu_fwd(xd, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, fs_d, fb_d)
    dx, dgamma, dbeta, dfs, dfb = G.gn_silu_bwd(
        xd, cl(dout), gamma.cuda(), beta.cuda(), mean, rstd, GROUPS, fs_d, fb_d)
    torch.cuda.synchronize()
    assert out.dtype == torch.bfloat16 and dx.dtype == torch.float32
    x_nhwc = x.permute(0, 2, 3, 1).contiguous().numpy()
    npf = None if fs is None else fs.numpy()
    npb = None if fb is None else fb.numpy()
    ref = O.gn_silu_fwd(x_nhwc, gamma.numpy(), beta.numpy(), GROUPS, 1e-5, npf, npb)
    assert_fwd_close(nhwc_bits(out.cpu()), ref, f"fp32 fwd {(n, c, h, w, film)}")
    # the bf16-rounded input would miss: normalising bf16(x) differs from the oracle here
    ref_b = O.gn_silu_fwd(nhwc_bits(x.to(torch.bfloat16)), gamma.numpy(), beta.numpy(), GROUPS,
                          1e-5, npf, npb)
    assert np.mean(ref_b != ref) > 0.05
    rdx, rdg, rdb, rdfs, rdfb = O.gn_silu_bwd(x_nhwc, nhwc_bits(dout), gamma.numpy(),
                                             beta.numpy(), GROUPS, 1e-5, npf, npb)
    got = dx.permute(0, 2, 3, 1).contiguous().cpu().numpy()
    assert rel(got, rdx) < 2e-5, rel(got, rdx)
    assert rel(dgamma.cpu().numpy(), rdg) < 1e-4
    assert rel(dbeta.cpu().numpy(), rdb) < 1e-4
    if film:
        assert rel(dfs.cpu().numpy(), rdfs) < 1e-4
        assert rel(dfb.cpu().numpy(), rdfb) < 1e-4


def test_gn_silu_fp32_autograd_and_fallback(G):
    """Through the autograd Functions: an fp32 input keeps an fp32 gradient, equal to the
    direct calls; a size outside the fp32 forms (96 x 96 = 9216 pixels) is cast to bf16 first,
    as before; the time-projection FiLM form takes fp32 x too."""
    n, c, groups = 2, 256, GROUPS
    g = torch.Generator().manual_seed(11)
    gamma, beta = (1.0 + 0.1 * torch.randn(c, generator=g)).cuda(), (0.1 * torch.randn(c, generator=g)).cuda()
    for h in (16, 96):
        x = cl(torch.randn((n, c, h, h), generator=g) * 1.5)
        xr = x.clone().requires_grad_(True)
        y = G.group_norm_silu(xr, gamma, beta, groups, 1e-5)
        dout = cl(torch.randn((n, c, h, h), generator=g) * 1e-2).to(torch.bfloat16)
        y.backward(dout)
        assert xr.grad.dtype == torch.float32
        if h == 16:
            assert G.f32_input_ok(x)
            out, mean, rstd = G.gn_silu_fwd(x, gamma, beta, groups, 1e-5)
            dx = G.gn_silu_bwd(x, dout, gamma, beta, mean, rstd, groups)[0]
        else:
            assert not G.f32_input_ok(x)
            xb = x.to(torch.bfloat16)
            out, mean, rstd = G.gn_silu_fwd(xb, gamma, beta, groups, 1e-5)
            dx = G.gn_silu_bwd(xb, dout, gamma, beta, mean, rstd, groups)[0].float()
        torch.cuda.synchronize()
        assert torch.equal(y, out), h
        assert torch.equal(xr.grad, dx), h
    # FiLM read from the bf16 time projection, fp32 x: equals the split form on the same x
    h = 16
    x = cl(torch.randn((n, c, h, h), generator=g))
    wb = (torch.randn((n, 2 * c, 1, 1), generator=g) * 0.2).cuda().to(torch.bfloat16)
    xr = x.clone().requires_grad_(True)
    y = G.group_norm_silu_film(xr, gamma, beta, groups, 1e-5, wb)
    w, b = torch.chunk(wb, 2, dim=1)
    x2 = x.clone().requires_grad_(True)
    y2 = G.group_norm_silu(x2, gamma, beta, groups, 1e-5, (w + 1).float(), b.float())
    dout = cl(torch.randn((n, c, h, h), generator=g) * 1e-2).to(torch.bfloat16)
    y.backward(dout)
    y2.backward(dout)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
    assert xr.grad.dtype == torch.float32 and torch.equal(xr.grad, x2.grad)


DROP_CASES = [
    # (n, c, h, w, x fp32): chunked (bf16 and fp32 x) and small-image forms
    (2, 128, 32, 32, True),
    (3, 256, 16, 16, False),
    (2, 512, 8, 8, True),
    (4, 256, 4, 4, False),
]


@pytest.mark.parametrize("n,c,h,w,x32", DROP_CASES, ids=lambda v: str(v))
def test_gn_silu_film_dropout_vs_oracle(G, n, c, h, w, x32):
    """The dropout of diffusion/unet.py:160 fused into GroupNormSiLUFilm: the mask is the
    oracle's splitmix64 mask of the seed the op draws (reproduced from the same torch CUDA
    generator state), kept values are scaled by RN32(1 / RN32(1 - p)) in fp32 before the bf16
    rounding; the backward recomputes the mask. Forward within one bf16 ulp of the float64
    oracle, exact zeros off the mask, keep rate within 5 sigma of 1 - p; gradients against
    the oracle's masked backward."""
    p = 0.2
    seed = n * 977 + c + h
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((n, c, h, w), generator=g) * 2.0 + 0.5
    if not x32:
        x = x.to(torch.bfloat16)
    gamma, beta, _, _ = params(c, n, seed + 2, False)
    wb = (0.3 * torch.randn((n, 2 * c, 1, 1), generator=g)).to(torch.bfloat16)
    dout = randn_bf16((n, c, h, w), seed=seed + 1, std=1e-2)

    torch.cuda.manual_seed(seed)
    drop_seed = int(G.new_dropout_seed("cuda").item())
    torch.cuda.manual_seed(seed)
    xd = cl(x).requires_grad_()
    gd, bd = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    wbd = wb.cuda().requires_grad_()
    y = G.group_norm_silu_film(xd, gd, bd, GROUPS, 1e-5, wbd, p)
    y.backward(cl(dout))
    torch.cuda.synchronize()

    x_nhwc = (x.float() if x32 else x).permute(0, 2, 3, 1).contiguous()
    x_in = x_nhwc.numpy() if x32 else nhwc_bits(x)
    wb32 = wb.float().reshape(n, 2 * c)
    fs = (wb32[:, :c].to(torch.bfloat16).float() + 1).to(torch.bfloat16).float().numpy()
    fb = wb32[:, c:].numpy()
    keep = O.dropout_keep(drop_seed, n * h * w * c, p)
    rate = keep.mean()
    assert abs(rate - (1 - p)) < 5 * np.sqrt(p * (1 - p) / keep.size), rate
    ref = O.gn_silu_fwd(x_in, gamma.numpy(), beta.numpy(), GROUPS, 1e-5, fs, fb, drop=(drop_seed, p))
    got = nhwc_bits(y.detach().cpu())
    assert (got.reshape(-1)[~keep] == 0).all()
    assert_fwd_close(got, ref, f"dropout fwd {(n, c, h, w, x32)}")
    rdx, rdg, rdb, rdfs, rdfb = O.gn_silu_bwd(x_in, nhwc_bits(dout), gamma.numpy(), beta.numpy(),
                                             GROUPS, 1e-5, fs, fb, drop=(drop_seed, p))
    # without the mask the gradient would be far off
    rdx0 = O.gn_silu_bwd(x_in, nhwc_bits(dout), gamma.numpy(), beta.numpy(), GROUPS, 1e-5, fs, fb)[0]
    assert rel(rdx0, rdx) > 0.1
    got_dx = xd.grad.float().permute(0, 2, 3, 1).contiguous().cpu().numpy()
    assert xd.grad.dtype == x.dtype
    assert rel(got_dx, rdx) < (2e-5 if x32 else 4e-3), rel(got_dx, rdx)
    assert rel(gd.grad.cpu().numpy(), rdg) < 1e-4
    assert rel(bd.grad.cpu().numpy(), rdb) < 1e-4
    dwb = wbd.grad.float().reshape(n, 2 * c).cpu().numpy()
    assert rel(dwb[:, :c], rdfs) < 4e-3
    assert rel(dwb[:, c:], rdfb) < 4e-3


@pytest.mark.parametrize("n,c,h,w,x32", [(1, 256, 16, 16, False), (1, 256, 8, 8, True)],
                         ids=lambda v: str(v))
def test_gn_silu_film_dropout_threshold_band(G, n, c, h, w, x32):
    """The keep threshold is floor(fp32(p) * 2^16). With p = 13107 / 2^16 - 2^-40 (fp32 value
    13107 / 2^16) a hash quarter of 13106 = floor(p * 2^16) must be dropped: the seed is built
    (by inverting splitmix64) so that element 0's quarter is that value. The kernel's whole
    mask, forward and backward, equals the oracle's."""
    p, seed, _ = dropout_band()
    g = torch.Generator().manual_seed(9)
    x = torch.randn((n, c, h, w), generator=g) + 0.5
    if not x32:
        x = x.to(torch.bfloat16)
    gamma, beta, _, _ = params(c, n, 10, False)
    wb = (0.3 * torch.randn((n, 2 * c, 1, 1), generator=g)).to(torch.bfloat16)
    G.DROPOUT_SEEDS.seeds = torch.tensor([seed], device="cuda", dtype=torch.int64)
    G.DROPOUT_SEEDS.next = 0
    try:
        xd = cl(x).requires_grad_()
        y = G.group_norm_silu_film(xd, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, wb.cuda(), p)
        assert G.DROPOUT_SEEDS.next == 1  # the op took the planted seed
    finally:
        G.DROPOUT_SEEDS.clear()
    y.backward(torch.ones_like(y))
    torch.cuda.synchronize()
    keep = O.dropout_keep(seed, n * h * w * c, p)
    assert not keep[0] and keep[1]
    got = nhwc_bits(y.detach().cpu()).reshape(-1)
    undropped = G.group_norm_silu_film(cl(x), gamma.cuda(), beta.cuda(), GROUPS, 1e-5,
                                       wb.cuda(), 0.0)
    ub = nhwc_bits(undropped.cpu()).reshape(-1)
    assert ub[0] & 0x7FFF != 0  # element 0 is nonzero before dropout, zero after
    assert got[0] & 0x7FFF == 0
    assert np.array_equal((got & 0x7FFF) == 0, (~keep) | ((ub & 0x7FFF) == 0))
    gx = xd.grad.float().permute(0, 2, 3, 1).contiguous().reshape(-1).cpu().numpy()
    assert np.isfinite(gx).all()


def test_gn_silu_film_dropout_zero_p_and_fresh_masks(G):
    """p = 0 gives the undropped op bit for bit; two calls draw two seeds (different masks);
    a size without a dropout form (96 x 96) is refused rather than silently undropped."""
    n, c, h, w = 2, 256, 16, 16
    g = torch.Generator().manual_seed(5)
    x = cl((torch.randn((n, c, h, w), generator=g) + 0.5).to(torch.bfloat16))
    gamma, beta, _, _ = params(c, n, 6, False)
    wb = (0.3 * torch.randn((n, 2 * c, 1, 1), generator=g)).to(torch.bfloat16).cuda()
    a = G.group_norm_silu_film(x, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, wb, 0.0)
    b = G.group_norm_silu_film(x, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, wb)
    assert torch.equal(a, b)
    d1 = G.group_norm_silu_film(x, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, wb, 0.5)
    d2 = G.group_norm_silu_film(x, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, wb, 0.5)
    z1, z2 = (d1 == 0) & (a != 0), (d2 == 0) & (a != 0)
    assert 0.45 < z1.float().mean().item() < 0.55
    assert not torch.equal(z1, z2)
    x96 = cl(torch.randn((n, c, 96, 96), generator=g).to(torch.bfloat16))
    with pytest.raises(ValueError):  # 9216 pixels: no form with fused dropout
        G.group_norm_silu_film(x96, gamma.cuda(), beta.cuda(), GROUPS, 1e-5, wb, 0.5)


@pytest.mark.parametrize("n,c,h,w,x32", [(2, 128, 32, 32, True), (3, 256, 16, 16, False),
                                         (2, 512, 8, 8, True), (4, 256, 4, 4, False),
                                         (2, 128, 12, 12, True), (1, 128, 96, 96, True)],
                         ids=lambda v: str(v))
def test_gn_silu_tee_accumulates_skip_gradient(G, n, c, h, w, x32):
    """GroupNormSiLUTee returns (silu(GroupNorm(x)), x); its backward adds the second output's
    gradient into dx in the kernel. x's gradient equals autograd's own accumulation over the
    unfused pair (GroupNormSiLU on x and x used again) bit for bit, in fp32 and bf16; 96 x 96
    (no fp32 form: x is cast to bf16) takes the separate add."""
    seed = n + c + h + 31
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((n, c, h, w), generator=g) * 2.0 + 0.5
    if not x32:
        x = x.to(torch.bfloat16)
    gamma, beta, _, _ = params(c, n, seed + 2, False)
    g1 = cl(randn_bf16((n, c, h, w), seed=seed + 1, std=1e-2))
    g2 = cl(torch.randn((n, c, h, w), generator=g).to(x.dtype))
    xa = cl(x).requires_grad_()
    ga, ba = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    ya, ra = G.group_norm_silu_tee(xa, ga, ba, GROUPS, 1e-5)
    torch.autograd.backward([ya, ra], [g1, g2])
    xb = cl(x).requires_grad_()
    gb, bb = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    yb = G.group_norm_silu(xb, gb, bb, GROUPS, 1e-5)
    torch.autograd.backward([yb, xb * 1], [g1, g2])
    torch.cuda.synchronize()
    assert torch.equal(ya, yb) and torch.equal(ra, xb)
    assert xa.grad.dtype == x.dtype
    assert torch.equal(xa.grad, xb.grad)
    assert torch.equal(ga.grad, gb.grad) and torch.equal(ba.grad, bb.grad)


@pytest.mark.parametrize("n,c,h,w,x32", [(2, 128, 32, 32, True), (2, 512, 8, 8, True),
                                         (3, 256, 16, 16, False), (2, 128, 12, 12, True)],
                         ids=lambda v: str(v))
def test_gn_silu_tee_bf16_skip_copy(G, n, c, h, w, x32):
    """With skip_bf16 the tee's second output is x.to(bfloat16) (written by the GroupNorm kernel
    for an fp32 x) and its bf16 gradient is accumulated into x's gradient as autograd does for
    the unfused pair (GroupNormSiLU on x, x.to(bfloat16) for the skip): outputs and all
    gradients bit-identical."""
    seed = n + c + h + 57
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((n, c, h, w), generator=g) * 2.0 + 0.5
    if not x32:
        x = x.to(torch.bfloat16)
    gamma, beta, _, _ = params(c, n, seed + 2, False)
    g1 = cl(randn_bf16((n, c, h, w), seed=seed + 1, std=1e-2))
    g2 = cl(randn_bf16((n, c, h, w), seed=seed + 3, std=1e-1))
    xa = cl(x).requires_grad_()
    ga, ba = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    ya, ra = G.group_norm_silu_tee(xa, ga, ba, GROUPS, 1e-5, True)
    torch.autograd.backward([ya, ra], [g1, g2])
    xb = cl(x).requires_grad_()
    gb, bb = gamma.cuda().requires_grad_(), beta.cuda().requires_grad_()
    yb = G.group_norm_silu(xb, gb, bb, GROUPS, 1e-5)
    rb = xb.to(torch.bfloat16)
    torch.autograd.backward([yb, rb], [g1, g2])
    torch.cuda.synchronize()
    assert ra.dtype == torch.bfloat16
    assert torch.equal(ya, yb) and torch.equal(ra, rb)
    assert xa.grad.dtype == x.dtype
    assert torch.equal(xa.grad, xb.grad)
    assert torch.equal(ga.grad, gb.grad) and torch.equal(ba.grad, bb.grad)


@pytest.mark.parametrize("n,c,groups,h,w,film,f32,p_drop", [
    (64, 128, 32, 33, 32, False, False, 0.0),    # 32-channel slabs, half of the lanes' room
    (51, 128, 32, 48, 41, True, False, 0.2),     # ragged pixels, images not a multiple of 8
    (16, 512, 32, 32, 64, False, True, 0.0),     # 2048 pixels, fp32
    (64, 128, 4, 32, 64, True, False, 0.0),      # one group a slab
    (31, 128, 32, 61, 61, False, False, 0.0),    # 16-channel slabs, odd image
    (33, 128, 32, 64, 64, True, True, 0.2),      # more slabs than one round; fp32, FiLM, dropout
    (8, 512, 32, 64, 64, True, False, 0.2),      # one group a slab
    (9, 256, 32, 64, 57, False, False, 0.0),     # the backward alone takes the thin slabs
], ids=str)
def test_thin_resident_slabs_vs_single_images(G, n, c, groups, h, w, film, f32, p_drop):
    """Images of 1025 to 4096 pixels in batches that fill the GPU run as resident slabs of 32
    or 16 channels; each image by itself runs the chunked form, which sums in another order.
    fp32 statistics differ by a few ulps (1e-5 holds every fp32 result); a bf16 result differs
    where that crosses a rounding boundary, by one ulp: of values off by 2e-6 relative at most
    one in 2^8 * 2e-6, so 2^-8 sqrt(5e-4) = 9e-5 normwise, 2e-4 with a margin. The dropout mask
    hashes the element's index in the batch, so with dropout image 0 alone compares."""
    print("thin slabs", n, c, groups, h, w, film, f32, p_drop, flush=True)
    L, K = dpa_mod("_lib"), dpa_mod("fp8_kernels")
    g = torch.Generator(device="cuda").manual_seed(n + c + h)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    x = (rnd(n, c, h, w) * 1.5 + 0.3).contiguous(memory_format=torch.channels_last)
    x = x if f32 else x.to(torch.bfloat16)
    dout = (rnd(n, c, h, w) * 1e-2).to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
    gamma, beta = 1.0 + 0.3 * rnd(c), 0.3 * rnd(c)
    wb = (0.3 * rnd(n, 2 * c)).to(torch.bfloat16) if film else None
    seed = torch.tensor([987654321], dtype=torch.int64, device="cuda") if p_drop else None
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    hw, dt, st = h * w, int(f32), torch.cuda.current_stream().cuda_stream

    def run(lo, hi):
        m = hi - lo
        xs, ds, ws = x[lo:hi], dout[lo:hi], None if wb is None else wb[lo:hi]
        out, dx = torch.empty_like(xs, dtype=torch.bfloat16), torch.empty_like(xs)
        stats = [torch.empty(m * groups, device="cuda") for _ in range(2)]
        dg, db = torch.empty(c, device="cuda"), torch.empty(c, device="cuda")
        dwb = None if wb is None else torch.empty_like(ws)
        nb = L.query("dpa_gn_silu_fwd_workspace_bytes", m, hw, c, groups)
        buf = torch.empty(nb, device="cuda", dtype=torch.uint8)
        L.call("dpa_gn_silu_fwd_ex", xs.data_ptr(), dt, gamma.data_ptr(), beta.data_ptr(), None,
               None, p(ws), out.data_ptr(), stats[0].data_ptr(), stats[1].data_ptr(),
               buf.data_ptr(), nb, m, hw, c, groups, 1e-5, p(seed), p_drop, None, st)
        nb = L.query("dpa_gn_silu_bwd_workspace_bytes", m, hw, c, groups)
        buf = torch.empty(nb, device="cuda", dtype=torch.uint8)
        L.call("dpa_gn_silu_bwd_ex", xs.data_ptr(), dt, ds.data_ptr(), gamma.data_ptr(),
               beta.data_ptr(), None, None, p(ws), stats[0].data_ptr(), stats[1].data_ptr(),
               dx.data_ptr(), None, 0, dg.data_ptr(), db.data_ptr(), None, None, p(dwb),
               buf.data_ptr(), nb, m, hw, c, groups, p(seed), p_drop, st)
        return out, dx, stats[0], stats[1], dg, db, dwb

    close = lambda a, b: float((a.double() - b.double()).norm() / b.double().norm())  # noqa: E731
    whole = run(0, n)
    singles = [run(i, i + 1) for i in range(1 if p_drop else n)]
    for i, one in enumerate(singles):
        assert close(whole[0][i], one[0][0]) < 2e-4, i
        assert close(whole[1][i], one[1][0]) < (1e-5 if f32 else 2e-4), i
        for k in (2, 3):
            assert close(whole[k][i * groups:(i + 1) * groups], one[k]) < 1e-5, i
        if film:
            assert close(whole[6][i], one[6][0]) < 2e-4, i
    if not p_drop:
        for k in (4, 5):
            assert close(whole[k], torch.stack([one[k].double() for one in singles]).sum(0)) < 1e-5
    # the e4m3 output and the bf16 copy of an fp32 x come from the same values
    hand = K.Fp8Handoff(torch.tensor(0.01, device="cuda"), torch.zeros(1 << 16, device="cuda",
                        dtype=torch.int32), torch.zeros(1, device="cuda", dtype=torch.int32))
    part = [torch.zeros_like(hand.partials), torch.zeros_like(hand.count)]
    x16 = torch.empty_like(x, dtype=torch.bfloat16) if f32 else None
    stats = [torch.empty(n * groups, device="cuda") for _ in range(2)]
    G._fwd_fp8_call(x, gamma, beta, wb, hand, *stats, groups, 1e-5, seed, p_drop, x16)
    q = K.quantize_fp8_delayed_deferred(whole[0], hand.scale, *part)
    assert torch.equal(hand.q.view(torch.uint8), q.view(torch.uint8))
    assert int(hand.partials[:int(hand.count)].max()) == int(part[0][:int(part[1])].max())
    if f32:
        assert torch.equal(x16, x.to(torch.bfloat16))
        (qa, sa), (qb, sb) = K.quantize_fp8_from_producer(x16, x16), K.quantize_fp8(x16)
        assert torch.equal(sa, sb) and torch.equal(qa.view(torch.uint8), qb.view(torch.uint8))

# images that fill their workgroup's pixels in part: one pixel, one more than a lane's first, half
# and most of the room, at every pixel count per lane
PART_CASES = [("bf16", 1, 128, 1, 1, True), ("bf16", 2, 256, 3, 11, False),
              ("bf16", 1, 128, 3, 43, True), ("bf16", 2, 128, 1, 193, False),
              ("bf16", 1, 128, 1, 257, True), ("bf16", 1, 128, 25, 40, False),
              ("f32", 1, 128, 1, 257, False), ("f32", 1, 256, 31, 33, False),
              ("f32", 2, 128, 3, 11, True), ("f32", 1, 128, 3, 43, False),
              ("drop", 1, 128, 1, 257, False), ("drop", 1, 128, 3, 43, True),
              ("drop", 1, 256, 25, 40, True), ("drop", 2, 128, 3, 11, False)]


@pytest.mark.parametrize("kind,n,c,h,w,flag", PART_CASES, ids=str)
def test_images_that_fill_their_workgroups_in_part(G, kind, n, c, h, w, flag):
    """Pixels past the image are left out of every pass: the oracle's tests at such sizes."""
    print("part", kind, n, c, h, w, flag, flush=True)
    {"bf16": test_gn_silu_fwd_bwd_vs_oracle, "f32": test_gn_silu_fp32_input_vs_oracle,
     "drop": test_gn_silu_film_dropout_vs_oracle}[kind](G, n, c, h, w, flag)


@pytest.mark.parametrize("h,w", [(16, 16), (12, 13)], ids=str)
def test_fp32_backward_of_many_images_equals_few(G, h, w):
    """Launches of two and more workgroups per CU form g twice instead of keeping it: the same
    bits as in launches of fewer (129 to 256 pixels, fp32 x, no FiLM, no dropout)."""
    n, c = 130, 256                                    # 520 workgroups, and 260 each half
    g = torch.Generator(device="cuda").manual_seed(h)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    x = (rnd(n, c, h, w) * 1.5 + 0.3).contiguous(memory_format=torch.channels_last)
    dout = (rnd(n, c, h, w) * 1e-2).to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
    gamma, beta = 1.0 + 0.3 * rnd(c), 0.3 * rnd(c)
    _, mean, rstd = G.gn_silu_fwd(x, gamma, beta, GROUPS, 1e-5)
    whole = G.gn_silu_bwd(x, dout, gamma, beta, mean, rstd, GROUPS)
    halves = [G.gn_silu_bwd(x[s], dout[s], gamma, beta, mean.view(n, -1)[s].reshape(-1),
                            rstd.view(n, -1)[s].reshape(-1), GROUPS)
              for s in (slice(0, n // 2), slice(n // 2, n))]
    assert torch.equal(whole[0], torch.cat([t[0] for t in halves]))
    for k in (1, 2):
        ref = halves[0][k].double() + halves[1][k].double()
        # the sums over images in fp32, in slices of another length: 2^-20 of their size
        assert float((whole[k].double() - ref).norm() / ref.norm()) < 2**-20


# (n, c, h, w, film, f32, p_drop, forward on thin slabs, backward on thin slabs): full and nearly
# full rounds of workgroups take them, launches that leave a round mostly empty the chunked form
THIN_LINES = [(32, 128, 64, 64, False, False, 0.0, True, True),
              (36, 128, 64, 64, False, False, 0.0, False, False),
              (64, 128, 64, 64, False, False, 0.0, False, True),
              (64, 128, 64, 64, True, False, 0.0, False, False),
              (8, 512, 64, 64, True, False, 0.2, True, False),
              (32, 128, 33, 32, False, False, 0.0, False, False),
              (48, 128, 33, 32, True, False, 0.0, True, True),
              (72, 128, 33, 32, False, False, 0.0, False, False),
              (96, 128, 33, 32, False, False, 0.0, True, False),
              (144, 128, 33, 32, False, False, 0.0, True, False),
              (112, 128, 33, 32, True, False, 0.2, False, True),
              (16, 512, 33, 32, False, True, 0.0, False, None),
              (16, 512, 36, 37, True, True, 0.2, True, None),
              (32, 512, 33, 32, False, True, 0.0, True, None),
              (32, 512, 33, 32, True, True, 0.2, False, None)]


@pytest.mark.parametrize("n,c,h,w,film,f32,p_drop,fwd_thin,bwd_thin", THIN_LINES, ids=str)
def test_thin_slab_lines_and_fused_casts(G, n, c, h, w, film, f32, p_drop, fwd_thin, bwd_thin):
    """Which form a launch of 1025 to 4096 pixels takes (a launch that casts counts its
    workgroups), and its casts: the e4m3 output and bf16 dx are the deferred casts of the plain
    ones, with the same maximum over the partials counted and nothing written behind them, and the
    partials of an fp32 x's bf16 copy fill their room, zeros where no workgroup wrote."""
    print("lines", n, c, h, w, film, f32, p_drop, flush=True)
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines below are those of 256 CUs")
    L, K = dpa_mod("_lib"), dpa_mod("fp8_kernels")
    hw, st = h * w, torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(n + c + h)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    x = (rnd(n, c, h, w) * 1.5 + 0.3).contiguous(memory_format=torch.channels_last)
    x = x if f32 else x.to(torch.bfloat16)
    gamma, beta = 1.0 + 0.3 * rnd(c), 0.3 * rnd(c)
    wb = (0.3 * rnd(n, 2 * c)).to(torch.bfloat16) if film else None
    seed = torch.tensor([24681357], dtype=torch.int64, device="cuda") if p_drop else None
    mean, rstd = torch.empty(n * GROUPS, device="cuda"), torch.empty(n * GROUPS, device="cuda")
    slab = 32 if hw <= 2048 else 16
    blocks = {True: n * c // slab, False: n * c // 64 * -(-hw // 128)}
    room = L.query("dpa_gn_silu_fp8_partials", n, hw, c, GROUPS)
    assert room == blocks[False]
    poison = 0x7F7F7F7F

    def hand():
        return K.Fp8Handoff(torch.tensor(0.01, device="cuda"),
                            torch.full((room + 64,), poison, device="cuda", dtype=torch.int32),
                            torch.zeros(1, device="cuda", dtype=torch.int32))

    def check_cast(hd, plain, thin):
        count = int(hd.count)
        assert count == blocks[thin]
        assert bool((hd.partials[count:] == poison).all())
        part = [torch.zeros(1 << 16, device="cuda", dtype=torch.int32),
                torch.zeros(1, device="cuda", dtype=torch.int32)]
        q = K.quantize_fp8_delayed_deferred(plain, hd.scale, *part)
        assert torch.equal(hd.q.view(torch.uint8), q.view(torch.uint8))
        assert int(hd.partials[:count].max()) == int(part[0][:int(part[1])].max())

    out = torch.empty_like(x, dtype=torch.bfloat16)
    ws_bytes = L.query("dpa_gn_silu_fwd_workspace_bytes", n, hw, c, GROUPS)
    ws = torch.empty(ws_bytes, device="cuda", dtype=torch.uint8)
    x16 = torch.empty_like(x, dtype=torch.bfloat16) if f32 else None
    args = (x.data_ptr(), int(f32), gamma.data_ptr(), beta.data_ptr(), None, None, p(wb),
            out.data_ptr(), mean.data_ptr(), rstd.data_ptr(), ws.data_ptr(), ws_bytes, n, hw, c,
            GROUPS, 1e-5, p(seed), p_drop, p(x16))
    if f32:
        xbp = torch.full((room + 64,), poison, device="cuda", dtype=torch.int32)
        L.call("dpa_gn_silu_fwd_ex_amax", *args, xbp.data_ptr(), room, st)
        assert bool((xbp[room:] == poison).all()) and bool((xbp[blocks[fwd_thin]:room] == 0).all())
        assert torch.equal(x16, x.to(torch.bfloat16))
        assert int(xbp[:room].max()) == int(x16.abs().max().view(torch.int16))
    else:
        L.call("dpa_gn_silu_fwd_ex", *args, st)
    fwd = hand()
    G._fwd_fp8_call(x, gamma, beta, wb, fwd, mean, rstd, GROUPS, 1e-5, seed, p_drop)
    check_cast(fwd, out, fwd_thin)
    if f32:
        return                                      # (the backward casts a bf16 dx)
    dout = (rnd(n, c, h, w) * 1e-2).to(torch.bfloat16).contiguous(memory_format=torch.channels_last)
    dx = torch.empty_like(x)
    grads = [torch.empty(c, device="cuda") for _ in range(2)]
    dwb = None if wb is None else torch.empty_like(wb)
    ws_bytes = L.query("dpa_gn_silu_bwd_workspace_bytes", n, hw, c, GROUPS)
    ws = torch.empty(ws_bytes, device="cuda", dtype=torch.uint8)
    L.call("dpa_gn_silu_bwd_ex", x.data_ptr(), 0, dout.data_ptr(), gamma.data_ptr(), beta.data_ptr(),
           None, None, p(wb), mean.data_ptr(), rstd.data_ptr(), dx.data_ptr(), None, 0,
           grads[0].data_ptr(), grads[1].data_ptr(), None, None, p(dwb), ws.data_ptr(), ws_bytes,
           n, hw, c, GROUPS, p(seed), p_drop, st)
    bwd = hand()
    bwd.q = torch.empty_like(x, dtype=torch.float8_e4m3fn)
    L.call("dpa_gn_silu_bwd_fp8", x.data_ptr(), dout.data_ptr(), gamma.data_ptr(), beta.data_ptr(),
           None, None, p(wb), mean.data_ptr(), rstd.data_ptr(), bwd.q.data_ptr(),
           bwd.scale.data_ptr(), bwd.partials.data_ptr(), room, bwd.count.data_ptr(),
           grads[0].data_ptr(), grads[1].data_ptr(), None, None, p(dwb), ws.data_ptr(), ws_bytes,
           n, hw, c, GROUPS, p(seed), p_drop, st)
    check_cast(bwd, dx, bwd_thin)
