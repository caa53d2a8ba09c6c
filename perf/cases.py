"""The work that this framework is measured by: single layers of the FP8 U-Net, a residual block
as a sampler runs it, and the whole training step.

``graph`` says how a case runs. The framework trains from a HIP graph captured once
(``trainer.prepare_cuda_graph``), so a training case captures its layer's forward and backward in
``prepare`` and ``run`` replays it; the other cases are eager calls, as a program makes them that
samples from a model or quantizes a tensor.

``exact`` restates the FP8 recipe in 64 bits: per-tensor scale amax / 448 and e4m3 operands
(both defined bit for bit), then sums, norms and products in float64.
"""
import importlib
import math

import torch
import torch.nn.functional as F

_PKG = "diffusion-profiled_amd"
K = importlib.import_module(_PKG + ".fp8_kernels")
GN = importlib.import_module(_PKG + ".gn_silu")
ATT = importlib.import_module(_PKG + ".attention")
UNET = importlib.import_module(_PKG + ".unet")
TRAINER = importlib.import_module(_PKG + ".trainer")

DEV = "cuda"
CL = torch.channels_last
BF16 = torch.bfloat16
T_EMB = 512          # width of the time embedding (4 x base width 128)
GROUPS = 32


# ---- the cases -------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a conv weight quantized by itself, as an op-level program does
        dict(name="quantize_weight", op="quantize", n=128, c=128, h=3, w=3),
        # the largest activation of the model: the 512-channel decoder input at 32x32
        dict(name="quantize_wide", op="quantize", n=128, c=512, h=32, w=32),
        # the attention block's qkv projection over 128 images of 16x16 tokens, both directions
        dict(name="linear_qkv", op="linear", m=32768, k=256, n=768, graph=True),
        # the top level's 3x3 conv at the training batch: forward, data and weight gradient
        dict(name="conv_top", op="conv", batch=128, cin=128, cout=128, h=32, w=32, k=3, stride=1,
             graph=True),
        # a decoder conv of the 16x16 level on a ragged last batch
        dict(name="conv_mid_ragged", op="conv", batch=50, cin=512, cout=256, h=16, w=16, k=3,
             stride=1, graph=True),
        # the 8x8 level's conv: few output tiles for the card
        dict(name="conv_low", op="conv", batch=128, cin=256, cout=256, h=8, w=8, k=3, stride=1,
             graph=True),
        # the top level's conv of a model for 64x64 images
        dict(name="conv_64", op="conv", batch=32, cin=128, cout=128, h=64, w=64, k=3, stride=1,
             graph=True),
        # the second norm of a top-level block as it trains: FiLM, SiLU, dropout
        dict(name="norm_film_top", op="norm", batch=128, c=128, h=32, w=32, film=True, p_drop=0.2,
             f32=False, graph=True),
        # the first norm of a top-level block for 64x64 images
        dict(name="norm_64", op="norm", batch=32, c=128, h=64, w=64, film=False, p_drop=0.0,
             f32=False, graph=True),
        # self-attention of the 16x16 level, forward and backward
        dict(name="attention_16x16", op="attention", batch=128, tokens=256, heads=4, graph=True),
        # one decoder block of a sampler that draws 16 images: eager, forward only
        dict(name="block_sample", op="block", batch=16, cin=512, cout=256, side=16, train=False,
             p_drop=0.0, graph=False),
        # the training step of the benchmark U-Net: forward, backward, AdamW, EMA
        dict(name="train_step", op="step", batch=128),
    ]


def _logint(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    op = rng.choice(["quantize", "linear", "conv", "conv", "conv", "norm", "norm", "attention",
                     "block", "block", "step"])
    if op == "quantize":
        if rng.random() < 0.4:      # weights
            k = rng.choice([1, 3])
            return dict(op=op, n=rng.choice([128, 256, 512]), c=rng.choice([128, 256, 512]), h=k, w=k)
        c, side = rng.choice([128, 256, 512]), _logint(rng, 4, 64)
        most = max(1, min(160, (1 << 26) // (c * side * side)))
        return dict(op=op, n=_logint(rng, 1, most), c=c, h=side, w=side)
    if op == "linear":
        return dict(op=op, m=_logint(rng, 32, 40000), k=128 * rng.randint(1, 6),
                    n=128 * rng.randint(1, 8), graph=rng.random() < 0.7)
    if op == "conv":
        cin, cout = 128 * rng.choice([1, 2, 2, 4]), 128 * rng.choice([1, 2, 2, 4])
        if rng.random() < 0.6:
            h = w = rng.choice([4, 8, 16, 32, 64])
        else:
            h, w = _logint(rng, 4, 64), _logint(rng, 4, 64)
        k, stride = rng.choice([(3, 1), (3, 1), (3, 1), (3, 2), (1, 1)])
        most = max(1, min(160, int(1.2e11 / (h * w * cin * cout * k * k * 2))))
        return dict(op=op, batch=_logint(rng, 1, most), cin=cin, cout=cout, h=h, w=w, k=k,
                    stride=stride, graph=rng.random() < 0.7)
    if op == "norm":
        c, film = rng.choice([128, 256, 512]), rng.random() < 0.5
        h, w = ((side, side) if (side := rng.choice([4, 8, 16, 32, 64, 0]))
                else (_logint(rng, 4, 64), _logint(rng, 4, 64)))
        most = max(1, min(160, (1 << 25) // (c * h * w)))
        return dict(op=op, batch=_logint(rng, 1, most), c=c, h=h, w=w, film=film,
                    p_drop=rng.choice([0.0, 0.2]) if film else 0.0, f32=rng.random() < 0.4,
                    graph=rng.random() < 0.7)
    if op == "attention":
        return dict(op=op, batch=_logint(rng, 1, 128), tokens=16 * _logint(rng, 1, 16),
                    heads=rng.choice([1, 2, 4, 8]), graph=rng.random() < 0.7)
    if op == "block":
        cin, cout = rng.choice([(128, 128), (128, 256), (256, 256), (512, 256)])
        train = rng.random() < 0.5
        side = rng.choice([4, 8, 16, 32])
        return dict(op=op, batch=_logint(rng, 1, 128 if cin < 512 or side < 32 else 64), cin=cin,
                    cout=cout, side=side, train=train, p_drop=0.1 if train else 0.0, graph=train)
    return dict(op=op, batch=_logint(rng, 16, 128))


# ---- inputs ----------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, shape, std=1.0, dtype=BF16, cl=False):
    t = (torch.randn(shape, generator=g, device=DEV) * std).to(dtype)
    return t.contiguous(memory_format=CL) if cl else t


def _uniform(g, shape, bound):
    t = (torch.rand(shape, generator=g, device=DEV) * 2 - 1) * bound
    return t.contiguous(memory_format=CL) if t.ndim == 4 else t


def _weight(g, shape):
    """Kaiming-uniform as nn.Conv2d and nn.Linear draw it."""
    return _uniform(g, shape, 1.0 / math.sqrt(math.prod(shape[1:])))


def _out_side(n, k, stride):
    return (n + 2 * (k // 2) - k) // stride + 1


def _inputs(case, seed):
    """The tensors of a case, from the seed alone (the training step makes its own)."""
    g, op = _gen(seed), case["op"]
    if op == "quantize":
        shape = (case["n"], case["c"], case["h"], case["w"])
        if case["h"] in (1, 3):
            return dict(x=_weight(g, shape).to(BF16).contiguous(memory_format=CL))
        return dict(x=_randn(g, shape, cl=True))
    if op == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(x=_randn(g, (m, k)), w=_weight(g, (n, k)), dy=_randn(g, (m, n), 1e-2))
    if op == "conv":
        b, cin, cout, k, s = (case[v] for v in ("batch", "cin", "cout", "k", "stride"))
        oh, ow = _out_side(case["h"], k, s), _out_side(case["w"], k, s)
        return dict(x=_randn(g, (b, cin, case["h"], case["w"]), cl=True),
                    w=_weight(g, (cout, cin, k, k)),
                    dy=_randn(g, (b, cout, oh, ow), 1e-2, cl=True))
    if op == "norm":
        b, c = case["batch"], case["c"]
        shape = (b, c, case["h"], case["w"])
        d = dict(x=_randn(g, shape, 1.5, torch.float32 if case["f32"] else BF16, cl=True),
                 gamma=1 + _uniform(g, (c,), 0.3), beta=_uniform(g, (c,), 0.3),
                 dy=_randn(g, shape, 1e-2, cl=True))
        if case["film"]:
            d["wb"] = _randn(g, (b, 2 * c, 1, 1), 0.3)
        return d
    if op == "attention":
        b, length, c = case["batch"], case["tokens"], 64 * case["heads"]
        return dict(x=_randn(g, (b, length, 3 * c)), dy=_randn(g, (b, length, c), 1e-2))
    if op == "block":
        b, cin, cout, s = case["batch"], case["cin"], case["cout"], case["side"]
        return dict(x=_randn(g, (b, cin, s, s), cl=True), t=F.silu(_randn(g, (b, T_EMB))),
                    conv_1=_weight(g, (cout, cin, 3, 3)), conv_2=_weight(g, (cout, cout, 3, 3)),
                    skip=_weight(g, (cout, cin, 1, 1)), film=_weight(g, (2 * cout, T_EMB)),
                    g1=1 + _uniform(g, (cin,), 0.3), b1=_uniform(g, (cin,), 0.3),
                    g2=1 + _uniform(g, (cout,), 0.3), b2=_uniform(g, (cout,), 0.3),
                    dy=_randn(g, (b, cout, s, s), 1e-2, cl=True))
    raise ValueError(op)


def _grad(t):
    return t.requires_grad_(True)


def _conv(x, w, case):
    if (case["k"], case["stride"]) == (3, 1) and (
            case["cin"], case["cout"], case["h"], case["w"]) in K.SUPPORTED_UNET_SHAPES:
        return K.triton_conv2d_fp8(x, w)
    return K.conv2d_fp8(x, w, case["stride"], case["k"] // 2)


def _block(case, d):
    config = UNET.cfg5_config(fp8_scaling_type="current", p_drop=case["p_drop"])
    block = UNET.ResidualBlock(config, case["cin"], case["cout"], p_drop=case["p_drop"])
    block = block.to(DEV).to(memory_format=CL)
    with torch.no_grad():
        named = [(block.conv_1.conv.weight, "conv_1"), (block.conv_2.conv.weight, "conv_2"),
                 (block.t_embed_wb.mlp.weight, "film"), (block.norm1.weight, "g1"),
                 (block.norm1.bias, "b1"), (block.norm2.weight, "g2"), (block.norm2.bias, "b2")]
        if case["cin"] != case["cout"]:
            named.append((block.skip_connection.weight, "skip"))
        for p, key in named:
            p.copy_(d[key])
    return block.train(case["train"])


def _capture(call):
    """One pass as a HIP graph: (graph, its output buffers)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            call()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def _train_state(batch, seed):
    """The benchmark U-Net's captured training step. The projections that start at zero get
    ordinary weights, as after some training; all weights lie in one buffer, so that they
    come back whole as one output."""
    g = _gen(seed)
    st = TRAINER.TrainState(UNET.cfg5_config(), batch, seed=seed)
    weights = [p for p in st.model.parameters()]
    sizes = [-(-p.numel() // 64) * 64 for p in weights]
    flat = torch.zeros(sum(sizes), device=DEV)
    at = 0
    with torch.no_grad():
        for p, size in zip(weights, sizes):
            if p.ndim > 1 and not bool(p.any()):
                p.copy_(_weight(g, tuple(p.shape)))
            home = flat[at:at + p.numel()]
            if p.ndim == 4:
                o, i, r, s = p.shape
                home = home.view(o, r, s, i).permute(0, 3, 1, 2)
            else:
                home = home.view(p.shape)
            p.data = home.copy_(p)
            at += size
        st.ema_ddpm.model.model.load_state_dict(st.model.state_dict())
    st.set_batch(torch.rand(st.static_batch.shape, generator=g, device=DEV) * 2 - 1)
    st.capture()
    return dict(op="step", st=st, flat=flat)


def prepare(case, seed):
    if case["op"] == "step":
        return _train_state(case["batch"], seed)
    torch.manual_seed(seed)
    d = _inputs(case, seed)
    s = dict(op=case["op"], graph=None)
    op = case["op"]
    if op == "quantize":
        s["call"] = lambda: K.quantize_fp8(d["x"])
    elif op == "linear":
        x, w = _grad(d["x"]), _grad(d["w"])

        def call():
            y = K.linear_fp8_autograd(x, w)
            return (y.detach(), *torch.autograd.grad(y, (x, w), d["dy"]))
        s["call"] = call
    elif op == "conv":
        x, w = _grad(d["x"]), _grad(d["w"])

        def call():
            y = _conv(x, w, case)
            return (y.detach(), *torch.autograd.grad(y, (x, w), d["dy"]))
        s["call"] = call
    elif op == "norm":
        x, gamma, beta = _grad(d["x"]), _grad(d["gamma"]), _grad(d["beta"])
        leaves = [x, gamma, beta]
        if case["film"]:
            leaves.append(_grad(d["wb"]))

        def call():
            if case["film"]:
                y = GN.group_norm_silu_film(x, gamma, beta, GROUPS, 1e-5, leaves[3],
                                            case["p_drop"])
            else:
                y = GN.group_norm_silu(x, gamma, beta, GROUPS, 1e-5)
            return (y.detach(), *torch.autograd.grad(y, leaves, d["dy"]))
        s["call"] = call
    elif op == "attention":
        x = _grad(d["x"])

        def call():
            y = ATT.self_attention_qkv(x, case["heads"])
            return (y.detach(), *torch.autograd.grad(y, (x,), d["dy"]))
        s["call"] = call
    else:
        block = _block(case, d)
        if case["train"]:
            x, t = _grad(d["x"]), _grad(d["t"])
            leaves = [x, t, *block.parameters()]

            def call():
                with torch.autocast(DEV, dtype=BF16):
                    y = block(x, t)
                return (y.detach(), *torch.autograd.grad(y, leaves, d["dy"]))
        else:
            def call():
                with torch.no_grad(), torch.autocast(DEV, dtype=BF16):
                    return block(d["x"], d["t"])
        s["call"] = call
    if case.get("graph"):
        s["graph"], s["out"] = _capture(s["call"])
    return s


def run(state):
    if state["op"] == "step":
        st = state["st"]
        st.loss_acc.zero_()
        st.replay()
        return dict(loss=st.loss_acc, weights=state["flat"])
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return state["call"]()


# ---- what a pass cannot do without -------------------------------------------------------
def work(case):
    op = case["op"]
    if op == "quantize":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        return dict(bytes=3 * n, flops=0)
    if op == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=4 * m * (k + n) + 8 * n * k, flops=6 * m * n * k)
    if op == "conv":
        pin = case["batch"] * case["h"] * case["w"]
        pout = (case["batch"] * _out_side(case["h"], case["k"], case["stride"])
                * _out_side(case["w"], case["k"], case["stride"]))
        nw = case["cin"] * case["cout"] * case["k"] ** 2
        return dict(bytes=4 * (pin * case["cin"] + pout * case["cout"]) + 8 * nw, flops=6 * pout * nw)
    if op == "norm":
        n = case["batch"] * case["c"] * case["h"] * case["w"]
        return dict(bytes=n * (12 if case["f32"] else 8), flops=0)
    if op == "attention":
        b, length, c = case["batch"], case["tokens"], 64 * case["heads"]
        return dict(bytes=16 * b * length * c, flops=14 * b * length * length * c)
    if op == "block":
        cin, cout, px = case["cin"], case["cout"], case["batch"] * case["side"] ** 2
        nw = 9 * cout * (cin + cout) + (cin * cout if cin != cout else 0)
        passes = 3 if case["train"] else 1
        return dict(bytes=2 * px * (cin + cout) * (2 if case["train"] else 1)
                    + 4 * nw * (2 if case["train"] else 1), flops=passes * 2 * px * nw)
    # the step: 4.1186 TFLOP of FP8 products at batch 128; 33.6 M weights, their two moments
    # and EMA read and written, and the gradient between the backward and the update
    return dict(bytes=33.6e6 * 4 * 10, flops=4.1186e12 * case["batch"] / 128)


def tolerance(case):
    op = case["op"]
    if op == "quantize":
        return "exact"
    if op == "step":
        # the split reductions summed in another order: loss off by 2.2e-4, weights by 3e-5
        # (one of them by 0.009 of their root mean square)
        return dict(rel=2e-3, max=0.04)
    if op == "block":
        # 2.6e-3 off the 64-bit result: bf16 stores between two e4m3 convs
        return dict(rel=1e-2, max=0.1)
    # bf16 outputs: 1.7e-3 off the 64-bit result (attention 2.4e-3)
    return dict(rel=7e-3, max=0.05)


# ---- the same in 64 bits -----------------------------------------------------------------
def _quantized64(t):
    """(e4m3 values, scale) of a tensor, both in float64: scale = RN32(amax / 448)."""
    b = t.detach().to(BF16).double()
    amax = float(b.abs().max())
    scale = float(torch.tensor(amax, dtype=torch.float64).div(448).float()) if amax > 0 else 1.0
    q = (b / scale).float().clamp(-448, 448).to(torch.float8_e4m3fn).double()
    return q, scale


def _dequantized64(t):
    q, scale = _quantized64(t)
    return q * scale


def _conv64(x, w, stride):
    """NHWC-logical float64 conv as one product per tap; x [N, C, H, W], w [O, C, k, k]."""
    k = w.shape[2]
    oh, ow = _out_side(x.shape[2], k, stride), _out_side(x.shape[3], k, stride)
    xp = F.pad(x.permute(0, 2, 3, 1), (0, 0, k // 2, k // 2, k // 2, k // 2))
    y = 0
    for r in range(k):
        for s in range(k):
            part = xp[:, r:r + (oh - 1) * stride + 1:stride, s:s + (ow - 1) * stride + 1:stride]
            y = y + part.reshape(-1, x.shape[1]) @ w[:, :, r, s].t().contiguous()
    return y.view(x.shape[0], oh, ow, w.shape[0]).permute(0, 3, 1, 2)


def _norm64(x, gamma, beta, scale=None, shift=None):
    n, c = x.shape[:2]
    g = x.reshape(n, GROUPS, -1)
    mean, var = g.mean(-1, keepdim=True), g.var(-1, unbiased=False, keepdim=True)
    h = ((g - mean) / (var + 1e-5).sqrt()).reshape(x.shape) * gamma.view(1, c, 1, 1)
    h = h + beta.view(1, c, 1, 1)
    if scale is not None:
        h = h * scale + shift
    return F.silu(h)


def _film64(wb):
    """The FiLM pair as the model rounds it: bf16(w + 1) and b."""
    w, b = wb.chunk(2, dim=1)
    return (w + 1).double(), b.double()


def _leaf64(t):
    return t.detach().double().requires_grad_(True)


def exact(case, seed):
    op = case["op"]
    if op == "step" or (op == "block" and case["train"]) or case.get("p_drop"):
        return None      # dropout's mask is the framework's own
    d = _inputs(case, seed)
    if op == "quantize":
        return _quantized64(d["x"])
    if op == "linear":
        x, w, dy = (_dequantized64(d[v]) for v in ("x", "w", "dy"))
        return x @ w.t().contiguous(), dy @ w, dy.t().contiguous() @ x
    if op == "conv":
        x = _dequantized64(d["x"]).requires_grad_(True)
        w = _dequantized64(d["w"]).requires_grad_(True)
        y = _conv64(x, w, case["stride"])
        return (y.detach(), *torch.autograd.grad(y, (x, w), _dequantized64(d["dy"])))
    if op == "norm":
        x, gamma, beta = _leaf64(d["x"]), _leaf64(d["gamma"]), _leaf64(d["beta"])
        film = [_leaf64(v) for v in _film64(d["wb"])] if case["film"] else []
        y = _norm64(x, gamma, beta, *film)
        grads = torch.autograd.grad(y, (x, gamma, beta, *film), d["dy"].double())
        if film:
            grads = (*grads[:3], torch.cat(grads[3:], dim=1))
        return (y.detach(), *grads)
    if op == "attention":
        x = _leaf64(d["x"])
        b, length, c3 = x.shape
        q, k, v = (t.reshape(b, length, case["heads"], 64).transpose(1, 2).contiguous()
                   for t in x.chunk(3, dim=-1))
        p = torch.softmax(q @ k.transpose(2, 3).contiguous() / 8.0, dim=-1)
        y = (p @ v).transpose(1, 2).reshape(b, length, c3 // 3)
        return (y.detach(), *torch.autograd.grad(y, (x,), d["dy"].double()))
    # the residual block, rounded where it stores bf16
    r = lambda t: t.to(BF16).double()  # noqa: E731
    wb = r(_dequantized64(d["t"]) @ _dequantized64(d["film"]).t().contiguous())
    scale, shift = _film64(wb.to(BF16)[:, :, None, None])
    x = d["x"].double()
    h = r(_norm64(x, d["g1"].double(), d["b1"].double()))
    h = r(_conv64(_dequantized64(h), _dequantized64(d["conv_1"]), 1))
    h = r(_norm64(h, d["g2"].double(), d["b2"].double(), scale, shift))
    h = _conv64(_dequantized64(h), _dequantized64(d["conv_2"]), 1)
    skip = x if case["cin"] == case["cout"] else r(
        _conv64(_dequantized64(x), _dequantized64(d["skip"]), 1))
    return (skip + r(h)) / math.sqrt(2.0)
