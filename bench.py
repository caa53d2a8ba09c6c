"""Benchmark of the MI355X FP8 conv path (one GPU).

A step is one pass of the hot path over one batch: the FP8 3x3 conv of BASELINE config 2
(NHWC [128,32,32,128] -> 128, stride 1, pad 1) forward + data gradient + weight gradient,
including the per-tensor e4m3 quantization of x, w and dy — exactly what
Conv2dFP8Specialized does per layer in the reference (diffusion/fp8_kernels.py:826-913).

    python bench.py [--steps K] [--warmup W] [--workload cfg2|cfg1|cfg3|cfg3s2|cfg3k1|cfg4|cfg5]

Prints ONE JSON line. `value` is TFLOP/s of algorithmic conv work (3 x 2*M*N*K per step)
with inputs resident in HBM; ten steps are captured back to back as one HIP graph
(--steps-per-graph) and exactly K steps are replayed (whole graphs, then a one-step graph for
any remainder; wall clock around the replays, synchronised on both sides). A replay boundary
costs ~4-7 µs that a conv inside a captured training step does not pay; the time with one
step per replay is reported beside it (`ms_per_step_one_step_graphs`). `roofline` is for the dominant
kernel: HIP events around a graph replay of many calls, recorded on the replay stream (the
stream every kernel of the library is launched on). `cpu_baseline` times the
oracle's CPU path (the reference recipe on torch CPU: e4m3 round trip + fp32 conv) on a
bounded sample of the same workload. The default run also measures the graph-captured U-Net
training step at batch 128 (`unet_train_step`, the second half of the metric).

cfg4 (one ResidualBlock fwd+bwd at 16x16/256/batch 128) and cfg5 (the full training step:
forward, backward, clip, AdamW, EMA) are model-level workloads; their `value` is TFLOP/s of
FP8 GEMM work (cfg4) and training steps/s (cfg5).
"""
from __future__ import annotations

import argparse
import importlib
import json
import os
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "FP8 conv/GEMM TFLOP/s (% of MFMA peak); U-Net train steps/s at batch 128"
PEAK_FP8_TFLOPS = 5000.0  # MI355X dense FP8 MFMA
PEAK_HBM_GBS = 8000.0
PROFILE_TRAFFIC = os.path.join(ROOT, "profiles", "traffic.json")


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--steps-per-graph", type=int, default=10,
                    help="cfg1-cfg3: steps captured back to back in one HIP graph (the timed "
                         "steps are exactly --steps: whole graphs, then single-step replays)")
    ap.add_argument("--workload", default="cfg2",
                    choices=["cfg2", "cfg1", "cfg3", "cfg3s2", "cfg3k1", "cfg4", "cfg5", "gn32",
                             "attn256"],
                    help="gn32 / attn256: component lines (profiling evidence) for the fused "
                         "GroupNorm and the self-attention kernels at cfg5's shapes")
    ap.add_argument("--no-unet", action="store_true", help="skip the U-Net step in the cfg2 line")
    ap.add_argument("--part", default=None,
                    help="profiling mode: run only this part (quantize|fwd|dgrad|wgrad) of the "
                         "workload --reps times, print nothing else")
    ap.add_argument("--reps", type=int, default=5)
    ap.add_argument("--copy-mib", type=int, default=0,
                    help="profiling mode: --reps device copies of this many MiB (counter "
                         "calibration: a plain copy reads and writes exactly that many bytes)")
    ap.add_argument("--kernel-reps", type=int, default=50)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--hconv-phases", action="store_true",
                    help="time attribution of the halo-patch conv on cfg2: builds a copy of "
                         "csrc/hconv.hip with per-wave clock stamps in a temporary directory "
                         "and reports where the launch's time goes")
    ap.add_argument("--cpu-seconds", type=float, default=15.0)
    return ap.parse_args()


def seeded(shape, seed, std=1.0, kaiming=False):
    g = torch.Generator().manual_seed(seed)
    if kaiming:
        import math

        fan_in = 1
        for d in shape[1:]:
            fan_in *= d
        b = 1.0 / math.sqrt(fan_in)
        return (torch.rand(shape, generator=g) * 2 * b - b).to(torch.bfloat16)
    return (torch.randn(shape, generator=g) * std).to(torch.bfloat16)


def library_kernels(n, h, w, cin, cout, k, stride, pad):
    """(forward, data gradient, weight gradient) kernels of a conv into aligned outputs."""
    lib = importlib.import_module("diffusion-profiled_amd._lib").load()
    names = (lib.dpa_conv2d_kernel(p, 16, n, h, w, cin, cout, k, k, stride, pad) for p in range(3))
    return tuple(v.decode() for v in names)


class ConvWorkload:
    """One FP8 conv layer fwd + dgrad + wgrad with current scaling."""

    def __init__(self, K, n, cin, cout, h, w, k, stride, pad, name):
        self.K = K
        self.n, self.cin, self.cout, self.h, self.w, self.k = n, cin, cout, h, w, k
        self.stride, self.pad = stride, pad
        self.p = (h + 2 * pad - k) // stride + 1
        self.q = (w + 2 * pad - k) // stride + 1
        self.name = name
        cl = torch.channels_last
        self.x = seeded((n, cin, h, w), 0).cuda().contiguous(memory_format=cl)
        self.wt = seeded((cout, cin, k, k), 1, kaiming=True).cuda().contiguous(memory_format=cl)
        self.dy = seeded((n, cout, self.p, self.q), 2, std=1e-2).cuda().contiguous(memory_format=cl)
        self.flop = 2.0 * n * self.p * self.q * cout * cin * k * k  # per GEMM (fwd/dgrad/wgrad)
        # algorithmic bytes (e4m3 operands, bf16 outputs)
        self.bytes = {
            "fwd": n * h * w * cin + cout * k * k * cin + 2 * n * self.p * self.q * cout,
            "dgrad": n * self.p * self.q * cout + cout * k * k * cin + 2 * n * h * w * cin,
            "wgrad": n * h * w * cin + n * self.p * self.q * cout + 2 * cout * k * k * cin,
        }
        self.quant_bytes = 3 * (n * h * w * cin + cout * k * k * cin + n * self.p * self.q * cout)
        self.wprep = None

    def quantize(self):
        """x and dy: quantize_fp8 (amax + cast each). The weight: its e4m3 copy, scale and the
        data gradient's transposed copy in a grouped weight preparation whose blocks run inside
        x's amax and cast launches (two launches for x and the weight, in place of
        quantize_fp8's two per tensor and the transpose); for the halo-patch kernel's shapes
        both copies are written in its fragment layouts."""
        self.quantize_xw()
        self.quantize_dy()

    def quantize_xw(self):
        if self.wprep is None:
            WP = importlib.import_module("diffusion-profiled_amd.weight_prep")
            self.wprep = WP.TensorPrep([self.wt], frag=[self.frag])
        self.xq, self.xs = self.wprep.run_with_quantize(self.x)
        self.wq, self.wq_t, self.ws = self.wprep.q[0], self.wprep.qt[0], self.wprep.scale(0)

    def quantize_dy(self):
        self.dyq, self.dys = self.K.quantize_fp8(self.dy)

    @property
    def frag(self):
        return self.K.hconv_shape(self.n, self.cin, self.cout, self.h, self.w, self.k,
                                  self.stride, self.pad)

    def fwd(self):
        if self.frag:   # q / qt hold the halo-patch kernel's fragment layouts
            return self.K.conv2d_fp8_fwd_wf(self.xq, self.wq, self.xs, self.ws, self.cout)
        return self.K.conv2d_fp8_fwd_general(self.xq, self.wq, self.xs, self.ws, self.stride, self.pad)

    def dgrad(self):
        """The data-gradient GEMM kernel alone (the transposed weight comes from quantize)."""
        if self.frag:
            return self.K.conv2d_fp8_dgrad_wf(self.dyq, self.wq_t, self.dys, self.ws, self.cin)
        return self.K.conv2d_fp8_dgrad_general(self.dyq, self.wq, self.dys, self.ws, (self.h, self.w),
                                               self.stride, self.pad, weight_t=self.wq_t)

    def wgrad(self):
        return self.K.conv2d_fp8_wgrad_general(self.xq, self.dyq, self.xs, self.dys, self.k,
                                               self.stride, self.pad)

    def step(self):
        """In the order of the reference's autograd Function (diffusion/fp8_kernels.py:823-913):
        x and w quantized, forward; then dy quantized, data and weight gradients."""
        self.quantize_xw()
        self.fwd()
        self.quantize_dy()
        self.dgrad()
        self.wgrad()

    def parts(self):
        return {"quantize": self.quantize, "fwd": self.fwd, "dgrad": self.dgrad,
                "wgrad": self.wgrad}

    def step_flop(self):
        return 3 * self.flop

    def kernel_names(self):
        """Kernels that the library says it launches for this layer's GEMMs."""
        fwd, dgrad, wg = library_kernels(self.n, self.h, self.w, self.cin, self.cout, self.k,
                                         self.stride, self.pad)
        return {"fwd": fwd, "dgrad": dgrad, "wgrad": wg + "+wgrad_reduce_kernel"}

    def config(self):
        return {
            "workload": self.name,
            "batch": self.n, "cin": self.cin, "cout": self.cout, "h": self.h, "w": self.w,
            "kernel": self.k, "stride": self.stride, "pad": self.pad,
            "layout": "NHWC activations, OHWI weights, e4m3 per-tensor current scaling",
            "step": "quantize x,w + conv fwd + quantize dy + dgrad + wgrad",
        }


class GemmWorkload:
    """cfg1: FP8 linear forward X[32768,256] . W[768,256]^T with current scaling."""

    def __init__(self, K):
        self.K = K
        self.m, self.nn, self.kk = 32768, 768, 256
        self.x = seeded((self.m, self.kk), 0).cuda()
        self.wt = seeded((self.nn, self.kk), 1, kaiming=True).cuda()
        self.flop = 2.0 * self.m * self.nn * self.kk
        self.bytes = {"fwd": self.m * self.kk + self.nn * self.kk + 2 * self.m * self.nn}
        self.quant_bytes = 3 * (self.m * self.kk + self.nn * self.kk)
        self.name = "cfg1: FP8 linear fwd X[32768,256] x W[768,256]^T -> bf16, incl. e4m3 quantization"

    def quantize(self):
        self.xq, self.xs = self.K.quantize_fp8_tensor(self.x)
        self.wq, self.ws = self.K.quantize_fp8_tensor(self.wt)

    def fwd(self):
        return self.K.linear_fp8_prequantized(self.xq, self.wq, self.xs, self.ws)

    def step(self):
        self.quantize()
        self.fwd()

    def parts(self):
        return {"quantize": self.quantize, "fwd": self.fwd}

    def step_flop(self):
        return self.flop

    def kernel_names(self):
        return {"fwd": library_kernels(self.m, 1, 1, self.kk, self.nn, 1, 1, 0)[0]}

    def config(self):
        return {"workload": self.name, "m": self.m, "n": self.nn, "k": self.kk}


def fp8_gemm_flops(model, batch, res=32):
    """Forward FLOPs (2*M*N*K) of every FP8 GEMM site of a U-Net (3x3 and 1x1 convs,
    linears) at the given batch, from one shape-tracing forward on the CPU with FP8 off."""
    import copy

    U = importlib.import_module("diffusion-profiled_amd.unet")
    cfg = copy.deepcopy(model.config)
    cfg.fp8_convs_enabled = cfg.fp8_linears = False
    probe = U.UNet(cfg)
    total = [0.0]

    def conv_hook(mod, inp, out):
        w = mod.conv.weight if isinstance(mod, U.Conv2dFP8) else mod.weight
        total[0] += 2.0 * out.shape[0] * out.shape[2] * out.shape[3] * w.shape[0] * w[0].numel()

    def lin_hook(mod, inp, out):
        total[0] += 2.0 * out.numel() * mod.in_features

    for m in probe.modules():
        if isinstance(m, (U.Conv2dFP8, U.Conv1x1FP8)):
            m.register_forward_hook(conv_hook)
        elif isinstance(m, U.LinearFP8):
            m.register_forward_hook(lin_hook)
    with torch.no_grad():
        probe(torch.zeros(1, cfg.in_channels, res, res), torch.zeros(1, dtype=torch.long))
    return total[0] * batch


class ResBlockWorkload:
    """cfg4: one ResidualBlock (GN+SiLU -> FP8 3x3 -> FiLM -> GN+SiLU -> dropout 0.1 -> FP8
    3x3 -> residual) at [128,256,16,16], forward + backward under bf16 autocast."""

    def __init__(self):
        U = importlib.import_module("diffusion-profiled_amd.unet")
        cfg = U.cfg5_config(fp8_scaling_type="current", p_drop=0.1)
        torch.manual_seed(0)
        self.blk = U.ResidualBlock(cfg, 256, 256, p_drop=0.1).cuda().to(memory_format=torch.channels_last)
        import math

        torch.nn.init.kaiming_uniform_(self.blk.conv_2.conv.weight, a=math.sqrt(5))
        cl = torch.channels_last
        self.x = seeded((128, 256, 16, 16), 0).cuda().contiguous(memory_format=cl).requires_grad_()
        g = torch.Generator().manual_seed(3)
        self.temb = torch.randn((128, 512), generator=g).to(torch.bfloat16).cuda().requires_grad_()
        self.dout = seeded((128, 256, 16, 16), 2, std=1e-2).cuda().contiguous(memory_format=cl)
        self.flop = 2.0 * 128 * 16 * 16 * 256 * 256 * 9      # one conv GEMM
        self.name = ("cfg4: ResidualBlock 256->256 @16x16, batch 128, fused GN+SiLU(+FiLM), FP8 3x3 "
                     "convs, dropout 0.1, fwd+bwd")

    def step(self):
        for p in self.blk.parameters():
            p.grad = None
        self.x.grad = None
        self.temb.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = self.blk(self.x, self.temb)
        out.backward(self.dout)

    def step_flop(self):
        return 6 * self.flop

    def config(self):
        return {"workload": self.name, "batch": 128, "channels": 256, "h": 16, "w": 16}


class UNetStepWorkload:
    """cfg5: the full DDPM U-Net training step at batch 128 (forward, eps-MSE, backward,
    clip_grad_norm, AdamW, EMA), captured as one HIP graph (the reference's
    prepare_cuda_graph, train.py:104-149)."""

    def __init__(self, batch=128):
        U = importlib.import_module("diffusion-profiled_amd.unet")
        T = importlib.import_module("diffusion-profiled_amd.trainer")
        self.batch = batch
        self.state = T.TrainState(U.cfg5_config(), batch=batch, lr=2e-4, seed=0)
        g = torch.Generator().manual_seed(4)
        self.state.set_batch((torch.rand((batch, 3, 32, 32), generator=g) * 2 - 1).cuda())
        self.fwd_flop = fp8_gemm_flops(self.state.model, batch)
        self.name = ("cfg5: DDPM U-Net train step, ch 128, mults (1,2,2,2), 2 ResBlocks/level, "
                     "attention at 16x16 and 8x8 + mid, 33.57M params, batch 128, FP8 convs+linears "
                     "(delayed scaling), AdamW lr 2e-4, EMA, one HIP graph")

    def capture(self):
        self.state.capture(warmup=3)

    def step(self):
        self.state.replay()

    def step_flop(self):
        return 3 * self.fwd_flop

    def config(self):
        return {"workload": self.name, "batch": self.batch, "image": [3, 32, 32],
                "params": sum(p.numel() for p in self.state.model.parameters())}


def time_graph_steps(g_replay, steps, warmup):
    for _ in range(warmup):
        g_replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        g_replay()
    torch.cuda.synchronize()
    return (time.perf_counter() - t0) / steps


def unet_step_summary(steps, warmup):
    wl = UNetStepWorkload()
    wl.capture()
    dt = time_graph_steps(wl.step, steps, warmup)
    loss = float(wl.state.loss_acc) / max(1, steps + warmup)
    return wl, dt, {
        "steps_per_s": round(1.0 / dt, 3),
        "ms_per_step": round(dt * 1e3, 3),
        "fp8_gemm_tflops": round(wl.step_flop() / dt / 1e12, 2),
        "fp8_gemm_tflop_per_step": round(wl.step_flop() / 1e12, 4),
        "mean_loss": round(loss, 5),
        "config": wl.config(),
    }


class GroupNormWorkload:
    """The residual block's second GroupNorm (diffusion/unet.py:157-160: GroupNorm(32) -> FiLM
    from the bf16 time projection -> SiLU -> dropout 0.2) at the 32x32 level of cfg5,
    [128, 128, 32, 32] bf16 channels-last, forward + backward. Algorithmic bytes: 4 B/element
    forward (x in, y out), 6 B/element backward (x, dout in, dx out)."""

    def __init__(self):
        self.G = importlib.import_module("diffusion-profiled_amd.gn_silu")
        n, c, h, w = 128, 128, 32, 32
        cl = torch.channels_last
        self.x = seeded((n, c, h, w), 0).cuda().contiguous(memory_format=cl).requires_grad_()
        g = torch.Generator().manual_seed(1)
        self.gamma = (1.0 + 0.1 * torch.randn(c, generator=g)).cuda()
        self.beta = (0.1 * torch.randn(c, generator=g)).cuda()
        self.wb = (0.3 * torch.randn((n, 2 * c, 1, 1), generator=g)).to(torch.bfloat16).cuda()
        self.dout = seeded((n, c, h, w), 2, std=1e-2).cuda().contiguous(memory_format=cl)
        self.elems = n * c * h * w
        self.name = ("gn32: GroupNorm(32)+FiLM+SiLU+dropout 0.2, [128,128,32,32] bf16 NHWC, "
                     "fwd+bwd (the residual block's norm2)")

    def fwd(self):
        return self.G.group_norm_silu_film(self.x, self.gamma, self.beta, 32, 1e-5, self.wb, 0.2)

    def step(self):
        self.x.grad = None
        self.fwd().backward(self.dout)


class AttentionWorkload:
    """The attention of cfg5's 16x16 level (diffusion/unet.py:181-203): qkv [128, 256, 768]
    bf16 (4 heads of 64), forward + backward. FLOP: forward 2 GEMMs (q k^T, p v) of
    2 L^2 64 per (image, head); backward 5 (q k^T and dO v^T recomputed, dV, dK, dQ)."""

    def __init__(self):
        self.A = importlib.import_module("diffusion-profiled_amd.attention")
        b, l, c = 128, 256, 256
        g = torch.Generator().manual_seed(5)
        self.qkv = torch.randn((b, l, 3 * c), generator=g).to(torch.bfloat16).cuda().requires_grad_()
        self.dout = (torch.randn((b, l, c), generator=g) * 1e-2).to(torch.bfloat16).cuda()
        self.gemm = 2.0 * b * 4 * l * l * 64
        self.name = "attn256: self-attention, qkv [128,256,768] bf16, 4 heads of 64, fwd+bwd"

    def fwd(self):
        return self.A.self_attention_qkv(self.qkv, 4)

    def step(self):
        self.qkv.grad = None
        self.fwd().backward(self.dout)


def component_main(args):
    """gn32 / attn256: fwd and fwd+bwd device times (HIP events around graph replays)."""
    wl = GroupNormWorkload() if args.workload == "gn32" else AttentionWorkload()
    t_fwd = time_part(wl.fwd, args.kernel_reps)
    t_step = time_part(wl.step, args.kernel_reps)
    t_bwd = t_step - t_fwd
    if args.workload == "gn32":
        kern = {"fwd": {"us": round(t_fwd, 2), "GB/s": round(4 * wl.elems / t_fwd / 1e3, 1)},
                "bwd": {"us": round(t_bwd, 2), "GB/s": round(6 * wl.elems / t_bwd / 1e3, 1)}}
        value, unit = round(10 * wl.elems / t_step / 1e3, 1), "GB/s"
    else:
        kern = {"fwd": {"us": round(t_fwd, 2), "TFLOP/s": round(2 * wl.gemm / t_fwd / 1e6, 1)},
                "bwd": {"us": round(t_bwd, 2), "TFLOP/s": round(5 * wl.gemm / t_bwd / 1e6, 1)}}
        value, unit = round(7 * wl.gemm / t_step / 1e6, 1), "TFLOP/s"
    print(json.dumps({"metric": f"{args.workload} component throughput", "value": value,
                      "unit": unit, "n_gpus": 1, "higher_is_better": True,
                      "ms_per_step": round(t_step / 1e3, 4), "dtype": "bf16 (fp32 statistics)",
                      "data": "synthetic (seeded N(0,1))", "config": {"workload": wl.name},
                      "kernels": kern}), flush=True)


def model_main(args):
    base = {
        "metric": METRIC, "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "scaling": "weak", "vs_baseline": None,
        "dtype": "fp8e4m3 GEMMs (fp32 accumulate), bf16 activations, fp32 master weights",
        "data": "synthetic (seeded images U[-1,1] / N(0,1) activations; random-init weights)",
        "higher_is_better": True,
    }
    if args.workload == "cfg5":
        wl, dt, summ = unet_step_summary(args.steps, args.warmup)
        out = dict(base, value=summ["steps_per_s"], unit="steps/s", ms_per_step=summ["ms_per_step"],
                   config=wl.config(), unet_train_step=summ, roofline=None)
    else:
        wl = ResBlockWorkload()
        g = capture(wl.step, 1)
        dt = time_graph_steps(g.replay, args.steps, args.warmup)
        out = dict(base, value=round(wl.step_flop() / dt / 1e12, 2), unit="TFLOP/s",
                   ms_per_step=round(dt * 1e3, 4), config=wl.config(), roofline=None)
    print(json.dumps(out), flush=True)


def make_workload(K, name):
    if name == "cfg1":
        return GemmWorkload(K)
    if name == "cfg2":
        return ConvWorkload(K, 128, 128, 128, 32, 32, 3, 1, 1,
                            "cfg2: FP8 3x3 conv s1 p1, NHWC [128,32,32,128] -> 128, fwd+dgrad+wgrad incl. e4m3 quantization")
    if name == "cfg3":
        return ConvWorkload(K, 128, 256, 256, 16, 16, 3, 1, 1,
                            "cfg3: FP8 3x3 conv s1 p1, NHWC [128,16,16,256] -> 256, fwd+dgrad+wgrad incl. quantization")
    if name == "cfg3s2":
        return ConvWorkload(K, 128, 256, 256, 16, 16, 3, 2, 1,
                            "cfg3: FP8 3x3 conv stride 2, [128,16,16,256] -> [128,8,8,256], fwd+dgrad+wgrad")
    if name == "cfg3k1":
        return ConvWorkload(K, 128, 128, 256, 32, 32, 1, 1, 0,
                            "cfg3: FP8 1x1 conv 128 -> 256 @ 32x32, fwd+dgrad+wgrad")
    raise ValueError(name)


def capture(fn, reps):
    """A HIP graph (torch.cuda.CUDAGraph) of reps back-to-back calls of fn on a side stream;
    replaying it launches the kernels with no host work in between."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()  # warm: allocator pools, library load
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(reps):
            fn()
    torch.cuda.synchronize()
    return g


def time_part(fn, reps):
    """Average device time per call of fn: HIP events around a graph replay of reps calls,
    recorded on the stream the replay (and so every kernel of this library) runs on."""
    g = capture(fn, reps)
    g.replay()
    torch.cuda.synchronize()
    s = torch.cuda.current_stream()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record(s)
    g.replay()
    end.record(s)
    end.synchronize()
    return start.elapsed_time(end) / reps * 1e3  # microseconds


def host_identity():
    """CPU model name (as lscpu prints it, from /proc/cpuinfo), nproc and os.cpu_count()."""
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    nproc = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else os.cpu_count()
    return {"cpu_model": model, "nproc": nproc, "os_cpu_count": os.cpu_count()}


def host_threads() -> int:
    """Threads for the CPU baseline: every core this process may run on (nproc), capped at
    the 16-core host share a one-GPU box grants a job."""
    return max(1, min(host_identity()["nproc"] or 1, 16))


def cpu_baseline(wl, seconds):
    """The reference recipe on torch CPU (e4m3 round trip, fp32 conv/dgrad/wgrad) on a bounded
    sample of the workload: the first `b` images, b grown until the run takes ~seconds."""
    from oracle import fp8_oracle  # noqa: F401  (the CPU restatement of the recipe)
    import torch.nn.functional as F

    threads = host_threads()
    torch.set_num_threads(threads)

    def q(t):
        t = t.float()
        amax = t.abs().max()
        s = amax / 448.0 if amax > 0 else torch.tensor(1.0)
        return (t / s).clamp(-448, 448).to(torch.float8_e4m3fn).float(), s

    if isinstance(wl, GemmWorkload):
        rows = 1024
        x = wl.x[:rows].cpu()
        w = wl.wt.cpu()
        done = 0
        t0 = time.perf_counter()
        while True:
            xq, xs = q(x)
            wq, ws = q(w)
            _ = ((xq @ wq.T) * (xs * ws)).to(torch.bfloat16)
            done += 1
            if time.perf_counter() - t0 > seconds:
                break
        dt = (time.perf_counter() - t0) / done
        flop = 2.0 * rows * wl.nn * wl.kk
        return {"value": flop / dt / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
                "sample": f"{rows} of {wl.m} rows, {done} reps, {dt * 1e3:.1f} ms/rep",
                "host": host_identity()}
    b = 1
    x = wl.x[:b].cpu().float()
    w = wl.wt.cpu()
    dy = wl.dy[:b].cpu()
    reps = 0
    t0 = time.perf_counter()
    while True:
        xq, xs = q(x)
        wq, ws = q(w)
        dq, ds = q(dy)
        y = (F.conv2d(xq, wq, stride=wl.stride, padding=wl.pad) * (xs * ws)).to(torch.bfloat16)
        dx = (torch.nn.grad.conv2d_input(xq.shape, wq, dq, stride=wl.stride, padding=wl.pad) * (ds * ws)).to(torch.bfloat16)
        dw = (torch.nn.grad.conv2d_weight(xq, wq.shape, dq, stride=wl.stride, padding=wl.pad) * (xs * ds)).to(torch.bfloat16)
        reps += 1
        el = time.perf_counter() - t0
        if el > seconds:
            break
    dt = el / reps
    flop = 3 * wl.flop * b / wl.n
    return {"value": flop / dt / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": "port",
            "sample": f"{b} of {wl.n} images (fwd+dgrad+wgrad incl. e4m3 round trip), {reps} reps, "
                      f"{dt * 1e3:.0f} ms/rep; torch CPU fp32",
            "host": host_identity()}


# ---- time attribution of the halo-patch conv (a stamped copy of the kernel) ----
# Markers in csrc/hconv.hip where the copy records s_memrealtime (100 MHz, device-wide) and
# the shader cycle counter (s_memtime) from lane 0 of every wave: kernel entry, after each
# chunk barrier, before it, around each tile's epilogue. The library itself carries no
# instrumentation.
_HCP_PATCHES = [
    ("namespace dpa {\n",
     "namespace dpa {\n__device__ unsigned long long g_hcp[4096 * 128];\n"
     "#define HCP(slot) do { if ((threadIdx.x & 63) == 0) {"
     " const unsigned long long i_ = (blockIdx.x * 8 + (threadIdx.x >> 6)) * 16 + (slot);"
     " g_hcp[i_] = __builtin_amdgcn_s_memrealtime(); g_hcp[i_ + 8] = __builtin_readcyclecounter(); }"
     " } while (0)\n", "first"),
    ("  const int tid = threadIdx.x;\n  const int lane = tid & 63;\n",
     "  HCP(0);\n  const int tid = threadIdx.x;\n  const int lane = tid & 63;\n", "once"),
    ("    wait_lgkmcnt0();\n    lds_barrier();\n",
     "    if (gc == 1) HCP(3);\n    wait_lgkmcnt0();\n    lds_barrier();\n    if (gc < 2) HCP(1 + gc);\n",
     "once"),
    ("    if (gc - j * p.KC == p.KC - 1) epilogue(cc.m0, cc.n0);\n",
     "    if (gc - j * p.KC == p.KC - 1) { if (gc < 2) HCP(4 + 2 * gc); epilogue(cc.m0, cc.n0);"
     " if (gc < 2) HCP(5 + 2 * gc); }\n", "once"),
]
_HCP_TAIL = """
extern "C" int dpa_hcp_conv(const void* act, const void* wf, const float* sa, const float* sb,
                            void* out, int N, int H, int W, int C, int Cout, int cus, void* s) {
  return dpa::hconv_run(act, wf, sa, sb, nullptr, out, N, H, W, C, Cout, 0, 1, cus,
                        (hipStream_t)s);
}
extern "C" int dpa_hcp_read(void* dst) {
  return (int)hipMemcpyFromSymbol(dst, HIP_SYMBOL(dpa::g_hcp), sizeof(dpa::g_hcp));
}
"""


def hconv_stamped_source(src: str) -> str:
    """csrc/hconv.hip with the stamps in its 256-pixel kernel (the first there)."""
    at = src.index("void hconv_fp8_kernel(")
    end = src.index("\n}\n", at)
    kernel = src[at:end]
    for old, new, mode in _HCP_PATCHES:
        if mode == "first":
            continue
        if kernel.count(old) != 1:
            raise RuntimeError(f"hconv_fp8_kernel no longer has the marker {old.strip()[:50]!r}")
        kernel = kernel.replace(old, new, 1)
    head = src[:at]
    for old, new, mode in _HCP_PATCHES:
        if mode == "first":
            head = head.replace(old, new, 1)
    return head + kernel + src[end:] + _HCP_TAIL


def hconv_phases_main(args):
    """cfg2 forward and data gradient through a stamped copy of the halo-patch conv, each
    graph-replayed; prints the launch time (HIP events) split into the workgroups' phases."""
    import ctypes
    import subprocess
    import tempfile
    import numpy as np

    B = importlib.import_module("diffusion-profiled_amd.build")
    K = importlib.import_module("diffusion-profiled_amd.fp8_kernels")
    src = hconv_stamped_source(open(os.path.join(B.CSRC_DIR, "hconv.hip")).read())
    tmp = tempfile.mkdtemp(prefix="hcp_")
    gen, lib_path = os.path.join(tmp, "hconv_stamped.hip"), os.path.join(tmp, "libhcp.so")
    with open(gen, "w") as f:
        f.write(src)
    cmd = [B.hipcc(), *B.HIPCC_FLAGS, "-shared", f"-I{B.CSRC_DIR}", gen, "-o", lib_path]
    print("building the stamped copy:", " ".join(cmd), flush=True)
    subprocess.run(cmd, check=True, capture_output=True)
    lib = ctypes.CDLL(lib_path)
    cus = torch.cuda.get_device_properties(0).multi_processor_count

    wl = make_workload(K, "cfg2")
    wl.quantize()
    y = torch.empty((wl.n, wl.h, wl.w, wl.cout), device="cuda", dtype=torch.bfloat16)
    dx = torch.empty((wl.n, wl.h, wl.w, wl.cin), device="cuda", dtype=torch.bfloat16)
    calls = {
        "fwd": (wl.xq, wl.wq, wl.xs, wl.ws, y, wl.cin, wl.cout),
        "dgrad": (wl.dyq, wl.wq_t, wl.dys, wl.ws, dx, wl.cout, wl.cin),
    }
    buf = np.zeros(4096 * 128, dtype=np.uint64)
    out = {}
    for name, (a, w, sa, sb, o, c, co) in calls.items():
        def launch():
            st = torch.cuda.current_stream().cuda_stream
            r = lib.dpa_hcp_conv(ctypes.c_void_p(a.data_ptr()), ctypes.c_void_p(w.data_ptr()),
                                 ctypes.c_void_p(sa.data_ptr()), ctypes.c_void_p(sb.data_ptr()),
                                 ctypes.c_void_p(o.data_ptr()), wl.n, wl.h, wl.w, c, co, cus,
                                 ctypes.c_void_p(st))
            assert r == 0, r
        us_launch = time_part(launch, args.kernel_reps)
        # the stamps hold the last launch of the last replay (graph-replayed, as timed)
        assert lib.dpa_hcp_read(ctypes.c_void_p(buf.ctypes.data)) == 0
        grid = (cus // 8) * 8
        raw = buf.reshape(4096, 8, 16)[:grid].astype(np.int64)
        s = raw[:, :, :8] / 100.0                                       # us
        cyc = raw[:, :, 8:]                                             # shader cycles
        w0 = s[:, 0, :]
        t0 = s[:, :, 0].min()
        span = s[:, :, 7].max() - t0
        med = lambda v: round(float(np.median(v)), 2)
        late = s[:, 4:, :]
        early = s[:, :4, :]
        out[name] = {
            "launch_us (HIP events, graph-replayed)": round(us_launch, 2),
            "workgroup span_us (first start to last end)": round(float(span), 2),
            "outside the span (dispatch, end-of-kernel)": round(us_launch - float(span), 2),
            "start skew_us (last workgroup start)": round(float(s[:, 0, 0].max() - t0), 2),
            "prologue_us (first patch, barrier)": med(w0[:, 1] - w0[:, 0]),
            "tile0_us waves 0-3 / 4-7": [med(early[:, :, 4] - early[:, :, 1]),
                                         med(late[:, :, 4] - late[:, :, 1])],
            "epilogue0_us waves 0-3 / 4-7": [med(early[:, :, 5] - early[:, :, 4]),
                                             med(late[:, :, 5] - late[:, :, 4])],
            "chunk-barrier wait_us (wave 0, after its epilogue)": med(w0[:, 2] - w0[:, 5]),
            "tile1_us waves 0-3 / 4-7": [med(early[:, :, 6] - early[:, :, 2]),
                                         med(late[:, :, 6] - late[:, :, 2])],
            "epilogue1_us waves 0-3 / 4-7": [med(early[:, :, 7] - early[:, :, 6]),
                                             med(late[:, :, 7] - late[:, :, 6])],
            "mfma work per tile per SIMD_us at 2.4 GHz": round(2 * 9 * 16 * 32 / 2400.0, 2),
            "shader clock_GHz over the tiles (s_memtime / s_memrealtime)": round(float(np.median(
                (cyc[:, :, 6] - cyc[:, :, 1]) / ((s[:, :, 6] - s[:, :, 1]) * 1e3))), 3),
            "tile0 shader cycles waves 0-3 / 4-7": [int(np.median(cyc[:, :4, 4] - cyc[:, :4, 1])),
                                                    int(np.median(cyc[:, 4:, 4] - cyc[:, 4:, 1]))],
            "mfma cycles per tile per SIMD (2 waves x 144 x 32)": 2 * 9 * 16 * 32,
        }
    print(json.dumps({"hconv_phases": out, "workload": "cfg2", "clock": "s_memrealtime 100 MHz",
                      "medians": "over workgroups (and over the four waves of a group)"}),
          flush=True)


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU only; multi-GPU scaling is not "
                                   "measured; the path would shard by data parallelism, one "
                                   "process per GPU, gradients all-reduced over RCCL",
                          "n_gpus": args.gpus}))
        sys.exit(2)
    K = importlib.import_module("diffusion-profiled_amd.fp8_kernels")
    importlib.import_module("diffusion-profiled_amd._lib").load()
    if args.copy_mib:
        # random bytes: constant fills may be stored compressed and under-report reads
        g = torch.Generator(device="cuda").manual_seed(0)
        src = torch.randint(0, 256, (args.copy_mib << 20,), dtype=torch.uint8, device="cuda",
                            generator=g)
        dst = torch.empty_like(src)
        for _ in range(args.reps):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(f"copied {args.copy_mib} MiB x {args.reps}", flush=True)
        return
    if args.part:
        wl = make_workload(K, args.workload)
        wl.quantize()
        fn = wl.parts()[args.part]
        for _ in range(args.reps):
            fn()
        torch.cuda.synchronize()
        print(f"{args.workload} {args.part} x {args.reps}", flush=True)
        return
    if args.hconv_phases:
        return hconv_phases_main(args)
    if args.workload in ("cfg4", "cfg5"):
        return model_main(args)
    if args.workload in ("gn32", "attn256"):
        return component_main(args)
    wl = make_workload(K, args.workload)

    # per-part device times (HIP events on the launch stream)
    wl.quantize()
    parts = {}
    for name, fn in wl.parts().items():
        parts[name] = time_part(fn, args.kernel_reps)

    # the step as HIP graphs: g holds `per` steps back to back (one replay launches them with
    # no host work and no graph boundary in between, as the conv runs inside a captured
    # training step), g1 one step; exactly args.steps steps are timed (whole g replays, then g1
    # replays for the remainder). The one-step-per-replay time is reported beside it.
    per = max(1, min(args.steps_per_graph, args.steps))
    g = capture(wl.step, per)
    g1 = capture(wl.step, 1)

    def run_steps(k):
        for _ in range(k // per):
            g.replay()
        for _ in range(k % per):
            g1.replay()

    def timed(fn, k):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        fn(k)
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / k

    run_steps(args.warmup)
    dt = timed(run_steps, args.steps)
    dt1 = timed(lambda k: [g1.replay() for _ in range(k)], args.steps)

    tflops = wl.step_flop() / dt / 1e12
    # dominant kernel = the MFMA kernel with the most device time per step: the conv kernel
    # (one fwd and one dgrad launch) or the weight-gradient pair (partial + split reduce)
    names = wl.kernel_names()
    conv_launches = [parts[k] for k in ("fwd", "dgrad") if k in parts]
    if "wgrad" in parts and parts["wgrad"] > sum(conv_launches):
        dominant, dom_us, dom_bytes = names["wgrad"], parts["wgrad"], wl.bytes["wgrad"]
    else:
        dominant = names["fwd"]
        dom_us = sum(conv_launches) / len(conv_launches)
        dom_bytes = sum(wl.bytes[k] for k in ("fwd", "dgrad") if k in parts) / len(conv_launches)
    achieved = wl.flop / (dom_us * 1e-6) / 1e12
    traffic = None
    if os.path.exists(PROFILE_TRAFFIC):
        with open(PROFILE_TRAFFIC) as f:
            traffic = json.load(f).get(args.workload, {}).get(dominant, {}).get("bytes_per_launch")
    # the bound is the roofline the dominant kernel's arithmetic intensity falls under: MFMA
    # above the ridge point (5 PFLOP/s / 8 TB/s = 625 FLOP/B), HBM below it (the K = 256 GEMM
    # of cfg1, the 1x1 convs)
    if wl.flop / dom_bytes >= PEAK_FP8_TFLOPS * 1e12 / (PEAK_HBM_GBS * 1e9):
        roofline = {"bound": "mfma", "kernel": dominant, "achieved": round(achieved, 2),
                    "peak": PEAK_FP8_TFLOPS, "unit": "TFLOP/s",
                    "frac": round(achieved / PEAK_FP8_TFLOPS, 4)}
    else:
        gbs = dom_bytes / (dom_us * 1e-6) / 1e9
        roofline = {"bound": "hbm", "kernel": dominant, "achieved": round(gbs, 1),
                    "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(gbs / PEAK_HBM_GBS, 4),
                    "mfma_frac": round(achieved / PEAK_FP8_TFLOPS, 4)}
    roofline.update({"traffic": traffic, "algorithmic_bytes": dom_bytes,
                     "launch_us": round(dom_us, 2)})
    kernels = {}
    for k, us in parts.items():
        if k == "quantize":
            kernels[k] = {"us": round(us, 2), "GB/s": round(wl.quant_bytes / (us * 1e-6) / 1e9, 1)}
        else:
            kernels[k] = {"us": round(us, 2), "TFLOP/s": round(wl.flop / (us * 1e-6) / 1e12, 1),
                          "frac_fp8_peak": round(wl.flop / (us * 1e-6) / 1e12 / PEAK_FP8_TFLOPS, 4),
                          "kernel": names.get(k, names["fwd"])}
    out = {
        "metric": METRIC,
        "value": round(tflops, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(dt * 1e3, 4),
        "ms_per_step_one_step_graphs": round(dt1 * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp8e4m3 (fp32 accumulate, bf16 out)",
        "data": "synthetic (seeded N(0,1) activations, Kaiming-uniform weights, N(0,1e-2) grad_out)",
        "config": dict(wl.config(), steps_per_graph=per),
        "roofline": roofline,
        "kernels": kernels,
    }
    if args.workload == "cfg2" and not args.no_unet:
        del g, g1
        _, _, out["unet_train_step"] = unet_step_summary(20, 3)
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline(wl, args.cpu_seconds)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
