"""The calls whose speed matters here, each as a program that trains with DP-SGD makes it.

A case names its ``kind`` of call, sizes, data type and options:

  linear     a DP Linear's clipped weight gradient (and bias gradient) by wgrad_clip, operand
             a = grad_output [B, T, out], b = input [B, T, in]
  conv1d     the same for the transposed weight of a DP Conv1D: a = input, b = grad_output
  bmm        bmm_clip: clipped sum of per-sample products a_b b_b, fp32 out
  layer      a DPLinear module's forward and backward through autograd
  layernorm  layernorm_fwd, then layernorm_bwd_clip on its statistics
  mlp        a small model wrapped by wrap_with_flashdp_layers under bf16 autocast

Inputs: activations are N(0, 1).  Gradients are N(0, 0.02^2) times a scale of each sample's own,
log-uniform over a factor of 100, and C sits in the middle of the norms that follow, so that some
samples clip and others do not.  Noise is drawn in the kernels with a quarter of the standard
deviation that the gradient's own elements have: its cost does not depend on its scale, and the
gradient can still be checked under it.
"""
import contextlib
import io
import math

import numpy as np
import torch
import torch.nn as nn
import torch.nn.functional as F

from flashdp4review_amd import DPLinear, wrap_with_flashdp_layers
from flashdp4review_amd.core import bmm_clip, layernorm_bwd_clip, layernorm_fwd, wgrad_clip

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
GRAD_RMS = 0.02


def listed():
    return [
        # A small wrapped model under autocast: one training step's forward and backward, where
        # launches and host time are all there is.
        dict(name="mlp_amp_small", kind="mlp", B=4, T=64, I=256, H=512, O=128),
        # The smallest single layer: an fp32 projection over a short batch.
        dict(name="layer_fp32_small", kind="layer", B=4, T=128, I=768, O=768, dtype="fp32", bias=True),
        # [batch, features] inputs (an MLP, a pooled classifier): one row a sample, many samples.
        dict(name="layer_fp32_rows", kind="layer", B=256, T=1, I=1024, O=4096, dtype="fp32", bias=True),
        # The MLP-up layer of a 768-wide decoder in bf16, with bias and noise.
        dict(name="linear_bf16_up", kind="linear", B=8, T=1024, I=768, O=3072, dtype="bf16", out="bf16", bias=True, noise=True),
        # The same layer trained in fp32, as a model that is wrapped without autocast runs it.
        dict(name="linear_fp32_up", kind="linear", B=8, T=1024, I=768, O=3072, dtype="fp32", out="fp32", bias=True, noise=True),
        # The MLP-up layer of a 2048-wide decoder: no bias, the largest layer of a full training step.
        dict(name="linear_bf16_wide", kind="linear", B=8, T=1024, I=2048, O=8192, dtype="bf16", out="bf16", bias=False, noise=True),
        # The attention projection of that decoder under fp16 autocast: fp32 master weights.
        dict(name="linear_fp16_amp", kind="linear", B=8, T=1024, I=2048, O=2048, dtype="fp16", out="fp32", bias=True, noise=True),
        # A vocabulary head that is wrapped too: an odd width, so that no row but the first is aligned.
        dict(name="linear_bf16_vocab", kind="linear", B=4, T=512, I=768, O=50257, dtype="bf16", out="bf16", bias=False, noise=True),
        # The fused QKV Conv1D of a 768-wide decoder.
        dict(name="conv1d_bf16_qkv", kind="conv1d", B=16, T=1024, I=768, O=2304, dtype="bf16", out="bf16", bias=True, noise=True),
        # The per-sample product operator on that layer's tensors.
        dict(name="bmm_bf16_qkv", kind="bmm", B=16, M=768, K=1024, N=2304, dtype="bf16"),
        # LayerNorm of a 1024-wide model in bf16.
        dict(name="layernorm_bf16", kind="layernorm", B=16, T=1024, H=1024, dtype="bf16"),
        # LayerNorm in fp32 over an odd number of odd rows.
        dict(name="layernorm_fp32_odd", kind="layernorm", B=24, T=197, H=1001, dtype="fp32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: mostly a multiple of 64, sometimes of 8, sometimes any number."""
    step = rng.choice((64, 64, 64, 8, 1))
    return max(lo, _log(rng, lo, hi) // step * step)


def draw(rng):
    kind = rng.choice(("mlp", "layer", "layer", "linear", "linear", "linear", "linear", "linear", "conv1d", "bmm",
                       "layernorm", "layernorm"))
    if kind == "mlp":
        return dict(kind=kind, B=_log(rng, 2, 16), T=_log(rng, 16, 256), I=_width(rng, 64, 512),
                    H=_width(rng, 128, 1024), O=_width(rng, 64, 512))
    if kind == "layernorm":
        dtype = rng.choice(("bf16", "fp16", "fp32"))
        c = dict(kind=kind, B=_log(rng, 2, 32), T=_log(rng, 16, 1024), H=_width(rng, 128, 4096), dtype=dtype)
        while c["B"] * c["T"] * c["H"] > 16 * 1024 * 1024:
            c["T"] = c["T"] // 2 + 1
        return c
    if kind == "layer":
        rows = rng.random() < 0.5  # [batch, features] or [batch, tokens, features]
        c = dict(kind=kind, B=_log(rng, 16, 512) if rows else _log(rng, 1, 16), T=1 if rows else _log(rng, 16, 512),
                 I=_width(rng, 64, 4096), O=_width(rng, 64, 4096), dtype=rng.choice(("fp32", "fp32", "bf16")),
                 bias=rng.random() < 0.75)
        limit = 2e9 if rows else 10e9
    elif kind == "bmm":
        c = dict(kind=kind, B=_log(rng, 2, 16), M=_width(rng, 64, 2048), K=_log(rng, 32, 1024), N=_width(rng, 64, 2304),
                 dtype=rng.choice(("bf16", "bf16", "fp16", "fp32")))
        limit = 58e9 if c["dtype"] != "fp32" else 39e9
        while 2.0 * c["B"] * c["M"] * c["K"] * c["N"] > limit:
            c["K"] = c["K"] // 2 + 1
        return c
    else:
        dtype = rng.choice(("bf16", "bf16", "fp16", "fp32")) if kind == "linear" else rng.choice(("bf16", "fp16", "fp32"))
        c = dict(kind=kind, B=_log(rng, 1, 32), T=_log(rng, 16, 1024), I=_width(rng, 128, 2048), O=_width(rng, 128, 8192),
                 dtype=dtype, out=rng.choice((dtype, "fp32")), bias=rng.random() < 0.5, noise=rng.random() < 0.75)
        odd = c["I"] % 8 != 0 or c["O"] % 8 != 0
        limit = 39e9 if dtype == "fp32" else 158e9 if odd else 275e9
    while 2.0 * c["B"] * c["T"] * c["I"] * c["O"] > limit:
        if c["T"] > 64:
            c["T"] = c["T"] // 2 + 1
        else:
            c["B"] = (c["B"] + 1) // 2
            c["O"] = max(64, c["O"] // 128 * 64)
    return c


# ------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _grads(shape, dtype, g):
    """Gradients [B, ...] whose samples' scales spread over a factor of 100."""
    u = torch.rand(shape[0], device="cuda", generator=g) * 2 - 1
    s = (GRAD_RMS * 10.0 ** u).reshape(-1, *([1] * (len(shape) - 1)))
    return (torch.randn(shape, device="cuda", generator=g) * s).to(dtype)


def _sizes(case):
    """B, T, in, out of a layer's case."""
    return case["B"], case["T"], case["I"], case["O"]


def _noise_scale(B, T):
    return 0.25 * GRAD_RMS * math.sqrt(T / B)


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    s = dict(case=case, kind=kind, seed=seed)
    if kind in ("linear", "conv1d"):
        B, T, I, O = _sizes(case)
        dt = DTYPES[case["dtype"]]
        s["x"] = torch.randn(B, T, I, device="cuda", generator=g).to(dt)
        s["g"] = _grads((B, T, O), dt, g)
    elif kind == "bmm":
        B, M, K, N = case["B"], case["M"], case["K"], case["N"]
        dt = DTYPES[case["dtype"]]
        s["a"] = torch.randn(B, M, K, device="cuda", generator=g).to(dt)
        s["b"] = _grads((B, K, N), dt, g)
        s["clip_args"] = torch.tensor([GRAD_RMS * math.sqrt(float(M) * K * N), 1.0], device="cuda")
    elif kind == "layer":
        B, T, I, O = _sizes(case)
        dt = DTYPES[case["dtype"]]
        shape = (B,) if T == 1 else (B, T)
        C = GRAD_RMS * math.sqrt(float(T) * I * O)
        # (no noise: a layer draws other noise at every pass)
        layer = DPLinear(I, O, bias=case["bias"], device="cuda", dtype=dt, C=C, noise_multiplier=0.0)
        with torch.no_grad():
            layer.weight.copy_(torch.randn(O, I, device="cuda", generator=g) * GRAD_RMS)
            if case["bias"]:
                layer.bias.copy_(torch.randn(O, device="cuda", generator=g) * GRAD_RMS)
        s["layer"] = layer
        s["x"] = torch.randn(*shape, I, device="cuda", generator=g).to(dt).requires_grad_(True)
        s["g"] = _grads((*shape, O), dt, g)
    elif kind == "layernorm":
        B, T, H = case["B"], case["T"], case["H"]
        dt = DTYPES[case["dtype"]]
        s["x"] = torch.randn(B, T, H, device="cuda", generator=g).to(dt)
        s["g"] = _grads((B, T, H), dt, g)
        s["w"] = (1 + 0.1 * torch.randn(H, device="cuda", generator=g)).to(dt)
        s["b"] = (0.1 * torch.randn(H, device="cuda", generator=g)).to(dt)
    else:
        I, H, O = case["I"], case["H"], case["O"]
        model = nn.Sequential(nn.Linear(I, H), nn.GELU(), nn.LayerNorm(H), nn.Linear(H, O)).cuda()
        with torch.no_grad():
            for p in model.parameters():
                wide = p.dim() > 1
                p.copy_(torch.randn(p.shape, device="cuda", generator=g) * (p.shape[-1] ** -0.5 if wide else 0.1)
                        + (1.0 if p is model[2].weight else 0.0))
        with contextlib.redirect_stdout(io.StringIO()):
            model = wrap_with_flashdp_layers(model, target_modules=[nn.Linear, nn.LayerNorm], skip_layers=[],
                                             C=_mlp_clip(case), noise_multiplier=0.0, feedback=False) or model
        s["model"] = model
        s["x"] = torch.randn(case["B"], case["T"], I, device="cuda", generator=g)
        s["g"] = _grads((case["B"], case["T"], O), torch.bfloat16, g)
    return s


def _mlp_clip(case):
    return GRAD_RMS * math.sqrt(float(case["T"]) * case["H"] * case["O"])


# ------------------------------------------------------------------------------------- one pass
def run(s):
    case, kind = s["case"], s["kind"]
    if kind in ("linear", "conv1d"):
        B, T, I, O = _sizes(case)
        a, b = (s["g"], s["x"]) if kind == "linear" else (s["x"], s["g"])
        std = _noise_scale(B, T)
        kw = {}
        if case["noise"]:
            kw.update(noise_scale=std, noise_key=(s["seed"], 0))
        db = None
        if case["bias"]:
            db = torch.empty(O, dtype=DTYPES[case["out"]], device="cuda")
            kw.update(bias_out=db, bias_scale=1.0 / (B * T), bias_operand="a" if kind == "linear" else "b")
            if case["noise"]:
                kw.update(bias_noise_scale=std / T, bias_noise_key=(s["seed"], (I * O + 3) // 4))
        dw = wgrad_clip(a, b, GRAD_RMS * math.sqrt(float(T) * I * O), 1.0, out_scale=1.0 / B,
                        out_dtype=DTYPES[case["out"]], **kw)
        return {"dw": dw} if db is None else {"dw": dw, "db": db}
    if kind == "bmm":
        return {"out": bmm_clip(s["a"], s["b"], s["clip_args"])}
    if kind == "layer":
        layer, x = s["layer"], s["x"]
        x.grad = layer.weight.grad = None
        if case["bias"]:
            layer.bias.grad = None
        y = layer(x)
        y.backward(s["g"])
        r = {"y": y.detach(), "dx": x.grad, "dw": layer.weight.grad}
        if case["bias"]:
            r["db"] = layer.bias.grad
        return r
    if kind == "layernorm":
        y, mean, rstd = layernorm_fwd(s["x"], s["w"], s["b"], 1e-5)
        dx, dw, db = layernorm_bwd_clip(s["g"], s["x"], s["w"], mean, rstd, _ln_clip(case), 1.0,
                                        noise_scale=_noise_scale(case["B"], case["T"]), noise_key=(s["seed"], 0))
        return {"y": y, "mean": mean, "rstd": rstd, "dx": dx, "dw": dw, "db": db}
    model = s["model"]
    model.zero_grad(set_to_none=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = model(s["x"])
    logits.backward(s["g"])
    return {"logits": logits.detach(), "grads": {n: p.grad for n, p in model.named_parameters()}}


def _ln_clip(case):
    return GRAD_RMS * math.sqrt(float(case["T"]) * case["H"])


# ------------------------------------------------------------------------------------- its work
def work(case):
    kind = case["kind"]
    size = {"bf16": 2, "fp16": 2, "fp32": 4}
    if kind in ("linear", "conv1d"):
        B, T, I, O = _sizes(case)
        e, o = size[case["dtype"]], size[case["out"]]
        return {"bytes": e * B * T * (I + O) + o * (I * O + (O if case["bias"] else 0)), "flops": 2 * B * T * I * O}
    if kind == "bmm":
        B, M, K, N = case["B"], case["M"], case["K"], case["N"]
        return {"bytes": size[case["dtype"]] * B * K * (M + N) + 4 * M * N, "flops": 2 * B * M * K * N}
    if kind == "layer":
        B, T, I, O = _sizes(case)
        p = I * O + (O if case["bias"] else 0)
        return {"bytes": size[case["dtype"]] * (2 * B * T * (I + O) + 2 * p), "flops": 6 * B * T * I * O}
    if kind == "layernorm":
        n, H = case["B"] * case["T"], case["H"]
        # forward: x in, y out; backward: x and dy in, dx out
        return {"bytes": size[case["dtype"]] * (5 * n * H + 5 * H) + 16 * n, "flops": 20 * n * H}
    n, I, H, O = case["B"] * case["T"], case["I"], case["H"], case["O"]
    p = I * H + H * O + 3 * H + O
    return {"bytes": 4 * n * I + 4 * n * O + 8 * p, "flops": 4 * n * I * H + 6 * n * H * O}


# ------------------------------------------------------------------------------------- checks
def tolerance(case):
    # about four times the largest error against exact() that was measured over these ranges
    kind = case["kind"]
    if kind == "mlp":
        return {"rel": 0.02, "max": 0.2}
    if kind == "bmm" or case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    # 16-bit operands: an output, a sample's product or a partial sum of samples is rounded once
    # to 16 bits on its way
    return {"rel": 0.01, "max": 0.1}


def _philox_normals(n, seed, offset, stream=0):
    """The normals that a noise key (seed, offset) stands for: Philox4x32-10 (Salmon et al., 2011)
    blocks of four words, and two Box-Muller pairs a block."""
    blocks = (n + 3) // 4
    q = np.arange(offset, offset + blocks, dtype=np.uint64)
    low = np.uint64(0xFFFFFFFF)
    half = np.uint64(32)
    w = [q & low, q >> half, np.full_like(q, stream), np.zeros_like(q)]
    key = [seed & 0xFFFFFFFF, seed >> 32 & 0xFFFFFFFF]
    for _ in range(10):
        p, r = w[0] * np.uint64(0xD2511F53), w[2] * np.uint64(0xCD9E8D57)
        w = [(r >> half) ^ w[1] ^ np.uint64(key[0]), r & low, (p >> half) ^ w[3] ^ np.uint64(key[1]), p & low]
        key = [(key[0] + 0x9E3779B9) & 0xFFFFFFFF, (key[1] + 0xBB67AE85) & 0xFFFFFFFF]
    z = np.empty((blocks, 4))
    for i in (0, 2):
        radius = np.sqrt(-2 * np.log((w[i].astype(np.float64) + 0.5) / 2.0 ** 32))
        angle = 2 * np.pi * ((w[i + 1] >> np.uint64(8)).astype(np.float64) + 0.5) / 2.0 ** 24
        z[:, i], z[:, i + 1] = radius * np.cos(angle), radius * np.sin(angle)
    return torch.from_numpy(z.reshape(-1)[:n]).cuda()


def _clip(norm, C):
    return (C / (norm + 1e-10)).clamp(max=1.0)


def _clipped_products(a, b, C, tn=True):
    """sum_b clip(||G_b||) G_b in 64 bits, one sample at a time."""
    total = 0
    for i in range(a.shape[0]):
        left = a[i].double()
        G = (left.t().contiguous() if tn else left) @ b[i].double()
        total = total + G * _clip(G.norm(), C)
    return total


def _clipped_bias(g, C):
    """(1 / (B T)) sum_b clip(||g_b||) sum_t g_bt in 64 bits."""
    g = g.double()
    c = _clip(g.flatten(1).norm(dim=1), C)
    return (c[:, None] * g.sum(1)).sum(0) / (g.shape[0] * g.shape[1])


def _layernorm_grads(g, xhat, C):
    """The clipped means over samples of sum_t g xhat and of sum_t g."""
    r = []
    for v in ((g * xhat).sum(1), g.sum(1)):
        r.append((_clip(v.norm(dim=1), C)[:, None] * v).mean(0))
    return r


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("linear", "conv1d"):
        B, T, I, O = _sizes(case)
        a, b = (s["g"], s["x"]) if kind == "linear" else (s["x"], s["g"])
        C, std = GRAD_RMS * math.sqrt(float(T) * I * O), _noise_scale(B, T)
        r = {"dw": _clipped_products(a, b, C) / B}
        if case["noise"]:
            r["dw"] += std * _philox_normals(I * O, seed, 0).reshape(r["dw"].shape)
        if case["bias"]:
            r["db"] = _clipped_bias(s["g"], C)
            if case["noise"]:
                r["db"] += std / T * _philox_normals(O, seed, (I * O + 3) // 4)
        return r
    if kind == "bmm":
        return {"out": _clipped_products(s["a"], s["b"], float(s["clip_args"][0]), tn=False)}
    if kind == "layer":
        B, T, I, O = _sizes(case)
        layer, x, g = s["layer"], s["x"].detach().double().reshape(B, T, I), s["g"].double().reshape(B, T, O)
        w = layer.weight.detach().double()
        y = x.reshape(-1, I) @ w.t() + (layer.bias.detach().double() if case["bias"] else 0)
        r = {"y": y.reshape(*s["g"].shape), "dx": (g.reshape(-1, O) @ w).reshape(s["x"].shape),
             "dw": _clipped_products(g, x, layer.C) / B}
        if case["bias"]:
            r["db"] = _clipped_bias(g, layer.C)
        return r
    if kind == "layernorm":
        H = case["H"]
        x, g, w, b = (s[k].double() for k in ("x", "g", "w", "b"))
        mean, var = x.mean(-1), x.var(-1, unbiased=False)
        rstd = (var + 1e-5).rsqrt()
        xhat = (x - mean[..., None]) * rstd[..., None]
        wg = w * g
        dx = rstd[..., None] * (wg - wg.mean(-1, keepdim=True) - xhat * (wg * xhat).mean(-1, keepdim=True))
        dw, db = _layernorm_grads(g, xhat, _ln_clip(case))
        std = _noise_scale(case["B"], case["T"])
        return {"y": xhat * w + b, "mean": mean.reshape(-1), "rstd": rstd.reshape(-1), "dx": dx,
                "dw": dw + std * _philox_normals(H, seed, 0, 0), "db": db + std * _philox_normals(H, seed, 0, 1)}
    # the model: its forward in 64 bits, and each layer's clipped sums from the gradients there
    p = {n: q.detach().double() for n, q in s["model"].named_parameters()}
    B, T, H, C = case["B"], case["T"], case["H"], _mlp_clip(case)
    x = s["x"].double()
    first = (x @ p["0.weight"].t() + p["0.bias"]).requires_grad_(True)
    h = F.gelu(first)
    mid = F.layer_norm(h, (H,))
    normed = mid * p["2.weight"] + p["2.bias"]
    logits = normed @ p["3.weight"].t() + p["3.bias"]
    g_out = s["g"].double()
    g_first, g_normed = torch.autograd.grad(logits, (first, normed), g_out)
    dw, db = _layernorm_grads(g_normed, mid.detach(), C)
    grads = {"0.weight": _clipped_products(g_first, x, C) / B, "0.bias": _clipped_bias(g_first, C),
             "2.weight": dw, "2.bias": db,
             "3.weight": _clipped_products(g_out, normed.detach(), C) / B, "3.bias": _clipped_bias(g_out, C)}
    return {"logits": logits.detach(), "grads": grads}
