"""The workloads this framework is timed on, through its public entry points.

``listed()`` holds the named cases, ``draw(rng)`` more of the same ranges.  ``prepare`` makes what a program
has in hand before the call (cell or model, weights, inputs), ``run`` is one pass, ``exact`` the same result
in float64 plain torch, ``work`` the bytes and operations a pass cannot do without and ``tolerance`` how far
another correct implementation at the same precision may be from the result.

A case's ``op`` names the entry point:
  gated / gdn              one layer forward: GatedCSSM.apply, GatedDeltaNetCSSM.apply
  block                    one CSSM-SHViT block forward: CSSMSHViTBlock.apply on images
  model                    SimpleCSSM.apply from images to logits
  train_gated / train_gdn  forward and backward of a layer (gated_train_apply, gdn_train_apply): the output and
                           the gradients of the input and of every parameter for a given output gradient
"""
import math

import torch
import torch.nn.functional as Fn

from cssm_amd import blocks, cells, simple_cssm, training


def listed():
    return [
        # a batch of small images through one layer at T = 1: the smallest call, a few launches
        dict(name="gated_image_32", op="gated", B=8, T=1, H=32, C=64, expand=2, K=1, gates="factored", convs=False,
             io="f32", data="normal"),
        # the headline layer: a full batch of large images repeated over time
        dict(name="gated_video_128", op="gated", B=128, T=8, H=128, C=64, expand=1, K=11, gates="factored",
             convs=False, io="f32", data="repeat"),
        # one long video through the layer with the cell's default dense gates and short convolutions
        dict(name="gated_long_16", op="gated", B=1, T=1024, H=16, C=256, expand=1, K=11, gates="dense", convs=True,
             io="f32", data="normal"),
        # the middle stage of an image backbone in bf16: odd planes, many of them, one step
        dict(name="gated_stage_7", op="gated", B=512, T=1, H=7, C=224, expand=2, K=1, gates="factored", convs=False,
             io="bf16", data="normal"),
        # the delta-rule layer on large images with the depthwise qkv convolution
        dict(name="gdn_video_128", op="gdn", B=128, T=8, H=128, C=64, dk=4, K=11, gates="factored", qkv=5, io="f32",
             data="normal"),
        # the delta-rule layer on sparse bf16 video
        dict(name="gdn_video_32", op="gdn", B=128, T=32, H=32, C=64, dk=4, K=11, gates="factored", qkv=1, io="bf16",
             data="dots"),
        # a single small clip through the delta-rule layer with the model's default gates and key dimension
        dict(name="gdn_clip_32", op="gdn", B=1, T=8, H=32, C=32, dk=2, K=11, gates="dense", qkv=1, io="f32",
             data="normal"),
        # one backbone block (norm, position conv, cell with short convs over 8 steps, MLP) on a batch of images
        dict(name="block_14", op="block", B=64, T=8, H=14, C=128, K=15, io="f32", data="normal"),
        # image classification from pixels to logits, the training script's default cell
        dict(name="model_128", op="model", B=64, T=8, H=128, C=32, K=11, gates="dense", io="f32", data="normal"),
        # training step of the headline layer
        dict(name="train_gated_128", op="train_gated", B=16, T=8, H=128, C=64, expand=1, K=11, gates="factored",
             convs=False, io="f32", data="repeat"),
        # training step of the default cell on the feature maps the default stem gives
        dict(name="train_gated_32", op="train_gated", B=32, T=8, H=32, C=64, expand=1, K=11, gates="dense",
             convs=True, io="f32", data="normal"),
        # training step of the delta-rule layer on video
        dict(name="train_gdn_32", op="train_gdn", B=32, T=8, H=32, C=64, dk=4, K=11, gates="factored", qkv=1,
             io="f32", data="normal"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """A case of the listed ranges: planes of 4 x 4 to 128 x 128, 1 to 1024 steps, 2^17 to 2^27 samples in the
    cell (training: to 2^25), every gate type and option the listed cases use."""
    op = rng.choice(["gated", "gated", "gdn", "gdn", "block", "model", "train_gated", "train_gdn"])
    samples = _log_uniform(rng, 2 ** 17, 2 ** 25 if op.startswith("train") else 2 ** 27)
    if op == "block":
        H, C = rng.choice([(14, 128), (7, 224), (4, 320), (16, 64), (13, 96)])
        T = rng.choice([1, 2, 4, 8])
        io = rng.choice(["f32", "bf16"])
        return dict(op=op, B=_batch(samples, T, H, C, 256), T=T, H=H, C=C, K=rng.choice([1, 11, 15]), io=io,
                    data="normal")
    if op == "model":
        H, C, T = rng.choice([32, 64, 128]), rng.choice([32, 64]), rng.choice([4, 8, 12])
        return dict(op=op, B=_batch(samples, T, H // 4, C, 128), T=T, H=H, C=C, K=11,
                    gates=rng.choice(["dense", "factored"]), io="f32", data="normal")
    H = rng.choice([7, 14, 16, 16, 32, 32, 64, 128])
    C = rng.choice([64, 96, 128, 160, 224] if H < 32 else [32, 48, 64])
    if op.endswith("gdn"):
        C = min(C, 128)                               # the widest the output norm takes
    T = int(round(_log_uniform(rng, 2, 24) if op.startswith("train") else _log_uniform(rng, 1, 64)))
    if op == "gated" and H == 16 and rng.random() < 0.5:
        T = int(_log_uniform(rng, 64, 1024))          # a long clip
    gates = rng.choice(["dense", "factored"]) if H < 128 else "factored"
    c = dict(op=op, T=T, H=H, C=C, K=rng.choice([1, 5, 11]), gates=gates, data=rng.choice(["normal", "dots"]),
             io="f32" if op.startswith("train") else rng.choice(["f32", "f32", "bf16"]))
    if op.endswith("gated"):
        c.update(expand=rng.choice([1, 1, 2]), convs=rng.random() < 0.5)
    else:
        c.update(dk=rng.choice([2, 4]), qkv=rng.choice([1, 1, 3, 5]))
    c["B"] = _batch(samples, T, H, C * c.get("expand", 1), 512)
    return c


def _batch(samples, T, H, C, most):
    return max(1, min(most, int(samples / (T * H * H * C))))


# ------------------------------------------------------------------------------------------------- inputs

def _cell(case):
    if case["op"].endswith("gated"):
        return cells.GatedCSSM(channels=case["C"], expand=case["expand"], kernel_size=case["K"],
                               gate_type=case["gates"], short_conv_size=4 if case["convs"] else 0,
                               short_conv_spatial_size=3 if case["convs"] else 0)
    if case["op"].endswith("gdn"):
        return cells.GatedDeltaNetCSSM(channels=case["C"], delta_key_dim=case["dk"], kernel_size=case["K"],
                                       gate_type=case["gates"], qkv_conv_size=case["qkv"])
    if case["op"] == "block":
        return blocks.CSSMSHViTBlock(dim=case["C"], num_timesteps=case["T"], kernel_size=case["K"])
    return simple_cssm.SimpleCSSM(num_classes=2, embed_dim=case["C"], cssm_type="gated", kernel_size=case["K"],
                                  pos_embed="none", seq_len=case["T"], gate_type=case["gates"])


def _randomise(tree, gen, gain=0.0):
    """Trained-like weights: no bias or scale is left at its initial constant, and the input and readout gates
    pass a frame at about unit gain.  (Around zero gain a bin sits on the scan's floor, a step in the gradient.)"""
    for name, v in tree.items():
        if isinstance(v, dict):
            _randomise(v, gen, 1.0 if name.startswith(("B_proj", "C_proj")) else 0.0)
        elif name in ("bias", "scale", "rms_scale"):
            v.add_(gain + 0.1 * torch.randn(v.shape, generator=gen, device=v.device))


def _shape(case):
    B, T, H, C = case["B"], case["T"], case["H"], case["C"]
    if case["op"] == "block":
        return (B, H, H, C)
    if case["op"] == "model":
        return (B, H, H, 3)
    return (B, T, H, H, C)


def _inputs(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    shape, data = _shape(case), case["data"]
    if data == "repeat":                              # one image per clip, repeated over time
        x = torch.randn((shape[0], 1) + shape[2:], generator=gen, device=dev).expand(shape).contiguous()
    elif data == "dots":                              # about 2 % of the pixels lit, moving, over faint noise
        B, T, H, W, C = shape
        x = torch.randn(shape, generator=gen, device=dev) * 0.01
        n = max(1, H * W // 50)
        pos = torch.randint(0, H * W, (B, n), generator=gen, device=dev)
        moves = torch.tensor([0, 1, -1, W, -W], device=dev)
        for t in range(T):
            lit = torch.zeros((B, H * W), dtype=torch.bool, device=dev).scatter_(1, pos, True)
            x[:, t].masked_fill_(lit.view(B, H, W, 1), 1.0)
            pos = (pos + moves[torch.randint(0, 5, (B, n), generator=gen, device=dev)]) % (H * W)
    else:
        x = torch.randn(shape, generator=gen, device=dev)
    if case["io"] == "bf16":
        x = x.bfloat16()
    cell = _cell(case)
    variables = cell.init(seed + 1, shape)
    _randomise(variables["params"], gen)
    dout = torch.randn(shape, generator=gen, device=dev) if case["op"].startswith("train") else None
    return cell, variables, x, dout


def _leaves(tree):
    out = []
    for v in tree.values():
        out += _leaves(v) if isinstance(v, dict) else [v]
    return out


def prepare(case, seed):
    cell, variables, x, dout = _inputs(case, seed)
    state = dict(op=case["op"], cell=cell, variables=variables, x=x)
    if dout is not None:
        leaves = [x] + _leaves(variables["params"])
        for t in leaves:
            t.requires_grad_(True)
        state.update(dout=dout, leaves=leaves)
    return state


def run(state):
    if not state["op"].startswith("train"):
        return state["cell"].apply(state["variables"], state["x"])
    apply = training.gated_train_apply if state["op"] == "train_gated" else training.gdn_train_apply
    out = apply(state["cell"], state["variables"], state["x"])
    return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["dout"])]


# ---------------------------------------------------------------------------------------------------- work

def _cell_flops(frames, H, C, ci, gdn_dk=0):
    """Projections (two operations per multiply-add) and, per plane, a real 2-D transform each way and the
    recurrence's arithmetic per frequency."""
    hw, bins = H * H, H * (H // 2 + 1)
    fft = 2.5 * hw * math.log2(hw)
    if gdn_dk:
        return frames * (2 * hw * C * 5 * C + 4 * C * fft + C * bins * (16 + 24 * gdn_dk))
    return frames * (2 * hw * C * 3 * ci + 2 * ci * fft + ci * bins * 16)


def work(case):
    op, B, T, H, C = case["op"], case["B"], case["T"], case["H"], case["C"]
    io = 2 if case["io"] == "bf16" else 4
    numel = math.prod(_shape(case))
    gdn = op.endswith("gdn")
    Hc = (H + 3) // 4 if op == "model" else H
    ci = C * case.get("expand", 1)
    gate = (Hc * (Hc // 2 + 1)) if case.get("gates") == "dense" else (Hc + Hc // 2 + 1)
    params = 4 * (5 * C * C + 4 * C * gate if gdn else 3 * C * ci + 3 * ci * gate)
    flops = _cell_flops(B * T, Hc, C, ci, case.get("dk", 0))
    if op == "model":
        flops += B * (2 * H * H * 27 * C + 2 * (H // 2) ** 2 * 9 * C * C)
        return {"bytes": numel * io + params + 8 * B, "flops": flops}
    if op == "block":
        flops += B * H * H * 2 * 8 * C * C
        return {"bytes": 2 * numel * io + params + 4 * 8 * C * C, "flops": flops}
    if op.startswith("train"):                        # x, dout -> out, dx; weights and their gradients
        return {"bytes": 4 * numel * io + 2 * params, "flops": 3 * flops}
    return {"bytes": 2 * numel * io + params, "flops": flops}


def tolerance(case):
    """About four times the largest error against ``exact`` over ninety drawn cases (bf16: the rounding of the
    result, and inside a block of the cell's input; training: the parameter whose gradient cancels most)."""
    if case["io"] == "bf16":
        return {"rel": 8e-3}
    return {"rel": 5e-5 if case["op"].startswith("train") else 4e-6}


# --------------------------------------------------------------------------------------------------- exact

def _double(tree):
    return {k: _double(v) if isinstance(v, dict) else v.detach().double() for k, v in tree.items()}


def _dense(x, p):
    return x @ p["kernel"] + p["bias"]


def _floor(z):
    return torch.where(z.real ** 2 + z.imag ** 2 < 1e-14, torch.full_like(z, 1e-7), z)


def _spectral_kernel(k, H, rho=0.999):
    K = k.shape[-1]
    if K > H:
        s = (K - H) // 2
        k = k[:, s:s + H, s:s + H]
    else:
        a = (H - K) // 2
        k = Fn.pad(k, (a, H - K - a, a, H - K - a))
    f = torch.fft.rfft2(k)
    return rho * f / (1.0 + f.abs())


def _depthwise(x, p):
    """SAME depthwise conv of channels-last frames (N, H, W, C)."""
    k, H, W = p["kernel"], x.shape[1], x.shape[2]
    n, lo = k.shape[0], (k.shape[0] - 1) // 2
    xp = Fn.pad(x, (0, 0, lo, n - 1 - lo, lo, n - 1 - lo))
    return sum(xp[:, i:i + H, j:j + W] * k[i, j, 0] for i in range(n) for j in range(n)) + p["bias"]


def _causal(x, p):
    """Causal depthwise conv over time of (B, T, H, W, C)."""
    k, T = p["kernel"], x.shape[1]
    n = k.shape[0]
    xp = Fn.pad(x, (0, 0, 0, 0, 0, 0, n - 1, 0))
    return sum(xp[:, j:j + T] * k[j, 0] for j in range(n)) + p["bias"]


def _planes(x):
    return x.permute(0, 1, 4, 2, 3)


def _gated(p, x, factored, convs):
    """GatedCSSM of (B, T, H, W, C) in float64."""
    B, T, H, W, _ = x.shape
    xz = _dense(x, p["in_proj"])
    xm, z = xz.chunk(2, dim=-1)
    if convs:
        xm = _depthwise(xm.reshape(B * T, H, W, -1), p["short_conv_spatial"]).reshape(xm.shape)
        xm = _causal(xm, p["short_conv_temporal"])
    xm = Fn.silu(xm)
    ctx = xm.mean(dim=(2, 3))

    def gate(name):
        if factored:
            g = _dense(ctx, p[name + "_h"])[..., :, None] * _dense(ctx, p[name + "_w"])[..., None, :]
        else:
            g = _dense(ctx, p[name]).reshape(B, T, H, W // 2 + 1)
        return g[:, :, None]
    d, gb, gc = Fn.softplus(gate("delta_proj")), gate("B_proj"), gate("C_proj")
    V = (d + 1e-8) * _floor(torch.fft.rfft2(_planes(xm)) * gb)
    A = _floor(_spectral_kernel(p["kernel"], H)) * torch.exp(-d)
    h, ys = torch.zeros_like(V[:, 0]), []
    for t in range(T):
        h = A[:, t] * h + V[:, t]
        ys.append(h * gc[:, t])
    y = torch.fft.irfft2(torch.stack(ys, 1), s=(H, W)).permute(0, 1, 3, 4, 2)
    return _dense(y * Fn.silu(z), p["out_proj"])


def _gdn(p, x, factored, dk):
    """GatedDeltaNetCSSM of (B, T, H, W, C) in float64: sinusoid context, RMS norm, SiLU gate."""
    B, T, H, W, C = x.shape
    nh, wf = C // dk, W // 2 + 1
    xq = _depthwise(x.reshape(B * T, H, W, C), p["qkv_dw"]).reshape(x.shape) if "qkv_dw" in p else x
    qkv = _dense(xq, p["qkv_proj"]).chunk(3, dim=-1)
    q, k, v = (Fn.silu(_causal(a, p["short_conv_" + n])) for a, n in zip(qkv, "qkv"))
    freq = 1e4 ** (-torch.arange(0, C, 2, dtype=torch.float64, device=x.device) / C)
    angle = torch.arange(T, dtype=torch.float64, device=x.device)[:, None] * freq
    ctx = x.mean(dim=(2, 3)) + torch.stack([angle.sin(), angle.cos()], -1).reshape(T, C)

    def gate(name, n):
        if factored:
            g = _dense(ctx, p[name + "_h"])[..., :, None] + _dense(ctx, p[name + "_w"])[..., None, :]
        else:
            g = _dense(ctx, p[name]).reshape(B, T, H, n)
        return torch.sigmoid(g)
    k = k * gate("B_k", W)[..., None]
    v = v * gate("B_v", W)[..., None]
    al, be = 0.1 + 0.89 * gate("alpha", wf)[:, :, None], gate("beta", wf)[:, :, None]

    def spectrum(a, unit):
        f = torch.fft.rfft2(_planes(a))
        if unit:
            f = f / torch.sqrt((f.real ** 2 + f.imag ** 2).sum(dim=(3, 4), keepdim=True) + 1e-6)
        return f.reshape(B, T, nh, dk, H, wf)
    q, k, v = spectrum(q, True), spectrum(k, True), spectrum(v, False)
    k = k / torch.sqrt((k.real ** 2 + k.imag ** 2).sum(dim=3, keepdim=True) + 1e-6)
    what = _spectral_kernel(p["kernel"], H)
    eye = torch.eye(dk, dtype=torch.float64, device=x.device)[None, None, :, :, None, None]
    s, outs = 0.0, []                                 # s[b, n, i, r, u, v]: value row i, key row r
    for t in range(T):
        kt, b = k[:, t], be[:, t, :, None, None]
        m = _floor((al[:, t] * what)[:, :, None, None] * (eye - b * kt[:, :, :, None] * kt.conj()[:, :, None]))
        s_in = _floor(b * v[:, t][:, :, :, None] * kt.conj()[:, :, None])
        s = s_in if t == 0 else torch.stack(
            [(m[:, :, r][:, :, None] * s).sum(dim=3) for r in range(dk)], dim=3) + s_in
        outs.append((s * q[:, t][:, :, None]).sum(dim=3))
    o = torch.stack(outs, 1).reshape(B, T, C, H, wf)
    o = torch.fft.irfft2(o, s=(H, W)).permute(0, 1, 3, 4, 2)
    o = o * torch.rsqrt((o * o).mean(dim=-1, keepdim=True) + 1e-6) * p["rms_scale"]
    return _dense(o * Fn.silu(_dense(x, p["gate_proj"])), p["output_proj"])


def _layer_norm(x, p, dims=(-1,)):
    mu = x.mean(dim=dims, keepdim=True)
    var = ((x - mu) ** 2).mean(dim=dims, keepdim=True)
    return (x - mu) * torch.rsqrt(var + 1e-6) * p["scale"] + p["bias"]


def _block(p, x, T):
    """CSSMSHViTBlock (default options) on images (B, H, W, C): the cell's last of T equal frames."""
    h = _layer_norm(x, p["norm1"], (1, 2, 3))
    h = h + _depthwise(h, p["pos_conv"])
    h = x + _gated(p["cssm"], h[:, None].expand(-1, T, -1, -1, -1), True, True)[:, -1]
    m = Fn.gelu(_dense(_layer_norm(h, p["norm2"]), p["mlp"]["fc1"]), approximate="tanh")
    m = m + _depthwise(m, p["mlp"]["dwconv"]["dwconv"])
    return h + _dense(m, p["mlp"]["fc2"])


def _model(p, x, T, factored):
    """SimpleCSSM (default stem and readout) on images (B, H, W, 3)."""
    for i in (1, 2):
        k, H, W = p[f"conv{i}"]["kernel"], x.shape[1], x.shape[2]
        xp = Fn.pad(x, (0, 0, 1, 1, 1, 1))
        x = sum(xp[:, a:a + H, b:b + W] @ k[a, b] for a in range(3) for b in range(3)) + p[f"conv{i}"]["bias"]
        x = _layer_norm(Fn.softplus(x), p[f"norm{i}"])
        x = Fn.max_pool2d(x.permute(0, 3, 1, 2), 2, 2, ceil_mode=True).permute(0, 2, 3, 1)
    x = x[:, None].expand(-1, T, -1, -1, -1)
    x = (x + _gated(p["cssm_0"], x, factored, True))[:, -1]
    x = Fn.softplus(_layer_norm(x, p["norm_pre"])).mean(dim=(1, 2))
    return _dense(_layer_norm(x, p["norm_post"]), p["head"])


def _exact_out(case, p, x):
    factored = case.get("gates", "factored") == "factored"
    if case["op"] == "block":
        return _block(p, x, case["T"])
    if case["op"] == "model":
        return _model(p, x, case["T"], factored)
    if case["op"].endswith("gated"):
        return _gated(p, x, factored, case["convs"])
    return _gdn(p, x, factored, case["dk"])


def exact(case, seed):
    _, variables, x, dout = _inputs(case, seed)
    p = _double(variables["params"])
    train = dout is not None
    leaves = _leaves(p)
    # the batch in pieces of bounded size; weight gradients add up over them
    per = max(1, int(2 ** 24 / (case["T"] * case["H"] ** 2 * case["C"] * case.get("expand", 1))))
    outs, dxs, dps = [], [], [torch.zeros_like(t) for t in leaves]
    if train:
        for t in leaves:
            t.requires_grad_(True)
    for b in range(0, case["B"], per):
        xb = x[b:b + per].detach().double()
        if not train:
            outs.append(_exact_out(case, p, xb))
            continue
        xb.requires_grad_(True)
        y = _exact_out(case, p, xb)
        g = torch.autograd.grad(y, [xb] + leaves, dout[b:b + per].double())
        outs.append(y.detach())
        dxs.append(g[0])
        for acc, gi in zip(dps, g[1:]):
            acc += gi
    out = torch.cat(outs)
    return [out, torch.cat(dxs), *dps] if train else out
