"""The GDN training kernels (cssm_gdn_qkv_act, cssm_gdn_norm_gate, the spectral core with its norms) and
their adjoints against float64 autograd at the edges of their channel, pixel and frame groups."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral
    return spectral


def close(got, ref, tol=2e-5):
    """fp32 kernels against float64: sums of at most a few hundred thousand products of O(1) terms, whose
    rounding stays near 1e-6 of the largest term; tol leaves an order of magnitude."""
    assert got.shape == ref.shape
    assert (got.double() - ref).abs().max() <= tol * max(1e-30, ref.abs().max().item())


def randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


# C around the 8-channel groups, planes of element and vector access, pixel groups masked and several per
# wave (128 x 128 of many batch elements), frames fewer than taps
CASES = [(2, 5, 8, 8, 4, 1), (1, 1, 5, 7, 4, 1), (2, 2, 9, 7, 3, 2), (1, 3, 3, 5, 1, 3), (1, 9, 12, 16, 8, 0),
         (2, 4, 7, 14, 0, 1), (1, 2, 17, 10, 2, 3), (3, 3, 64, 128, 4, 1), (1, 4, 2, 3, 4, 2)]


@pytest.mark.parametrize("B,T,C,H,kt,mode", CASES)
@pytest.mark.parametrize("wide", [False, True])
def test_qkv_act_and_adjoint(S, B, T, C, H, kt, mode, wide):
    print_case(test="qkv_act", B=B, T=T, C=C, H=H, kt=kt, mode=mode, wide=wide)
    gen = torch.Generator(device="cuda").manual_seed(C * H + kt)
    F, HW = B * T, H * H
    n = 4 * C if wide else 3 * C
    raw = randn(gen, F, n, HW)[:, :3 * C]
    convs = [randn(gen, kt, 1, C) if i % 2 == 0 else randn(gen, C) for i in range(6)] if kt else []
    gshape = {0: None, 1: (2, F, HW), 2: (2, F), 3: (F, 2 * C, HW)}[mode]
    gates = torch.rand(gshape, generator=gen, device="cuda") if mode else None
    dout = randn(gen, F, 3 * C, HW)
    draw = torch.zeros((F, n, HW), device="cuda")[:, :3 * C]
    out = S.gdn_qkv_act(raw, B, T, convs, mode, gates)
    dgates, sums = S.gdn_qkv_act_backward(raw, B, T, convs, mode, gates, dout, draw)

    leaves = [t.double().requires_grad_(True) for t in (raw, *convs, *([gates] if mode else []))]
    x = leaves[0].view(B, T, 3, C, HW)
    cs, g = leaves[1:1 + len(convs)], leaves[-1] if mode else None
    parts = []
    for i in range(3):
        v = x[:, :, i]
        if kt:
            pad = torch.cat([v.new_zeros(B, kt - 1, C, HW), v], dim=1)
            v = sum(pad[:, j:j + T] * cs[2 * i][j, 0][:, None] for j in range(kt)) + cs[2 * i + 1][:, None]
            v = torch.nn.functional.silu(v)
        if i and mode:
            gi = (g[i - 1].view(B, T, 1, -1) if mode < 3 else g.view(B, T, 2, C, HW)[:, :, i - 1])
            v = v * gi
        parts.append(v)
    ref = torch.stack(parts, 2).reshape(F, 3 * C, HW)
    grads = torch.autograd.grad(ref, leaves, dout.double())
    close(out, ref.detach())
    close(draw, grads[0])
    close(sums[:, kt + 1], grads[0].sum(dim=(0, 2)), 1e-4)      # cancels: a sum of mixed signs
    for i in range(3 if kt else 0):
        close(sums[i * C:(i + 1) * C, :kt].t().unsqueeze(1), grads[1 + 2 * i], 1e-4)
        close(sums[i * C:(i + 1) * C, kt], grads[2 + 2 * i], 1e-4)
    if mode:
        close(dgates, grads[-1], 1e-4)


@pytest.mark.parametrize("F,C,H", [(3, 1, 7), (2, 5, 5), (4, 32, 8), (3, 33, 6), (2, 64, 32), (2, 65, 3), (1, 128, 9)])
@pytest.mark.parametrize("norm", ["none", "rms", "layer"])
@pytest.mark.parametrize("act", ["silu", "sigmoid"])
def test_norm_gate_and_adjoint(S, F, C, H, norm, act):
    print_case(test="norm_gate", F=F, C=C, H=H, norm=norm, act=act)
    if C == 1 and norm == "layer":
        pytest.skip("one channel: variance 0, the gradient is a difference of equal terms")
    gen = torch.Generator(device="cuda").manual_seed(C + H)
    HW = H * H
    o, dy = 0.7 + randn(gen, F, C, HW), randn(gen, F, C, HW)
    g = randn(gen, F, 4 * C, HW)[:, 3 * C:]
    scale = 1 + 0.2 * randn(gen, C) if norm != "none" else None
    shift = 0.3 * randn(gen, C) if norm == "layer" else None
    dg = torch.zeros((F, 2 * C, HW), device="cuda")[:, C:]
    y = S.gdn_norm_gate(o, g, norm, scale, shift, act)
    do, sums = S.gdn_norm_gate_backward(o, g, norm, scale, shift, act, dy, dg)
    leaves = [t.double().requires_grad_(True) for t in (o, g)]
    ps = [t.double().requires_grad_(True) for t in (scale, shift) if t is not None]
    v = leaves[0]
    if norm == "rms":
        v = v * torch.rsqrt((v * v).mean(dim=1, keepdim=True) + 1e-6) * ps[0][:, None]
    elif norm == "layer":
        mu = v.mean(dim=1, keepdim=True)
        v = ((v - mu) * torch.rsqrt(((v - mu) ** 2).mean(dim=1, keepdim=True) + 1e-6) * ps[0][:, None]
             + ps[1][:, None])
    s = torch.sigmoid(leaves[1])
    ref = v * (leaves[1] * s if act == "silu" else s)
    grads = torch.autograd.grad(ref, leaves + ps, dy.double())
    close(y, ref.detach())
    close(do, grads[0], 1e-4)
    close(dg, grads[1])
    close(sums[2], grads[1].sum(dim=(0, 2)), 1e-4)
    for i, r in enumerate(grads[2:]):
        close(sums[i], r, 1e-4)


@pytest.mark.parametrize("dk,H,W,T", [(4, 16, 16, 3), (2, 7, 7, 1), (1, 8, 8, 4), (3, 14, 14, 2)])
@pytest.mark.parametrize("l2", [False, True])
def test_core_adjoint_includes_norms_and_transforms(S, dk, H, W, T, l2):
    """gdn_core_train / gdn_core_backward between rfft2 and irfft2 against float64 autograd from the planes."""
    from oracle.cssm_cpu_fp32 import gdn_bins_core
    print_case(test="gdn_core_adjoint", dk=dk, H=H, T=T, l2=l2)
    gen = torch.Generator().manual_seed(dk * H)
    B, C, Wf = 2, 2 * dk, W // 2 + 1
    qkv = torch.randn((B, T, 3 * C, H, W), generator=gen, dtype=torch.float64)
    ab = torch.rand((B, T, H * Wf, 2), generator=gen, dtype=torch.float64)
    what = torch.randn((C // dk, H, Wf), generator=gen, dtype=torch.complex128) * 0.5
    dy = torch.randn((B, T, C, H, W), generator=gen, dtype=torch.float64)
    leaves = [t.requires_grad_(True) for t in (qkv, ab, what)]
    spec = torch.fft.rfft2(qkv)
    if l2:
        qk = spec[:, :, :2 * C]
        qk = qk * torch.rsqrt((qk.real ** 2 + qk.imag ** 2).sum(dim=(3, 4), keepdim=True) + 1e-6)
        spec = torch.cat([qk, spec[:, :, 2 * C:]], dim=2)
    ref = torch.fft.irfft2(gdn_bins_core(spec, ab, what, "dense", dk), s=(H, W))
    refs = torch.autograd.grad(ref, leaves, dy)
    d = [t.detach().to("cuda", torch.complex64 if t.is_complex() else torch.float32) for t in leaves]
    sp, norms = S.rfft2(d[0], want_norms=l2)
    ohat, states = S.gdn_core_train(sp, norms, d[1], "dense", d[2], dk, W)
    dos, _ = S.rfft2(dy.to("cuda", torch.float32))
    dspec, dab, dwhat = S.gdn_core_backward(sp, norms, d[1], "dense", d[2], states, dos, dk, W)
    close(S.irfft2(ohat, W).cpu(), ref.detach())
    close(S.irfft2(dspec, W).cpu(), refs[0], 1e-4)
    close(dab.sum(dim=2).cpu(), refs[1], 1e-4)
    close(torch.view_as_real(dwhat.sum(dim=0).cpu()), torch.view_as_real(refs[2]), 1e-4)
