"""The gated cell's training kernels (short-convolution adjoint, spectral-kernel adjoint, depthwise-conv weight
gradient) against float64 autograd at the edges of their plane groups, frame chunks and strips, and the whole
layer with short convolutions on small and power-of-two planes."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
Fn = torch.nn.functional


@pytest.fixture(scope="module")
def S():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral
    return spectral


def close(got, ref, tol=2e-5):
    """fp32 sums of up to a few hundred thousand O(1) products against float64 (rounding near 1e-6 of the
    largest value; tol leaves an order of magnitude)."""
    assert got.shape == ref.shape
    assert (got.double() - ref).abs().max() <= tol * max(1e-30, ref.abs().max().item())


def randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda")


CASES = [((2, 3, 5, 7, 7), 3, 4), ((1, 2, 3, 1, 1), 3, 4), ((3, 1, 7, 4, 4), 3, 4), ((1, 37, 6, 16, 16), 3, 4),
         ((1, 20, 3, 14, 14), 3, 2), ((2, 5, 3, 13, 15), 3, 3), ((1, 9, 2, 17, 17), 3, 4), ((1, 20, 2, 32, 32), 3, 4),
         ((1, 4, 2, 33, 31), 3, 4), ((1, 19, 2, 64, 64), 3, 4), ((1, 9, 1, 128, 128), 3, 4), ((2, 5, 3, 9, 9), 3, 0),
         ((2, 5, 3, 9, 9), 0, 4), ((1, 3, 2, 64, 64), 0, 1), ((1, 3, 2, 128, 128), 0, 2)]


@pytest.mark.parametrize("shape,ks,kt", CASES)
def test_short_conv_adjoint(S, shape, ks, kt):
    print_case(test="short_conv_adjoint", shape=shape, ks=ks, kt=kt)
    B, T, C, H, W = shape
    gen = torch.Generator(device="cuda").manual_seed(sum(shape) + 10 * ks + kt)
    x, do = randn(gen, *shape), randn(gen, *shape)
    sp = (randn(gen, ks, ks, 1, C) / 3, randn(gen, C)) if ks else None
    tp = (randn(gen, kt, 1, C) / 2, randn(gen, C)) if kt else None
    assert S.short_conv_train_supported(T, H, W, ks, kt)
    wide = torch.zeros((B * T, 2 * C, H * W), device="cuda")
    o, ctx = S.short_conv_train(x, sp, tp)
    sums = S.short_conv_backward(x, do, sp, tp, wide[:, :C])
    leaves = [t.double().requires_grad_(True) for t in (x, *(sp or ()), *(tp or ()))]
    v, rest = leaves[0], leaves[1:]
    if ks:
        v = (Fn.conv2d(v.reshape(B * T, C, H, W), rest[0].permute(3, 2, 0, 1), padding=1, groups=C)
             + rest[1][:, None, None]).view(shape)
    if kt:
        w, b = rest[-2:]
        pad = torch.cat([v.new_zeros(B, kt - 1, C, H, W), v], dim=1)
        v = sum(pad[:, j:j + T] * w[j, 0][:, None, None] for j in range(kt)) + b[:, None, None]
    grads = torch.autograd.grad(v, leaves, do.double())
    close(o, v.detach())
    close(ctx, Fn.silu(v.detach()).mean(dim=(3, 4)))
    close(wide[:, :C].reshape(shape), grads[0])
    assert not wide[:, C:].any()
    if ks:
        close(sums[:, :9].t().reshape(ks, ks, 1, C), grads[1])
        close(sums[:, 9], grads[2])
    if kt:
        close(sums[:, 10:10 + kt].flip(1).t().reshape(kt, 1, C), grads[-2])
        close(sums[:, 14], grads[-1])
    close(sums[:, 15], grads[0].sum(dim=(0, 1, 3, 4)), 1e-4)       # cancels


# taps inside the plane, as wide as it, cropped; one bin column; even and odd planes; the scan's orders at 128
@pytest.mark.parametrize("C,K,H", [(3, 5, 16), (2, 1, 7), (3, 7, 7), (2, 11, 9), (2, 15, 4), (3, 14, 9), (2, 11, 128), (70, 3, 14)])
@pytest.mark.parametrize("squash,floor,order", [(True, True, True), (True, False, False), (False, False, False)])
def test_spectral_kernel_adjoint(S, C, K, H, squash, floor, order):
    from cssm_amd import training
    print_case(test="spectral_kernel_adjoint", C=C, K=K, H=H, squash=squash, floor=floor)
    gen = torch.Generator(device="cuda").manual_seed(C * K + H)
    k = 0.3 * randn(gen, C, K, K)
    k[0] = 0.0                                             # a floored channel
    B, Wf = 3, H // 2 + 1
    d = torch.complex(randn(gen, B, C, H, Wf), randn(gen, B, C, H, Wf))
    assert S.spectral_kernel_bwd_supported(C, K, H, H)
    dk = S.spectral_kernel_backward(k, d, H, 0.999, squash, floor, order)
    kd = k.double().requires_grad_(True)
    if order:
        ref = training.khat_planes(kd, H, H, 0.999)
    else:
        ref = training.what_planes(kd, H, H, 0.999, squash)
    if squash:                                             # |F| has no gradient at 0: the zero channel apart
        g = torch.autograd.grad(ref[1:], kd, d.sum(dim=0)[1:].to(torch.complex128))[0]
        close(dk[1:], g[1:])
        if floor:
            assert not dk[0].any()
    else:
        close(dk, torch.autograd.grad(ref, kd, d.sum(dim=0).to(torch.complex128))[0])


@pytest.mark.parametrize("ks,shape", [(3, (2, 7, 7, 12)), (5, (3, 14, 14, 128)), (7, (2, 5, 9, 36)), (5, (1, 9, 17, 96)),
                                      (3, (2, 3, 1, 4)), (3, (1, 4, 20, 260))])
def test_depthwise_wgrad_on_any_row(S, ks, shape):
    """Rows that are no multiple of eight pixels and channel quads that do not divide a wave."""
    print_case(test="dw_wgrad", ks=ks, shape=shape)
    gen = torch.Generator(device="cuda").manual_seed(ks)
    F, H, W, C = shape
    x, dy = randn(gen, *shape), randn(gen, *shape)
    got = S.depthwise_conv_wgrad(x, dy, ks)
    w = torch.zeros((C, 1, ks, ks), dtype=torch.float64, device="cuda", requires_grad=True)
    y = Fn.conv2d(x.double().permute(0, 3, 1, 2), w, padding=ks // 2, groups=C)
    (ref,) = torch.autograd.grad(y, w, dy.double().permute(0, 3, 1, 2))
    close(got, ref.permute(2, 3, 1, 0))


@pytest.mark.parametrize("shape,gate_type,convs", [((2, 3, 7, 7, 6), "factored", (3, 4)), ((1, 4, 16, 16, 8), "dense", (3, 4)),
                                                   ((2, 2, 14, 14, 5), "dense", (0, 3)), ((1, 5, 13, 13, 4), "factored", (3, 0)),
                                                   ((1, 2, 32, 32, 4), "factored", (3, 4)), ((2, 3, 9, 9, 4), "dense", (0, 0))])
def test_layer_gradients_with_short_convs(S, shape, gate_type, convs):
    """gated_train_apply against float64 autograd of the layer (gates at about unit gain, away from the floor)."""
    from cssm_amd import cells, training
    from oracle import cssm_cpu_fp32 as P
    print_case(test="gated_layer_grad", shape=shape, gates=gate_type, convs=convs)
    B, T, H, W, C = shape
    cell = cells.GatedCSSM(channels=C, kernel_size=5, gate_type=gate_type, short_conv_spatial_size=convs[0],
                           short_conv_size=convs[1])
    var = cell.init(3, shape)
    gen = torch.Generator(device="cuda").manual_seed(5)
    for n, sub in var["params"].items():
        if isinstance(sub, dict):
            sub["bias"].add_(0.1 * randn(gen, *sub["bias"].shape) + (1.0 if n.startswith(("B_", "C_")) else 0.0))
    x, dout = randn(gen, *shape), randn(gen, *shape)

    def leaves(tree):
        return [t for v in tree.values() for t in (leaves(v) if isinstance(v, dict) else [v])]

    def double(tree):
        return {k: double(v) if isinstance(v, dict) else v.detach().cpu().double().numpy() for k, v in tree.items()}
    ref_m = P.GatedCPU(double(var["params"]), C, kernel_size=5, gate_type=gate_type, short_conv_size=convs[1],
                       short_conv_spatial_size=convs[0], dtype=torch.float64, requires_grad=True)
    xr = x.cpu().double().requires_grad_(True)
    yr = ref_m(xr)
    refs = torch.autograd.grad(yr, [xr] + leaves(ref_m.p), dout.cpu().double())
    ls = [x.requires_grad_(True)] + [t.requires_grad_(True) for t in leaves(var["params"])]
    y = training.gated_train_apply(cell, var, x)
    grads = torch.autograd.grad(y, ls, dout)
    close(y.detach().cpu(), yr.detach())
    for g, r in zip(grads, refs):
        close(g.cpu(), r, 2e-4)
