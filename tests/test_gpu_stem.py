"""The stem layer kernel (convolution, activation, LayerNorm, maximum) against float64 torch on the CPU, at the
edges of its 32 x 16 pixel tiles, odd planes, channel chunks of 4 and 8 with and without a remainder."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W,Ci,Co", [(2, 16, 32, 3, 32), (1, 17, 33, 3, 64), (3, 1, 1, 1, 32), (1, 2, 31, 4, 32),
                                         (2, 15, 16, 32, 32), (1, 33, 65, 8, 64), (1, 34, 7, 11, 32),
                                         (2, 64, 64, 64, 64), (1, 5, 40, 5, 64)])
@pytest.mark.parametrize("act,ln", [("softplus", True), ("gelu", True), ("relu", False), ("none", False)])
def test_stem_layer(N, H, W, Ci, Co, act, ln):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral as S
    print_case(test="stem", N=N, H=H, W=W, Ci=Ci, Co=Co, act=act, ln=ln)
    gen = torch.Generator().manual_seed(H * W + Ci)
    x = torch.randn((N, H, W, Ci), generator=gen) - 0.5
    conv = {"kernel": torch.randn((3, 3, Ci, Co), generator=gen) / (3 * Ci ** 0.5), "bias": torch.randn(Co, generator=gen)}
    norm = {"scale": 1 + 0.3 * torch.randn(Co, generator=gen), "bias": torch.randn(Co, generator=gen)} if ln else None
    F = torch.nn.functional
    r = F.conv2d(x.double().permute(0, 3, 1, 2), conv["kernel"].double().permute(3, 2, 0, 1), conv["bias"].double(),
                 padding=1)
    r = {"softplus": F.softplus, "relu": torch.relu, "none": lambda v: v,
         "gelu": lambda v: F.gelu(v, approximate="tanh")}[act](r).permute(0, 2, 3, 1)
    if ln:
        r = F.layer_norm(r, (Co,), norm["scale"].double(), norm["bias"].double(), eps=1e-6)
    r = F.max_pool2d(r.permute(0, 3, 1, 2), 2, 2, ceil_mode=True).permute(0, 2, 3, 1)
    dev = [{k: v.cuda() for k, v in d.items()} if d is not None else None for d in (conv, norm)]
    xd = x.cuda()
    assert S.stem_conv_supported(xd, *dev)
    y = S.stem_conv(xd, *dev, act).cpu().double()
    assert y.shape == r.shape
    # sums of 9 Ci products in float32 (a few 1e-7 of RMS), divided by a spread of about a third of it
    assert (y - r).abs().max() <= 2e-5 * r.pow(2).mean().sqrt()


def test_stem_layer_spreads_nan_and_takes_offset_vectors():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral as S
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((1, 9, 9, 8), generator=gen, device="cuda")
    x[0, 4, 4, 2] = float("nan")
    conv = {"kernel": torch.randn((3, 3, 8, 32), generator=gen, device="cuda"),
            "bias": torch.randn(33, generator=gen, device="cuda")[1:]}
    y = S.stem_conv(x, conv)
    ref = torch.nn.functional.max_pool2d(
        torch.nn.functional.conv2d(x.cpu().permute(0, 3, 1, 2), conv["kernel"].cpu().permute(3, 2, 0, 1),
                                   conv["bias"].cpu(), padding=1), 2, 2, ceil_mode=True).permute(0, 2, 3, 1)
    assert torch.equal(torch.isnan(y).cpu(), torch.isnan(ref))
    assert (y.cpu() - ref).nan_to_num().abs().max() <= 1e-4
    assert not S.stem_conv_supported(x, {"kernel": torch.zeros((3, 3, 8, 48), device="cuda"),
                                         "bias": torch.zeros(48, device="cuda")}, None)
    assert not S.stem_conv_supported(x, {"kernel": torch.zeros((5, 5, 8, 32), device="cuda"),
                                         "bias": torch.zeros(32, device="cuda")}, None)
