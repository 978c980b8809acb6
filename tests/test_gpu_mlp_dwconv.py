"""The block MLP's gelu + depthwise convolution kernel against float64 torch on the CPU, at the edges of its row tiles:
one tile without halo rows (H W <= 512), tiles with them, a remainder row, single rows and columns."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W,C", [(2, 14, 14, 64), (1, 1, 1, 32), (3, 7, 7, 96), (1, 8, 64, 32), (2, 9, 64, 32),
                                     (1, 25, 61, 32), (1, 40, 1, 32), (1, 1, 40, 64), (2, 22, 23, 32), (1, 23, 23, 32)])
def test_mlp_dwconv(N, H, W, C):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral as S
    print_case(test="mlp_dwconv", N=N, H=H, W=W, C=C)
    gen = torch.Generator().manual_seed(H * W)
    x, k, b = (torch.randn(s, generator=gen) for s in ((N, H, W, C), (3, 3, 1, C), (C,)))
    F = torch.nn.functional
    g = F.gelu(x.double(), approximate="tanh").permute(0, 3, 1, 2)
    r = (g + F.conv2d(g, k.double().permute(3, 2, 0, 1), b.double(), padding=1, groups=C)).permute(0, 2, 3, 1)
    xd, kd, bd = x.cuda(), k.cuda(), b.cuda()
    assert S.mlp_dwconv_supported(xd, kd, bd)
    y = S.mlp_dwconv(xd, kd, bd).cpu().double()
    # nine products, a gelu of a few units in the last place: under 1e-6 of RMS per term
    assert (y - r).abs().max() <= 5e-6 * r.pow(2).mean().sqrt()


def test_mlp_dwconv_refuses():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral as S
    z = lambda *s: torch.zeros(s, device="cuda")
    assert not S.mlp_dwconv_supported(z(1, 4, 4, 48), z(3, 3, 1, 48), z(48))
    assert not S.mlp_dwconv_supported(z(1, 4, 65, 32), z(3, 3, 1, 32), z(32))
    assert not S.mlp_dwconv_supported(z(1, 4, 4, 32), z(3, 3, 1, 32), z(33)[1:])
