"""GPU parity of the fused activation + per-row LayerNorm (cssm_layer_norm) against float64."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
Fn = torch.nn.functional
ACTS = {"none": lambda v: v, "gelu": lambda v: Fn.gelu(v, approximate="tanh"), "relu": torch.relu,
        "softplus": Fn.softplus}


@pytest.fixture(scope="module")
def S():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral
    return spectral


# channel counts over the lanes-per-row and vectors-per-lane choices, C % 4 != 0 and a row count that
# leaves the last workgroup partial; offset 1: pointers off a 16-byte boundary (element accesses)
@pytest.mark.parametrize("C,offset", [(1, 0), (3, 0), (4, 0), (12, 0), (32, 0), (36, 1), (130, 0), (320, 0), (511, 0),
                                      (512, 1), (2048, 0)])
@pytest.mark.parametrize("pre,post", [("none", "none"), ("softplus", "none"), ("none", "softplus"), ("relu", "gelu")])
def test_layer_norm(S, C, offset, pre, post):
    print_case(test="layer_norm", C=C, offset=offset, pre=pre, post=post)
    gen = torch.Generator(device="cuda").manual_seed(C)
    M = 77
    x = (1.0 + 2.0 * torch.randn(M * C + offset, generator=gen, device="cuda"))[offset:].view(M, C)
    sc = 1.0 + 0.3 * torch.randn(C, generator=gen, device="cuda")
    bi = 0.3 * torch.randn(C, generator=gen, device="cuda")

    def ref(v):
        v = ACTS[pre](v.double())
        mu = v.mean(dim=1, keepdim=True)
        var = ((v - mu) ** 2).mean(dim=1, keepdim=True)
        return ACTS[post]((v - mu) * torch.rsqrt(var + 1e-6) * sc.double() + bi.double())
    # a row of one channel (or a relu row of equal values) has variance 0: the difference x - mean is
    # exact there and the result the bias; else fp32 rounding of x - mean (a few ulp of |x| ~ 1..10) over
    # a standard deviation of ~0.5 and up
    got = S.layer_norm(x, sc, bi, pre=pre, post=post)
    assert (got.double() - ref(x)).abs().max() <= 2e-5 * max(1.0, ref(x).abs().max().item())
    xb = x.bfloat16()
    gb = S.layer_norm(xb, sc, bi, pre=pre, post=post)
    # one bf16 rounding of the result
    assert ((gb.double() - ref(xb)).abs() <= 2.0 ** -8 * ref(xb).abs() + 2e-4).all()
    if pre == post == "none":
        x5 = x.reshape(M, 1, 1, 1, C)
        two = S.block_norm_posconv(x5, S.block_norm_stats(x5, "layer"), "layer", sc, bi, None, None, 1)
        assert (got - two.reshape(M, C)).abs().max() <= 1e-6 * max(1.0, two.abs().max().item())
