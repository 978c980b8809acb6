"""GPU parity of the gated cell's factored short convolution (cssm_short_conv) against the float64
oracle at the sizes where its plane groups, frame chunks and borders can go wrong."""
import numpy as np
import pytest

from oracle import cssm_oracle as O
from tests.gpu_util import print_case, rel_err, to_np

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral
    return spectral


def reference(x, sp, tp):
    """float64 u and ctx of plane-major x (B, T, C, H, W)."""
    B, T, C, H, W = x.shape
    v = x
    if sp is not None:
        cl = np.moveaxis(v, 2, -1).reshape(B * T, H, W, C)
        v = np.moveaxis(O.depthwise_conv2d_same(cl, sp).reshape(B, T, H, W, C), -1, 2)
    if tp is not None:
        v = np.moveaxis(O.causal_conv_t(np.moveaxis(v, 2, -1), tp), -1, 2)
    u = v / (1.0 + np.exp(-v))
    return u, u.mean(axis=(3, 4))


# (B, T, C, H, W), ks, kt: planes sharing a workgroup with a masked last group, one to four pixels per
# thread, one plane per workgroup, several waves per plane; frames in chunks (few planes, long T); both
# convolutions alone; ks = 5 and kt = 6 take the general kernel
CASES = [((2, 3, 5, 7, 7), 3, 4), ((1, 2, 3, 1, 1), 3, 4), ((3, 1, 7, 4, 4), 3, 4), ((1, 67, 6, 16, 16), 3, 4),
         ((1, 40, 3, 14, 14), 3, 2), ((2, 5, 3, 13, 15), 3, 3), ((1, 9, 2, 17, 17), 3, 4), ((1, 20, 2, 32, 32), 3, 4),
         ((1, 4, 2, 33, 31), 3, 4), ((1, 19, 2, 64, 64), 3, 4), ((1, 9, 1, 128, 128), 3, 4), ((2, 5, 3, 9, 9), 3, 0),
         ((2, 5, 3, 9, 9), 0, 4), ((1, 3, 2, 64, 64), 0, 1), ((2, 5, 3, 9, 9), 5, 4), ((1, 8, 2, 8, 8), 3, 6)]


@pytest.mark.parametrize("shape,ks,kt", CASES)
def test_short_conv(S, shape, ks, kt):
    print_case(test="short_conv", shape=shape, ks=ks, kt=kt)
    rng = np.random.default_rng(sum(shape) + 10 * ks + kt)
    C = shape[2]
    x = rng.standard_normal(shape)
    sp = {"kernel": rng.standard_normal((ks, ks, 1, C)) / 3, "bias": rng.standard_normal(C)} if ks else None
    tp = {"kernel": rng.standard_normal((kt, 1, C)) / 2, "bias": rng.standard_normal(C)} if kt else None

    def dev(p):
        return None if p is None else {k: torch.from_numpy(v).to("cuda", torch.float32) for k, v in p.items()}
    xd = torch.from_numpy(x).to("cuda", torch.float32)
    ref, cref = reference(to_np(xd), sp, tp)
    u, ctx = S.short_conv(xd, dev(sp), dev(tp))
    # at most 25 + 6 products per sum in fp32 (2^-24 each) and a SiLU: far below 1e-5 of RMS
    assert rel_err(to_np(u), ref) <= 1e-5
    assert np.max(np.abs(to_np(ctx) - cref)) <= 1e-5 * np.sqrt(np.mean(ref ** 2))
    ub, _ = S.short_conv(xd.bfloat16(), dev(sp), dev(tp), out_dtype=torch.float32)
    assert rel_err(to_np(ub), reference(to_np(xd.bfloat16()), sp, tp)[0]) <= 1e-5
    assert torch.equal(S.short_conv(xd, dev(sp), dev(tp), out_dtype=torch.bfloat16)[0], u.bfloat16())
