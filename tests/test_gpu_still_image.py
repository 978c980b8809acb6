"""An image repeated over time with only the last frame kept: the cell's one-frame path against the last
frame of the cell on the repeated frames, at plane sizes of every kernel and around the convolution's taps."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# T below, at and above the four taps; ragged plane groups (C, B) of the small-plane kernel; 128: column order
@pytest.mark.parametrize("B,T,C,H,kt,ks", [(2, 8, 24, 14, 4, 3), (3, 3, 24, 14, 4, 3), (1, 5, 5, 13, 4, 3),
                                           (5, 4, 7, 7, 2, 0), (1, 2, 40, 5, 0, 3), (2, 8, 16, 15, 0, 0),
                                           (2, 8, 32, 3, 4, 3), (1, 8, 32, 4, 1, 3), (3, 8, 6, 8, 4, 3),
                                           (1, 1, 8, 16, 4, 3), (2, 9, 4, 32, 4, 3), (1, 6, 2, 64, 0, 0),
                                           (1, 7, 2, 128, 4, 3), (3, 8, 5, 9, 4, 3), (2, 6, 9, 11, 3, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_still_equals_repeated_frames(B, T, C, H, kt, ks, dtype):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd.cells import GatedCSSM
    print_case(test="still_image", B=B, T=T, C=C, H=H, kt=kt, ks=ks, dtype=str(dtype))
    cell = GatedCSSM(channels=C, short_conv_size=kt, short_conv_spatial_size=ks, kernel_size=5)
    gen = torch.Generator(device="cuda").manual_seed(H)
    x = torch.randn((B, 1, H, H, C), generator=gen, device="cuda").to(dtype)
    v = cell.init(1, (B, T, H, H, C))
    for q in v["params"].values():                      # every bias non-zero
        if isinstance(q, dict) and "bias" in q:
            q["bias"].normal_(0.0, 0.3, generator=gen)
    ref = cell.apply(v, x.expand(B, T, H, H, C), out_dtype=torch.float32)[:, -1:]
    got = cell._apply_still(v, x, T, out_dtype=torch.float32)
    # the same fp32 arithmetic frame by frame; only the summation order of the projections' and transforms'
    # blocks may differ: a few 1e-6 of RMS
    assert got.shape == ref.shape
    assert (got - ref).abs().max() <= 2e-5 * ref.pow(2).mean().sqrt()


@pytest.mark.parametrize("size,kt", [(2, 4), (4, 2), (4, 6), (1, 3), (4, 0)])
def test_block_image_with_other_taps_than_the_cell_names(size, kt):
    """The cell convolves with the taps of its parameters; a block's image gives the last frame of that."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import blocks, spectral as S
    print_case(test="still_taps", size=size, kt=kt)
    C, T, shape = 32, 8, (2, 14, 14, 32)
    v = blocks.CSSMSHViTBlock(dim=C, num_timesteps=T, kernel_size=5, short_conv_size=kt).init(1, shape)
    block = blocks.CSSMSHViTBlock(dim=C, num_timesteps=T, kernel_size=5, short_conv_size=size)
    assert block.cell._still_pays(2, T, 14, 14, v["params"]["cssm"]) == (kt <= 4)
    gen = torch.Generator(device="cuda").manual_seed(kt)
    x = torch.randn(shape, generator=gen, device="cuda")
    got = block.token_mixer(v, x)
    p, x5 = v["params"], x.unsqueeze(1)
    n, pc = p["norm1"], p["pos_conv"]
    xc = S.block_norm_posconv(x5, S.block_norm_stats(x5, "global_layer"), "global_layer", n["scale"], n["bias"],
                              pc["kernel"], pc["bias"], T)
    ref = x + block.cell.apply({"params": p["cssm"]}, xc)[:, -1]
    assert (got - ref).abs().max() <= 2e-5 * ref.pow(2).mean().sqrt()      # as above


def test_still_rule():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd.cells import GatedCSSM
    c = GatedCSSM(channels=32)
    assert c._still_pays(1, 2, 14, 14) and c._still_pays(64, 5, 32, 32) and not c._still_pays(1, 1, 14, 14)
    assert not c._still_pays(64, 4, 32, 32) and not c._still_pays(64, 8, 16, 32)
    assert not c._still_pays(1, 5, 32, 32) and not c._still_pays(65536, 8, 14, 14)
    assert not GatedCSSM(channels=32, short_conv_size=5)._still_pays(1, 8, 14, 14)
    assert not GatedCSSM(channels=32, short_conv_spatial_size=5)._still_pays(1, 8, 14, 14)
