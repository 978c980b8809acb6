"""The GDN cell's paths for few sequences, heads or bins against those for many: the same values."""
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


def randn(gen, *shape, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


@pytest.mark.parametrize("dk,H,T", [(1, 8, 5), (2, 7, 1), (3, 14, 2), (4, 16, 9), (4, 128, 2)])
def test_scan_bins_ahead_equals_plain(S, dk, H, T):
    """Few bins load a step ahead in 64-thread workgroups; a batch past 512 workgroups does not."""
    print_case(test="bins_ahead", dk=dk, H=H, T=T)
    gen = torch.Generator(device="cuda").manual_seed(dk * H)
    C, Wf = 2 * dk, H // 2 + 1
    B = 512 // (2 * ((H * Wf + 255) // 256)) + 1
    spec = randn(gen, B, T, 3 * C, H, Wf, dtype=torch.complex64)
    spec[:, :, C] = 0                                     # zero keys: the floored form of the step
    norms = torch.rand((B, T, 3 * C), generator=gen, device="cuda") + 0.5
    ab = torch.rand((B, T, H * Wf, 2), generator=gen, device="cuda")
    what = 0.4 * randn(gen, C // dk, H, Wf, dtype=torch.complex64)
    many = S.gdn_scan_bins(spec, norms, ab, "dense", what, dk)
    few = S.gdn_scan_bins(spec[-1:].contiguous(), norms[-1:].contiguous(), ab[-1:].contiguous(), "dense", what, dk)
    assert torch.equal(few[0], many[-1])


# one, two, four and eight frames a workgroup, ragged last groups
@pytest.mark.parametrize("B,T,C,H", [(1, 3, 4, 8), (1, 401, 8, 8), (1, 1030, 4, 16), (3, 700, 4, 16), (1, 77, 4, 64)])
@pytest.mark.parametrize("kv", [True, False])
def test_dense_gates_do_not_depend_on_the_frame_count(S, B, T, C, H, kv):
    print_case(test="gdn_dense_gates", B=B, T=T, C=C, H=H, kv=kv)
    gen = torch.Generator(device="cuda").manual_seed(T)
    Wf = H // 2 + 1
    ctx = randn(gen, B, T, C)
    p = {n: {"kernel": randn(gen, C, m), "bias": randn(gen, m)}
         for n, m in (("alpha", H * Wf), ("beta", H * Wf), ("B_k", H * H), ("B_v", H * H))}
    ab, bkv = S.gdn_gates(ctx, p, H, H, 2, "dense", kv, "none")
    f = [torch.sigmoid(ctx.double() @ p[n]["kernel"].double() + p[n]["bias"].double()) for n in p]
    # sums of at most nine fp32 products through a sigmoid
    assert (ab.double() - torch.stack([0.1 + 0.89 * f[0], f[1]], dim=-1)).abs().max() <= 2e-6
    assert (bkv is None) == (not kv)
    if kv:
        assert (bkv.double() - torch.stack(f[2:], dim=-1)).abs().max() <= 2e-6
    sa, _ = S.gdn_gates(ctx, p, H, H, 2, "dense", kv, "sinusoid")
    one, _ = S.gdn_gates(ctx[:, :3].contiguous(), p, H, H, 2, "dense", kv, "sinusoid")
    assert torch.equal(sa[:, :3], one)


@pytest.mark.parametrize("B,T,H,C", [(1, 4, 64, 32), (1, 5, 8, 64), (4, 8, 32, 64), (65, 4, 8, 8)])
def test_qkv_of_few_sequences_equals_many(S, B, T, H, C):
    """Up to 64 (element, 64-pixel block) sequences take the projection and the post pass."""
    print_case(test="qkv_few", B=B, T=T, H=H, C=C)
    gen = torch.Generator(device="cuda").manual_seed(C)
    x, W, b = randn(gen, 70, T, H, H, C), 0.1 * randn(gen, C, 3 * C), randn(gen, 3 * C)
    convs = [{"kernel": randn(gen, 4, 1, C), "bias": randn(gen, C)} for _ in range(3)]
    g = torch.rand((70, T, H * H, 2), generator=gen, device="cuda")
    many = S.gdn_qkv_proj(x, W, b, 70, T, H, H, convs, 1, g, out_dtype=torch.float32)
    few = S.gdn_qkv_proj(x[:B].contiguous(), W, b, B, T, H, H, convs, 1, g[:B].contiguous(), out_dtype=torch.float32)
    assert torch.equal(few, many[:B])


def test_fused_core_rule(S):
    assert S.gdn_core_fused_pays(128, 32, 64, 4) and S.gdn_core_fused_pays(1, 1, 64, 4)
    assert not S.gdn_core_fused_pays(1, 8, 64, 4) and not S.gdn_core_fused_pays(16, 4, 64, 4)
