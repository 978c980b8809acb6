"""The gated scan through spectra in HBM (cssm_gated_scan_bins between the batched transforms) against
the fused kernel and, with a plane of zeros on the floor, at the edges of its frame and batch pieces."""
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


def _case(S, B, T, C, H, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    u = torch.randn((B, T, C, H, H), generator=gen, device="cuda")
    u[:, :max(1, T // 2), 0] = 0.0                          # every bin of the first frames on the floor
    z = torch.randn(u.shape, generator=gen, device="cuda")
    ctx = torch.randn((B, T, C), generator=gen, device="cuda")
    Wf = H // 2 + 1
    p = {n: {"kernel": 0.2 * torch.randn((C, H * Wf), generator=gen, device="cuda"),
             "bias": 0.5 * torch.randn(H * Wf, generator=gen, device="cuda")}
         for n in ("delta_proj", "B_proj", "C_proj")}
    gates = S.gated_gates(ctx, p, H, H, "dense", "softplus", S.scan_c_scale(H, H))
    k = 0.3 * torch.randn((C, 5, 5), generator=gen, device="cuda")
    return u, z, gates, S.spectral_kernel(k, H, H, scan_order=True)


# T around the eight frames held in flight; 128: the scan's column and K_hat orders
@pytest.mark.parametrize("B,T,C,H", [(2, 1, 32, 8), (1, 7, 40, 16), (1, 8, 8, 16), (3, 9, 8, 16), (1, 17, 6, 32),
                                     (2, 3, 3, 64), (1, 5, 2, 128), (2, 9, 7, 7), (1, 5, 40, 3), (3, 4, 11, 14),
                                     (1, 11, 19, 13), (2, 3, 32, 4)])
@pytest.mark.parametrize("pieces", [None, "batch", "frames"])
def test_split_scan_equals_fused(S, monkeypatch, B, T, C, H, pieces):
    print_case(test="split_scan", B=B, T=T, C=C, H=H, pieces=pieces)
    u, z, gates, khat = _case(S, B, T, C, H)
    monkeypatch.setattr(S, "gated_split_rule", lambda *a: False)
    ref = S.gated_scan(u, z, gates, khat)
    frame = C * H * (H // 2 + 1) * 8
    kw = {None: {}, "batch": {"max_bytes": frame * T}, "frames": {"max_bytes": frame * 3}}[pieces]
    got = S._gated_scan_split(u, z, gates, khat, torch.empty_like(u), **kw)
    # both are fp32 transforms of <= 2^14 samples around the same recurrence: a few 1e-6 of RMS
    assert (got - ref).abs().max() <= 2e-5 * ref.pow(2).mean().sqrt()
    # the floored plane is about 1e-7 of the rest: on its own scale
    got, ref = got[:, :max(1, T // 2), 0], ref[:, :max(1, T // 2), 0]
    assert ref.abs().max() > 0 and (got - ref).abs().max() <= 2e-5 * ref.pow(2).mean().sqrt()


def test_rule_picks_the_split_form_for_few_planes(S):
    assert S.gated_split_rule(256, 1024, 16, 16) and S.gated_split_rule(64, 8, 128, 128)
    assert not S.gated_split_rule(8192, 8, 128, 128) and not S.gated_split_rule(1024, 1, 32, 32)
    assert S.gated_split_rule(64, 64, 7, 7) and not S.gated_split_rule(64, 4, 7, 7)
    assert not S.gated_split_rule(64, 64, 16, 32)


def test_what_the_fused_scan_refuses_stays_refused(S):
    """Channels that are no whole group and planes off 16 bytes, at sizes where the rule takes the split form."""
    from cssm_amd._lib import CssmError
    print_case(test="split_refuses")
    assert S.gated_split_rule(4, 64, 16, 16) and S.gated_split_rule(5, 64, 7, 7)
    u, z, gates, khat = _case(S, 1, 64, 4, 16)
    with pytest.raises(CssmError, match="multiple of 8"):
        S.gated_scan(u, z, gates, khat)
    u, z, gates, khat = _case(S, 1, 64, 5, 7)
    with pytest.raises(CssmError, match="non-null"):        # an empty tensor has no address
        S.gated_scan(u[:0], z[:0], gates[:0], khat)
    off = torch.zeros(u.numel() + 1, device="cuda")[1:].view(u.shape)
    for a in ((off, z, None), (u, off, None), (u, z, off)):
        with pytest.raises(CssmError, match="misaligned"):
            S.gated_scan(a[0], a[1], gates, khat, out=a[2])


@pytest.mark.parametrize("H", [3, 7, 12, 14, 15])
def test_small_plane_transforms_with_fused_work(S, H):
    """cssm_rfft2_ex / cssm_irfft2_ex on small planes: strided halves of a (F, 2C, HW) tensor, activations,
    the factor, the per-plane addend and SiLU', against torch in float64 (a few fp32 roundings: 2e-6 of RMS)."""
    print_case(test="small_ex", H=H)
    gen = torch.Generator(device="cuda").manual_seed(H)
    F, C, HW = 3, 13, H * H
    xz, m = (torch.randn((F, n, HW), generator=gen, device="cuda") for n in (2 * C, C))
    x, a = xz[:, :C], xz[:, C:]
    add = torch.randn((F, C), generator=gen, device="cuda")
    sil = torch.nn.functional.silu

    def close(got, ref):
        assert (got - ref).abs().max() <= 1e-5 * ref.abs().pow(2).mean().sqrt()
    spec = S.rfft2_ex(x, H, H, x_silu=True, a=a, a_silu=True)
    ref = torch.fft.rfft2((sil(x.double()) * sil(a.double())).view(F, C, H, H))
    close(spec.to(torch.complex128), ref)
    close(S.rfft2_ex(a, H, H).to(torch.complex128), torch.fft.rfft2(a.double().reshape(F, C, H, H)))
    out = torch.zeros_like(xz)
    S.irfft2_ex(spec, H, out[:, C:], add=add, m=m, d=x)
    s = torch.sigmoid(x.double())
    want = ((torch.fft.irfft2(ref, s=(H, H)).view(F, C, HW) + add.double()[..., None]) * m.double()
            * s * (1 + x.double() * (1 - s)))
    close(out[:, C:].double(), want)
    assert not out[:, :C].any()
