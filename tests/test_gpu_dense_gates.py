"""Dense gates over the frames-per-workgroup choices (cssm_gated_gates) against float64."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# frames below and above the counts where one, two, four and eight frames share a workgroup, ragged last
# groups, one bin run and several, the scan's column order at 128
@pytest.mark.parametrize("B,T,C,H", [(1, 1, 3, 7), (3, 171, 8, 8), (1, 1030, 5, 16), (2, 37, 12, 64), (1, 2051, 4, 7),
                                     (1, 35, 6, 128), (1, 131, 4, 64), (1, 4100, 3, 5)])
def test_dense_gates(B, T, C, H):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import spectral as S
    print_case(test="dense_gates", B=B, T=T, C=C, H=H)
    gen = torch.Generator(device="cuda").manual_seed(T)
    Wf = H // 2 + 1
    ctx = torch.randn((B, T, C), generator=gen, device="cuda")
    p = {n: {"kernel": torch.randn((C, H * Wf), generator=gen, device="cuda"),
             "bias": torch.randn(H * Wf, generator=gen, device="cuda")} for n in ("delta_proj", "B_proj", "C_proj")}
    got = S.gated_gates(ctx, p, H, H, "dense", "softplus", 0.5)
    g = [(ctx.double() @ p[n]["kernel"].double() + p[n]["bias"].double()).view(B, T, H, Wf) for n in p]
    d = torch.nn.functional.softplus(g[0])
    ref = torch.stack([torch.exp(-d), (d + 1e-8) * g[1], 2e-7 * (d + 1e-8), 0.5 * g[2]], dim=-1)
    ref = ref[:, :, :, S.scan_col_order(H, H)]
    # sums of at most 13 fp32 products, then O(1) functions of them
    assert ((got.double() - ref).abs() <= 2e-6 * (1 + ref.abs().amax())).all()
    # the same whatever the frames it shares a workgroup with: a frame alone
    one = S.gated_gates(ctx[-1:, -1:].contiguous(), p, H, H, "dense", "softplus", 0.5)
    assert torch.equal(one[0, 0], got[-1, -1])
