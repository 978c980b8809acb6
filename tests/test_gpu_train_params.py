"""Parameter tensors of the training entry points in other layouts than a fresh tree's: strided, broadcast and
16-bit ones give the gradients of their contiguous float32 copies, and what no kernel may read is refused."""
import pytest

from tests.gpu_util import print_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mods():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cssm_amd import cells, spectral, training
    return cells, spectral, training


def strided(t):
    """t as one slice of tensors stacked on the last axis."""
    return torch.stack([t, torch.full_like(t, 3.0)], dim=-1)[..., 0]


def leaves(tree):
    return [t for v in tree.values() for t in (leaves(v) if isinstance(v, dict) else [v])]


def grads(apply, cell, variables, x, dout):
    """Output and gradients of x and of every parameter."""
    ls = [x.detach().requires_grad_(True)] + [t.detach().requires_grad_(True) for t in leaves(variables["params"])]
    it = iter(ls[1:])

    def put(tree):
        return {k: put(v) if isinstance(v, dict) else next(it) for k, v in tree.items()}
    y = apply(cell, {"params": put(variables["params"])}, ls[0])
    return [y.detach(), *torch.autograd.grad(y, ls, dout)]


def layer(cls, seed, shape, **kw):
    cell = cls(channels=shape[-1], kernel_size=5, **kw)
    v = cell.init(seed, shape)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for t in leaves(v["params"]):
        t.add_(0.1 * torch.randn(t.shape, generator=gen, device="cuda"))
    x, dout = (torch.randn(shape, generator=gen, device="cuda") for _ in range(2))
    return cell, v, x, dout


def close(got, ref):
    """The same float32 arithmetic through other kernels: sums of some 1e4 O(1) terms, whose rounding stays near
    1e-6 of the largest value."""
    for g, r in zip(got, ref):
        assert g.shape == r.shape
        assert (g.double() - r.double()).abs().max() <= 1e-4 * max(1e-30, r.abs().max().item())


@pytest.mark.parametrize("norm", ["rms", "layer"])
@pytest.mark.parametrize("form", ["strided", "scalar", "bf16", "one"])
def test_gdn_norm_scale_layouts(mods, norm, form):
    """A strided slice, an expanded scalar, 16 bits and a (1,) that broadcasts."""
    cells, _, training = mods
    print_case(test="gdn_norm_scale", norm=norm, form=form)
    cell, v, x, dout = layer(cells.GatedDeltaNetCSSM, 7, (2, 3, 7, 7, 12), delta_key_dim=4, gate_type="factored",
                             output_norm=norm)
    p = v["params"]
    names = [(p, "rms_scale")] if norm == "rms" else [(p["output_layernorm"], n) for n in ("scale", "bias")]
    for d, n in names:                                     # values that every form holds
        d[n] = (d[n][:1].expand(12) if form in ("scalar", "one") else d[n]).bfloat16().float()
    ref = grads(training.gdn_train_apply, cell, v, x, dout)
    for d, n in names:
        t = d[n]
        d[n] = {"strided": strided(t), "scalar": t[:1].expand(12), "bf16": t.bfloat16(), "one": t[:1]}[form]
        assert form in ("bf16", "one") or not d[n].is_contiguous()
    got = grads(training.gdn_train_apply, cell, v, x, dout)
    i = {id(t): k for k, t in enumerate(leaves(p))}
    for d, n in names:
        k = 2 + i[id(d[n])]
        if form == "one":       # the sum over the channels: cancels, so its error is that of its terms, 1e-4 of each
            assert got[k].shape == (1,)
            assert (got[k].double() - ref[k].double().sum()).abs() <= 1e-4 * ref[k].double().abs().sum()
            got[k] = ref[k]
        if form == "bf16":      # rounded to 16 bits
            assert got[k].dtype == torch.bfloat16
            assert (got[k].double() - ref[k].double()).abs().max() <= 2 ** -8 * ref[k].abs().max()
            got[k] = ref[k]
    close(got, ref)


GATED = [((2, 3, 7, 7, 6), "factored", 3), ((1, 2, 16, 16, 8), "dense", 3), ((2, 2, 9, 9, 4), "dense", 0),
         ((1, 3, 32, 32, 2), "factored", 3)]


@pytest.mark.parametrize("shape,gate_type,ks", GATED)
@pytest.mark.parametrize("form", ["strided", "bf16_bias", "one_bias"])
def test_gated_parameter_layouts(mods, shape, gate_type, ks, form):
    """Strided spectral, gate and convolution weights; gate biases in 16 bits or one for all bins."""
    cells, _, training = mods
    print_case(test="gated_params", shape=shape, gates=gate_type, form=form)
    cell, v, x, dout = layer(cells.GatedCSSM, 9, shape, gate_type=gate_type, short_conv_spatial_size=ks,
                             short_conv_size=4 if ks else 0)
    p = v["params"]
    gates = [q for n, q in p.items() if n.startswith(("delta_proj", "B_proj", "C_proj"))]
    for q in gates:
        q["bias"] = (q["bias"][:1].expand_as(q["bias"]).contiguous() if form == "one_bias" else q["bias"] + 0.5)
        q["bias"] = q["bias"].bfloat16().float()
    ref = grads(training.gated_train_apply, cell, v, x, dout)
    if form == "strided":
        p["kernel"] = strided(p["kernel"])
        for n, q in p.items():
            if n not in ("kernel", "in_proj", "out_proj"):
                p[n] = {k: strided(t) for k, t in q.items()}
                assert not any(t.is_contiguous() for t in p[n].values() if t.numel() > 1)
    i = {id(t): k for k, t in enumerate(leaves(p))}
    kept = [2 + i[id(q["bias"])] for q in gates] if form != "strided" else []
    if form != "strided":
        for q in gates:
            q["bias"] = q["bias"].bfloat16() if form == "bf16_bias" else q["bias"][:1].contiguous()
    got = grads(training.gated_train_apply, cell, v, x, dout)
    for k in kept:                                        # as test_gdn_norm_scale_layouts
        r = ref[k].double()
        if form == "one_bias":
            assert (got[k].double() - r.sum()).abs() <= 1e-4 * r.abs().sum()
        else:
            assert got[k].dtype == torch.bfloat16 and (got[k].double() - r).abs().max() <= 2 ** -8 * r.abs().max()
        got[k] = ref[k]
    close(got, ref)


@pytest.mark.parametrize("form", ["strided", "bf16_bias", "one_bias"])
@pytest.mark.parametrize("H", [14, 16])
def test_qkv_depthwise_layouts(mods, form, H):
    """Rows of eight pixels and others: taps and bias strided, the bias in 16 bits or one for all channels."""
    cells, _, training = mods
    print_case(test="qkv_dw_params", form=form, H=H)
    cell, v, x, dout = layer(cells.GatedDeltaNetCSSM, 6, (1, 2, H, H, 8), delta_key_dim=4, gate_type="factored",
                             qkv_conv_size=3)
    q = v["params"]["qkv_dw"]
    q["bias"] = (q["bias"][:1].expand(8).contiguous() if form == "one_bias" else q["bias"]).bfloat16().float()
    i = 2 + [id(t) for t in leaves(v["params"])].index(id(q["bias"]))
    ref = grads(training.gdn_train_apply, cell, v, x, dout)
    if form == "strided":
        q["kernel"], q["bias"] = strided(q["kernel"]), strided(q["bias"])
    else:
        q["bias"] = q["bias"].bfloat16() if form == "bf16_bias" else q["bias"][:1].contiguous()
    got = grads(training.gdn_train_apply, cell, v, x, dout)
    if form != "strided":                                  # as test_gdn_norm_scale_layouts
        r = ref[i].double()
        if form == "one_bias":
            assert (got[i].double() - r.sum()).abs() <= 1e-4 * r.abs().sum()
        else:
            assert got[i].dtype == torch.bfloat16 and (got[i].double() - r).abs().max() <= 2 ** -8 * r.abs().max()
        got[i] = ref[i]
    close(got, ref)


@pytest.mark.parametrize("cls,gate_type", [("gated", "factored"), ("gated", "dense"), ("gdn", "factored"),
                                           ("gdn", "dense"), ("gdn", "channel"), ("gdn", "scalar")])
def test_training_under_autocast(mods, cls, gate_type):
    """A forward and backward inside autocast: the layer computes in float32, torch's products in bf16."""
    cells, _, training = mods
    print_case(test="autocast", cls=cls, gates=gate_type)
    kw = dict(gate_type=gate_type, **({"delta_key_dim": 4} if cls == "gdn" else {}))
    apply = training.gdn_train_apply if cls == "gdn" else training.gated_train_apply
    cell, v, x, dout = layer(cells.GatedDeltaNetCSSM if cls == "gdn" else cells.GatedCSSM, 8, (1, 2, 16, 16, 8), **kw)
    ref = grads(apply, cell, v, x, dout)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got = grads(apply, cell, v, x, dout)
    for g, r in zip(got, ref):                             # bf16 operands: 2^-9 each, sums that cancel some
        assert g.dtype == r.dtype
        assert (g - r).pow(2).sum() <= (5e-2) ** 2 * r.pow(2).sum()


@pytest.mark.parametrize("cls,path", [("gated", "short_conv_spatial"), ("gated", "short_conv_temporal"),
                                      ("gated", "delta_proj_h"), ("gdn", "short_conv_k"), ("gdn", "short_conv_q"),
                                      ("gdn", "alpha_w"), ("gdn", "gate_proj"), ("gdn", "rms_scale")])
def test_mismatched_parameters_raise(mods, cls, path):
    """Parameters of another channel count or plane size than the call's."""
    cells, _, training = mods
    print_case(test="mismatched", cls=cls, path=path)
    kw = dict(gate_type="factored", **({"delta_key_dim": 4} if cls == "gdn" else {}))
    cell, v, x, _ = layer(cells.GatedCSSM if cls == "gated" else cells.GatedDeltaNetCSSM, 3, (1, 2, 16, 16, 8), **kw)
    p = v["params"]
    p[path] = ({k: t[..., :-1].contiguous() for k, t in p[path].items()} if isinstance(p[path], dict)
               else p[path][:-1].contiguous())
    with pytest.raises((ValueError, RuntimeError)):
        (training.gated_train_apply if cls == "gated" else training.gdn_train_apply)(cell, v, x)


def test_taps_follow_the_tree(mods):
    """q, k and v with taps of their own, and trees with fewer taps than the cell's default."""
    cells, _, training = mods
    print_case(test="taps_of_the_tree")
    kw = dict(delta_key_dim=4, gate_type="factored")
    cell, v, x, dout = layer(cells.GatedDeltaNetCSSM, 5, (2, 5, 8, 8, 8), **kw)
    p = v["params"]
    p["short_conv_k"]["kernel"][:2] = 0.0                  # taps a shorter kernel leaves out
    ref = grads(training.gdn_train_apply, cell, v, x, dout)
    i = 2 + [id(t) for t in leaves(p)].index(id(p["short_conv_k"]["kernel"]))
    p["short_conv_k"]["kernel"] = p["short_conv_k"]["kernel"][2:].contiguous()
    ref[i] = ref[i][2:]
    close(grads(training.gdn_train_apply, cell, v, x, dout), ref)
    cell, v, x, dout = layer(cells.GatedCSSM, 5, (1, 5, 16, 16, 8), gate_type="factored", short_conv_size=2)
    ref = grads(training.gated_train_apply, cell, v, x, dout)
    wide = cells.GatedCSSM(channels=8, kernel_size=5, gate_type="factored", short_conv_size=4)
    close(grads(training.gated_train_apply, wide, v, x, dout), ref)


@pytest.mark.parametrize("cls", ["gated", "gdn"])
def test_more_taps_than_the_prep_kernel_holds(mods, cls):
    """65 x 65 taps on 128 x 128 planes: K_hat by torch; zero outer taps give the gradients of the 63 x 63 ones."""
    cells, S, training = mods
    print_case(test="many_taps", cls=cls)
    assert S.spectral_kernel_supported(63, 128, 128) and not S.spectral_kernel_supported(64, 128, 128)
    kw = dict(gate_type="factored", **({"delta_key_dim": 2} if cls == "gdn" else {}))
    apply = training.gdn_train_apply if cls == "gdn" else training.gated_train_apply
    cell, v, x, dout = layer(cells.GatedDeltaNetCSSM if cls == "gdn" else cells.GatedCSSM, 4, (1, 2, 128, 128, 4), **kw)
    k = v["params"]["kernel"]
    k63 = torch.nn.functional.pad(k, (29, 29, 29, 29))
    v["params"]["kernel"] = k63
    i = 2 + [id(t) for t in leaves(v["params"])].index(id(k63))
    ref = grads(apply, cell, v, x, dout)
    v["params"]["kernel"] = torch.nn.functional.pad(k63, (1, 1, 1, 1))
    got = grads(apply, cell, v, x, dout)
    got[i] = got[i][:, 1:-1, 1:-1]
    close(got, ref)


def test_training_wrappers_refuse_other_shapes(mods):
    _, S, _ = mods
    print_case(test="wrappers_refuse")
    r = lambda *s: torch.randn(s, device="cuda")
    x, do, dx = r(1, 2, 8, 7, 7), r(1, 2, 8, 7, 7), r(2, 8, 49)
    good = ((r(3, 3, 1, 8), r(8)), (r(4, 1, 8), r(8)))
    for sp, tp in (((r(3, 3, 1, 7), r(8)), good[1]), ((r(3, 3, 1, 8), r(7)), good[1]), (good[0], (r(4, 1, 7), r(8))),
                   (good[0], (r(4, 1, 8), r(7)))):
        with pytest.raises(ValueError):
            S.short_conv_train(x, sp, tp)
        with pytest.raises(ValueError):
            S.short_conv_backward(x, do, sp, tp, dx)
    with pytest.raises(ValueError):
        S.short_conv_backward(x, do[:, :1].contiguous(), *good, dx)
    with pytest.raises(ValueError):
        S.short_conv_backward(x, do, *good, dx[:1])
    raw, g = r(2, 24, 49), r(2, 2, 49)
    convs = [r(4, 1, 8), r(8)] * 3
    for i, t in ((2, r(3, 1, 8)), (4, r(4, 1, 7)), (1, r(7))):
        bad = convs[:i] + [t] + convs[i + 1:]
        with pytest.raises(ValueError):
            S.gdn_qkv_act(raw, 1, 2, bad, 1, g)
        with pytest.raises(ValueError):
            S.gdn_qkv_act_backward(raw, 1, 2, bad, 1, g, torch.empty_like(raw), torch.empty_like(raw))
    with pytest.raises(ValueError):
        S.gdn_qkv_act(raw, 1, 2, convs, 1, g[:, :1].contiguous())
    with pytest.raises(ValueError):
        S.gdn_qkv_act(raw, 1, 3, convs, 1, g)
    spec, _ = S.rfft2(r(1, 2, 24, 8, 8))
    ab, what = r(1, 2, 40, 2), torch.zeros((2, 8, 5), dtype=torch.complex64, device="cuda")
    norms = r(1, 2, 24)
    S.gdn_core_train(spec, norms, ab, "dense", what, 4, 8)
    for a in ((spec, norms, ab[:, :, :39].contiguous(), what), (spec, norms, ab, what[:1]),
              (spec, norms[:, :, :23].contiguous(), ab, what)):
        with pytest.raises(ValueError):
            S.gdn_core_train(a[0], a[1], a[2], "dense", a[3], 4, 8)


def test_norm_gate_refuses_what_it_would_misread(mods):
    _, S, _ = mods
    print_case(test="norm_gate_refuses")
    o, g = (torch.randn((2, 8, 16), device="cuda") for _ in range(2))
    ok = torch.ones(8, device="cuda")
    bad = [strided(ok), ok[:1].expand(8), ok.double(), ok.bfloat16(), ok.cpu(), ok[:7], torch.ones(9, device="cuda")]
    for t in bad:
        for scale, shift in ((t, None), (ok, t)):
            with pytest.raises(ValueError):
                S.gdn_norm_gate(o, g, "layer", scale, shift, "silu")
            with pytest.raises(ValueError):
                S.gdn_norm_gate_backward(o, g, "layer", scale, shift, "silu", torch.empty_like(o), torch.empty_like(g))
