"""The fp32 convolution on weights that were taken apart beforehand: each tile height forced at the edges of its tiles and steps,
its error against float64 beside the fp32 instructions', the operands that those multiply instead, and the layer that keeps the
pieces."""
import numpy as np
import pytest
import torch

from test_gpu_direct import bound, forced, tiles_of  # noqa: F401

pytestmark = pytest.mark.gpu

FORMS = ["pieces32", "pieces64", "pieces64+32"]
# "pieces64+32" forced takes half of the whole 64-row tiles and leaves the rest to 32-row ones.
# (B, nH, nW, C, K): M = 1, 17, 33, 65, 130, 255 rows; C below, at and past 16, 32 and 64 indices; K below, at and past 64, and more
# than four columns of tiles; the last one has more tiles than a GPU has CUs
SHAPES = [(1, 1, 1, 4, 4), (1, 1, 17, 36, 20), (3, 1, 11, 64, 68), (1, 5, 13, 16, 64), (2, 5, 13, 160, 36), (1, 15, 17, 128, 132),
          (1, 7, 10, 96, 328), (1, 13, 15, 20, 64), (6, 40, 70, 64, 40)]


def dev(a):
    return torch.from_numpy(a).cuda()


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
def test_pieces_forms(oracle, forced, form, shape):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    B, nH, nW, C, K = shape
    rng = np.random.default_rng(81)
    ti = np.maximum(rng.standard_normal((16, B, nH, nW, C)), 0).astype(np.float32)
    w = (rng.standard_normal((16, C, K)) * 0.05).astype(np.float32)
    tii = rng.integers(-4, 5, size=ti.shape).astype(np.float32)
    wi = rng.integers(-4, 5, size=w.shape).astype(np.float32)
    scale, shift = rng.standard_normal(K).astype(np.float32), rng.standard_normal(K).astype(np.float32)
    res = rng.standard_normal((B, 2 * nH, 2 * nW, K)).astype(np.float32)
    pieces, pieces_i = winograd2x2_weight_pieces(dev(w)), winograd2x2_weight_pieces(dev(wi))
    assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
    got = winograd2x2_conv(dev(ti), dev(w), pieces=pieces).cpu().numpy()
    assert forced.swc_winograd2x2_conv_last_form().decode() == form
    exact = winograd2x2_conv(dev(tii), dev(wi), pieces=pieces_i).cpu().numpy()
    ep = winograd2x2_conv(dev(ti), dev(w), scale=dev(scale), shift=dev(shift), residual=dev(res), residual_relu=True, pieces=pieces).cpu().numpy()
    buf = dev(res)
    winograd2x2_conv(dev(ti), dev(w), out=buf, residual=buf, pieces=pieces)   # residual aliasing the output
    want = oracle.conv(ti, w, acc64=True)
    err = np.abs(tiles_of(got, nH, nW).astype(np.float64) - tiles_of(want, nH, nW))
    # the fp32 instructions' bound, and one more rounding a product for the products of pieces that are left out
    more = 1 + 1 / (w.shape[1] + 8)
    assert (err <= more * bound(ti, w)[:, None, :] + 2.0 ** -24 * np.abs(tiles_of(want, nH, nW))).all()
    assert np.array_equal(exact, oracle.conv(tii, wi))
    assert np.array_equal(ep, oracle.affine(got, scale, shift) + np.maximum(res, 0))
    assert np.array_equal(buf.cpu().numpy(), got + res)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("C,K", [(16, 320), (16, 448), (16, 512), (192, 512), (16, 576), (16, 832)])
def test_panels_of_columns(forced, form, C, K):  # noqa: F811
    """5, 7, 8, 9 and 13 columns of tiles: in one panel, in two of four (the weights of 192 channels are too large for one), five and
    four, seven and six.  Whole numbers are exact in any order of the sums."""
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    gen = torch.Generator(device="cuda").manual_seed(86)
    ti = torch.randint(-4, 5, (16, 3, 7, 11, C), device="cuda", generator=gen).float()
    w = torch.randint(-4, 5, (16, C, K), device="cuda", generator=gen).float()
    assert forced.swc_winograd2x2_conv_force_tiling(b"direct32x64") == 0
    want = winograd2x2_conv(ti, w)
    assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
    assert torch.equal(winograd2x2_conv(ti, w, pieces=winograd2x2_weight_pieces(w)), want)
    assert forced.swc_winograd2x2_conv_last_form().decode() == form


@pytest.mark.parametrize("shape,precision,want", [
    ((64, 4, 4, 512, 512), "fp32", "pieces32"),
    ((64, 5, 5, 192, 320), "fp32", "pieces32"),        # five columns of tiles
    ((21, 25, 4, 512, 96), "fp32", "split32"),         # planes beyond 64 MiB and 32-row tiles
    ((54, 13, 13, 64, 256), "fp32", "pieces64+32"),    # five rounds of 32-row tiles are no faster than short16
    ((64, 7, 7, 256, 256), "fp32", "pieces64"),
    ((128, 7, 7, 512, 512), "fp32", "pieces64+32"),    # three rounds of 64-row tiles over two panels, the rest in 32-row ones
    ((64, 4, 4, 512, 512), "bf16", "pieces32"),
    ((4, 29, 31, 256, 512), "bf16", "whole"),          # two rounds of 64-row tiles, planes of 59 MB
    ((128, 7, 7, 256, 256), "bf16", "pieces64"),       # two, 103 MB
    ((128, 7, 7, 512, 512), "bf16", "pieces64+32"),
    ((64, 7, 7, 256, 256), "bf16", "split64"),
])
def test_where_prepared_weights_are_used(forced, shape, precision, want):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the picks are those of 256 CUs")
    B, nH, nW, C, K = shape
    w = torch.ones((16, C, K), device="cuda")
    winograd2x2_conv(torch.ones((16, B, nH, nW, C), device="cuda"), w, precision, pieces=winograd2x2_weight_pieces(w, precision))
    assert forced.swc_winograd2x2_conv_last_form().decode() == want
    gain = {"fp32": forced.swc_winograd2x2_conv_pieces_gain, "bf16": forced.swc_winograd2x2_conv_pieces_bf16_gain}[precision]
    assert (gain(C, B, nH, nW, K) > 0) == want.startswith("pieces")


@pytest.mark.parametrize("C", [64, 72, 256, 512])
@pytest.mark.parametrize("density", [0.1, 0.3, 1.0])
@pytest.mark.parametrize("magnitude", [(1.0, 0.05), (1e-6, 1e-5), (3e4, 20.0)])
def test_no_further_from_float64_than_in_one_kernel(forced, C, density, magnitude):  # noqa: F811
    """Against the forms that take the weights apart themselves and the fp32 instructions."""
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    gen = torch.Generator(device="cuda").manual_seed(82)
    ti = torch.randn((16, 4, 16, 16, C), device="cuda", generator=gen).relu_() * magnitude[0]
    w = torch.randn((16, C, 128), device="cuda", generator=gen)
    w *= magnitude[1] * (w.abs() >= w.abs().flatten()[::7].quantile(1 - density))     # the largest are kept
    p = torch.bmm(ti.reshape(16, -1, C).double(), w.double()).reshape(4, 4, -1, 128)
    rows = torch.stack([p[0] + p[1] + p[2], p[1] - p[2] - p[3]])
    want = torch.stack([rows[:, 0] + rows[:, 1] + rows[:, 2], rows[:, 1] - rows[:, 2] - rows[:, 3]], 1)   # [dy,dx,M,K]
    want = want.reshape(2, 2, 4, 16, 16, 128).permute(2, 3, 0, 4, 1, 5).reshape(4, 32, 32, 128)
    pieces = winograd2x2_weight_pieces(w)
    errors = {}
    for form in FORMS + ["direct16x64", "split64"]:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        errors[form] = ((winograd2x2_conv(ti, w, pieces=pieces).double() - want).norm() / want.norm()).item()
        assert forced.swc_winograd2x2_conv_last_form().decode() == form
    # with few products (64 channels at 10 %) the outputs' own nine-term sums make most of either's error: equal to 1 %
    assert all(errors[f] <= 1.01 * min(errors["direct16x64"], errors["split64"]) for f in FORMS), errors


@pytest.mark.parametrize("name", ["infinite", "nan", "late outlier", "large weights", "large activations", "tiny", "infinite weight"])
def test_operands_left_to_the_fp32_instructions(forced, name):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    gen = torch.Generator(device="cuda").manual_seed(83)
    ti = torch.randn((16, 1, 8, 12, 96), device="cuda", generator=gen).relu_()
    w = torch.randn((16, 96, 64), device="cuda", generator=gen) * 0.05
    if name == "infinite":
        ti[3, 0, 2, 5, 40] = float("inf")
    elif name == "infinite weight":
        w[9, 70, 11] = float("-inf")
    elif name == "nan":
        ti[5, 0, 7, 7, 95] = float("nan")
    elif name == "late outlier":
        ti[:, :, :, :, 64:] *= 1e12
    elif name == "large weights":
        w, ti = w * 1e34, ti * 1e-34
    elif name == "large activations":
        w, ti = w * 1e-34, ti * 1e34
    elif name == "tiny":
        w, ti = w * 1e-10, ti * 1e-20
    pieces = winograd2x2_weight_pieces(w)
    assert forced.swc_winograd2x2_conv_force_tiling(b"direct32x64") == 0
    want = winograd2x2_conv(ti, w)
    finite = torch.isfinite(want)
    for form in FORMS:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        got = winograd2x2_conv(ti, w, pieces=pieces)
        assert torch.equal(torch.isnan(got), torch.isnan(want)), form
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]), form
        # sums of 96 products and nine terms in another order
        assert (got[finite].double() - want[finite]).norm() <= 1e-5 * want[finite].double().norm(), form


@pytest.mark.parametrize("form", FORMS)
def test_scaling_by_powers_of_two_commutes(forced, form):  # noqa: F811
    """Rows, columns and channels scaled against each other down to 2^-50: nothing may round differently."""
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    gen = torch.Generator(device="cuda").manual_seed(84)
    ti = torch.randn((16, 2, 9, 8, 96), device="cuda", generator=gen).relu_()
    w = torch.randn((16, 96, 72), device="cuda", generator=gen)
    assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
    run = lambda a, b: winograd2x2_conv(a, b, pieces=winograd2x2_weight_pieces(b))   # noqa: E731
    plain = run(ti, w)
    powers = torch.tensor([0, 0, -24, 0, -28, -34, 0, -44, -46, 0, -50], device="cuda")
    pick = lambda n: (2.0 ** powers[torch.arange(n, device="cuda") % len(powers)].double()).float()   # noqa: E731
    rows, cols = pick(144), pick(72)
    by_pixel = rows.reshape(2, 9, 1, 8, 1, 1).expand(2, 9, 2, 8, 2, 1).reshape(2, 18, 16, 1)
    assert torch.equal(run(ti * rows.reshape(1, 2, 9, 8, 1), w), plain * by_pixel)
    assert torch.equal(run(ti, w * cols), plain * cols)
    channels = (2.0 ** ((torch.arange(96, device="cuda") * 7 % 41 - 20).double())).float()
    assert torch.equal(run(ti * channels, w / channels.reshape(96, 1)), plain)


@pytest.mark.parametrize("masked", [False, True])
def test_layer_follows_its_weights(oracle, masked):
    """The layer's pieces are those of the weights it has at the call: written in place, replaced, masked anew; with gradients
    and without."""
    import swc_hip
    from winograd_conv import WinogradConv
    gen = torch.Generator(device="cuda").manual_seed(85)
    B, n, C = 64, 7, 256
    ti = torch.randn((16, B, n, n, C), device="cuda", generator=gen).relu_()
    w = torch.randn((16, C, C), device="cuda", generator=gen) * 0.05
    mask = (torch.rand((16, C, C), device="cuda", generator=gen) < 0.3).float() if masked else None
    layer = WinogradConv(C, C, mask=mask, W_init=w, device="cuda")

    def check():
        m = layer.W.detach().double() if layer.mask is None else layer.W.detach().double() * layer.mask
        p = torch.bmm(ti.reshape(16, -1, C).double(), m).reshape(4, 4, -1, C)
        r = torch.stack([p[0] + p[1] + p[2], p[1] - p[2] - p[3]])
        want = torch.stack([r[:, 0] + r[:, 1] + r[:, 2], r[:, 1] - r[:, 2] - r[:, 3]], 1).reshape(2, 2, B, n, n, C)
        want = want.permute(2, 3, 0, 4, 1, 5).reshape(B, 2 * n, 2 * n, C)
        for grad in (False, True):
            with torch.set_grad_enabled(grad):
                y = layer(ti)
            if torch.cuda.get_device_properties(0).multi_processor_count == 256:
                assert swc_hip.lib().swc_winograd2x2_conv_last_form() == b"pieces64"
            assert (y.detach().double() - want).norm() <= 1e-6 * want.norm()

    check()
    with torch.no_grad():
        layer.W.mul_(-1.5)
    check()
    if masked:
        layer.mask.copy_(1 - layer.mask)
        check()
    else:
        layer.W.data.mul_(0.5)      # no trace on W: nothing may be kept of it
        check()
    layer.W = torch.nn.Parameter(torch.randn((16, C, C), device="cuda", generator=gen))
    check()
    layer.load_state_dict({k: v.flip(1) for k, v in layer.state_dict().items()})
    check()


def test_pieces_that_are_not_the_weights_are_refused():
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    ti, w = torch.zeros((16, 1, 2, 2, 64), device="cuda"), torch.zeros((16, 64, 64), device="cuda")
    pieces = winograd2x2_weight_pieces(w)
    for bad in (pieces[:-16], pieces.view(torch.int8), pieces.cpu()):
        with pytest.raises(ValueError):
            winograd2x2_conv(ti, w, pieces=bad)
    with pytest.raises(ValueError):
        winograd2x2_conv(ti, w, precision="bf16", pieces=pieces)


@pytest.mark.parametrize("form", ["pieces32", "pieces64", "pieces64+32"])
@pytest.mark.parametrize("shape", [(1, 1, 1, 64, 4), (1, 4, 8, 192, 64), (2, 5, 6, 64, 68), (1, 13, 5, 128, 132), (2, 8, 8, 128, 64), (3, 9, 7, 320, 200)])
def test_bf16_operands(shape, form):
    # Rows and columns below, at and beyond a tile (32 or 64 rows, 64 columns), one, two, three and five times the four half steps of 16
    # indices that are on their way.  Whole numbers are exact in bf16 and in any order of the sums; for others the kernel's products are those of
    # the rounded operands, summed in fp32: at most C roundings of 2^-24 each for sums of at most sum|a b|.
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    import swc_hip
    B, nH, nW, C, K = shape
    gen = torch.Generator().manual_seed(17)
    dev = torch.device("cuda:0")
    whole = [torch.randint(-4, 5, s, generator=gen).float() for s in ((16, B, nH, nW, C), (16, C, K))]
    real = [torch.relu(torch.randn((16, B, nH, nW, C), generator=gen)), torch.randn((16, C, K), generator=gen)]
    lib = swc_hip.lib()

    def conv(ti, w, name):
        pieces = winograd2x2_weight_pieces(w.to(dev), "bf16")
        assert lib.swc_winograd2x2_conv_force_tiling(name.encode() if name else None) == 0
        try:
            y = winograd2x2_conv(ti.to(dev), w.to(dev), "bf16", pieces=pieces if name else None).cpu()
            assert name is None or lib.swc_winograd2x2_conv_last_form().decode() == name
            return y
        finally:
            lib.swc_winograd2x2_conv_force_tiling(None)
    assert torch.equal(conv(*whole, form), conv(*whole, None))
    ti, w = (v.bfloat16().double() for v in real)

    def out_of(p):   # A^T p A in float64, p [16,B,nH,nW,K]; with magnitudes for the bound
        return p.reshape(4, 4, B, nH, nW, K)
    a = torch.tensor([[1, 1, 1, 0], [0, 1, -1, -1]], dtype=torch.float64)
    p = out_of(torch.matmul(ti.reshape(16, -1, C), w))
    size = out_of(torch.matmul(ti.reshape(16, -1, C).abs(), w.abs()))
    fold = lambda m, q: torch.einsum("ai,bj,ijnhwk->nhawbk", m, m, q).reshape(B, 2 * nH, 2 * nW, K)   # noqa: E731
    got = conv(*real, form).double()
    assert ((got - fold(a, p)).abs() <= (C + 16) * 2.0 ** -24 * fold(a.abs(), size)).all()
    # an infinity stays in its own tile's outputs
    bad = real[0].clone()
    bad[5, 0, nH - 1, nW - 1, 0] = float("inf")
    got, want = conv(bad, real[1], form), conv(bad, real[1], None)
    assert torch.equal(got.isfinite(), want.isfinite())
    assert (~got.isfinite()).sum() == 4 * K


@pytest.mark.parametrize("precision,shape,form", [
    ("bf16", (95, 7, 7, 512, 256), "pieces64+32"),     # 292 tiles: a round of 64-row ones, the rest in 32-row ones
    ("bf16", (128, 7, 7, 512, 512), "pieces64+32"),    # three rounds, two panels of columns
    ("bf16", (128, 7, 7, 256, 256), "pieces64"),       # two rounds, the second of 136 tiles
    ("fp32", (128, 7, 7, 512, 512), "pieces64+32"),
    ("fp32", (68, 28, 4, 192, 256), "pieces64"),       # two rounds
])
def test_several_rounds_as_the_launcher_takes_them(precision, shape, form):
    """A workgroup's later tiles, whose operands are loaded beside the one before, panels of columns and the lower tiles behind: against
    float64 of the operands as they are multiplied, all rows."""
    import swc_hip
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    B, nH, nW, C, K = shape
    gen = torch.Generator(device="cuda").manual_seed(31)
    ti = torch.randn((16, B, nH, nW, C), device="cuda", generator=gen).relu_()
    w = torch.randn((16, C, K), device="cuda", generator=gen) * 0.05
    got = winograd2x2_conv(ti, w, precision, pieces=winograd2x2_weight_pieces(w, precision))
    if form is not None and torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert swc_hip.lib().swc_winograd2x2_conv_last_form().decode() == form
    a, b = (ti.reshape(16, -1, C), w) if precision == "fp32" else (ti.reshape(16, -1, C).bfloat16().float(), w.bfloat16().float())
    y = torch.zeros((2, 2, B * nH * nW, K), dtype=torch.float64, device="cuda")
    size = torch.zeros_like(y)
    at = torch.tensor([[1, 1, 1, 0], [0, 1, -1, -1]], dtype=torch.float64)
    for i in range(16):
        p, q = torch.mm(a[i].double(), b[i].double()), torch.mm(a[i].double(), b[i].double().abs())
        for dy in range(2):
            for dx in range(2):
                f = float(at[dy, i // 4] * at[dx, i % 4])
                if f:
                    y[dy, dx] += f * p
                    size[dy, dx] += q
    got = got.reshape(B, nH, 2, nW, 2, K).permute(2, 4, 0, 1, 3, 5).reshape(y.shape)
    # at most C roundings of a sum, and what nine terms and three pieces add
    assert ((got.double() - y).abs() <= (C + 16) * 2.0 ** -24 * size).all()
    assert (got.double() - y).norm() <= 1e-6 * y.norm()


@pytest.mark.parametrize("C", [4, 48, 80, 96])
def test_bf16_operands_of_other_channels_are_multiplied_with_the_weights_themselves(forced, C):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weight_pieces
    gen = torch.Generator(device="cuda").manual_seed(32)
    ti, w = torch.randn((16, 2, 5, 6, C), device="cuda", generator=gen), torch.randn((16, C, 68), device="cuda", generator=gen)
    want = winograd2x2_conv(ti, w, "bf16")
    assert torch.equal(winograd2x2_conv(ti, w, "bf16", pieces=winograd2x2_weight_pieces(w, "bf16")), want)
    assert not forced.swc_winograd2x2_conv_last_form().startswith(b"pieces")


@pytest.mark.parametrize("masked", [True, False])
def test_a_bf16_layer_is_the_op_on_its_weights(masked):
    # 7x7x512 at batch 64 is multiplied with the layer's prepared weights where it has a mask; a write to them is noticed.
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    from winograd_conv import WinogradConv
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(23)
    ti = torch.randint(0, 5, (16, 64, 4, 4, 512), device=dev, generator=gen).float()
    mask = (torch.rand((16, 512, 512), device=dev, generator=gen) < 0.3).float() if masked else None
    layer = WinogradConv(512, 512, mask=mask, W_init=torch.randint(-4, 5, (16, 512, 512), device=dev, generator=gen).float(), device=dev, precision="bf16")
    with torch.no_grad():
        for _ in range(2):
            w = layer.W.detach() if mask is None else layer.W.detach() * mask
            assert torch.equal(layer(ti), winograd2x2_conv(ti, w, "bf16"))
            assert (layer._pieces is not None) == masked
            layer.W.mul_(2)


def masked_layer(precision, C):
    """A masked layer, planes of a shape whose convolution uses kept pieces and of one whose does not, and the former's output in float64."""
    from winograd_conv import WinogradConv
    gen = torch.Generator(device="cuda").manual_seed(29)
    B, n = (64, 7) if precision == "fp32" else (128, 8)
    ti = torch.randn((16, B, n, n, C), device="cuda", generator=gen).relu_()
    w = torch.randn((16, C, C), device="cuda", generator=gen) * 0.05
    layer = WinogradConv(C, C, mask=(torch.rand((16, C, C), device="cuda", generator=gen) < 0.3).float(), W_init=w, device="cuda", precision=precision)
    wm, t = layer.W.detach() * layer.mask, ti.reshape(16, -1, C)
    if precision == "bf16":
        wm, t = wm.bfloat16(), t.bfloat16()
    p = torch.bmm(t.double(), wm.double()).reshape(4, 4, -1, C)
    r = torch.stack([p[0] + p[1] + p[2], p[1] - p[2] - p[3]])
    want = torch.stack([r[:, 0] + r[:, 1] + r[:, 2], r[:, 1] - r[:, 2] - r[:, 3]], 1).reshape(2, 2, B, n, n, C)
    return layer, ti, ti[:, :1, :2, :2].contiguous(), want.permute(2, 3, 0, 4, 1, 5).reshape(B, 2 * n, 2 * n, C)


LAYERS = [("fp32", 256), ("bf16", 512)]


def close(y, want):   # sums of at most 512 products in fp32, from the same operands
    return (y.double() - want).norm() <= 1e-6 * want.norm()


@pytest.mark.parametrize("precision,C", LAYERS)
@pytest.mark.parametrize("warm", [True, False])
@pytest.mark.parametrize("external", [True, False])
def test_kept_weights_are_there_on_every_stream(precision, C, warm, external):
    """What a layer keeps is made on the stream of the call that first wants it; a call on another stream may follow at once."""
    layer, ti, small, want = masked_layer(precision, C)
    busy = torch.ones((4096, 4096), device="cuda")
    with torch.no_grad():
        if warm:
            layer(small)
        assert layer._pieces is None
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream() for _ in range(3)]
        if external:   # a stream that is not torch's
            import ctypes
            hip, handle = ctypes.CDLL("libamdhip64.so.7"), ctypes.c_void_p()
            assert hip.hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0
            streams[0] = torch.cuda.ExternalStream(handle.value)
        with torch.cuda.stream(streams[0]):
            for _ in range(20):
                busy = torch.mm(busy, busy).clamp_(max=1)
            outputs = [layer(ti), layer(ti)]
        for s in streams[1:]:
            with torch.cuda.stream(s):
                outputs.append(layer(ti))
        torch.cuda.synchronize()
        outputs.append(layer(ti))
        assert all(close(y, want) for y in outputs)
        layer.W.mul_(1)   # makes anew, and drops what other streams have read
        with torch.cuda.stream(streams[1]):
            assert close(layer(ti), want) and close(layer(ti), want)
        torch.cuda.synchronize()


@pytest.mark.parametrize("precision,C", LAYERS)
@pytest.mark.parametrize("warm", [True, False])
def test_a_capture_keeps_no_weights(precision, C, warm):
    """Weights that a capture would make are written when the graph runs: nothing of them may be kept for eager calls.  What eager
    calls kept before is used in a capture."""
    layer, ti, small, want = masked_layer(precision, C)
    with torch.no_grad():
        if warm:
            layer(small)
        torch.cuda.synchronize()
        for kept in (False, True):
            before = layer._masked, layer._pieces
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                y = layer(ti)
            assert (layer._masked, layer._pieces) == before and (layer._pieces is None) == (not kept)
            assert close(layer(ti), want)
            for _ in range(3):
                y.zero_()
                graph.replay()
                layer(small)
                torch.cuda.synchronize()
                assert close(y, want)
            layer(ti)


def test_a_copied_layer_brings_no_kept_weights():
    import copy
    import pickle
    layer, ti, _, want = masked_layer("fp32", 256)
    with torch.no_grad():
        layer(ti)
        assert layer._masked is not None
        for other in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer))):
            assert (other._masked, other._bf16, other._pieces) == (None, None, None)
            assert close(other(ti), want)
        state = dict(layer.__getstate__(), _masked=(b"", torch.zeros_like(layer.W)), _pieces=None)   # as layers kept them before
        other.__setstate__(state)
        assert close(other(ti), want)


@pytest.mark.parametrize("precision,C", [("fp32", 512), ("bf16", 512)])
def test_a_layer_repeats_itself(precision, C):
    """The first call on new weights, later ones and one that is captured: the same bits, whether one call pays for the pieces or not."""
    import swc_hip
    from winograd_conv import WinogradConv
    gen = torch.Generator(device="cuda").manual_seed(30)
    layer = WinogradConv(C, C, mask=(torch.rand((16, C, C), device="cuda", generator=gen) < 0.3).float(), device="cuda", precision=precision)
    ti = torch.randn((16, 64, 4, 4, C), device="cuda", generator=gen).relu_()
    with torch.no_grad():
        for _ in range(2):
            first = layer(ti)
            if torch.cuda.get_device_properties(0).multi_processor_count == 256:
                assert swc_hip.lib().swc_winograd2x2_conv_last_form() == b"pieces32"
            assert torch.equal(layer(ti), first)
            layer.refresh()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                y = layer(ti)
            for _ in range(3):
                y.zero_()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(y, first)
            layer.W.mul_(2)
