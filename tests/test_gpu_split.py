"""The convolution with the positions split over eight waves (fp32 operands in three bf16 pieces, or bf16 operands): each
tile height forced at the edges of its tiles and steps, its error against float64 beside the fp32 instructions', and the
operands that those multiply instead."""
import numpy as np
import pytest
import torch

from test_gpu_direct import bound, forced, tiles_of  # noqa: F401

pytestmark = pytest.mark.gpu

FORMS = ["split32", "split48", "split64", "split64+32", "split64+48"]
# "split64+32" forced takes half of the whole 64-row tiles and leaves the rest to 32-row ones.
# (B, nH, nW, C, K): M = 1, 17, 33, 49, 65, 130, 255 rows; C below, at and past a step of 32 indices; K below, at and past 64;
# the last two have more columns than rows (column tiles are numbered the other way round)
SHAPES = [(1, 1, 1, 4, 4), (1, 1, 17, 36, 20), (3, 1, 11, 64, 68), (1, 7, 7, 100, 132), (1, 5, 13, 28, 64), (2, 5, 13, 160, 36), (1, 15, 17, 64, 132),
          (1, 7, 10, 64, 200), (1, 10, 13, 32, 260)]


@pytest.mark.parametrize("form,precision", [(f, "fp32") for f in FORMS] + [(f, "bf16") for f in FORMS[:3]])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_forms(oracle, forced, form, precision, shape):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    B, nH, nW, C, K = shape
    rng = np.random.default_rng(71)
    ti = np.maximum(rng.standard_normal((16, B, nH, nW, C)), 0).astype(np.float32)
    w = (rng.standard_normal((16, C, K)) * 0.05).astype(np.float32)
    tii = rng.integers(-4, 5, size=ti.shape).astype(np.float32)
    wi = rng.integers(-4, 5, size=w.shape).astype(np.float32)
    scale, shift = rng.standard_normal(K).astype(np.float32), rng.standard_normal(K).astype(np.float32)
    res = rng.standard_normal((B, 2 * nH, 2 * nW, K)).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()
    assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
    got = winograd2x2_conv(dev(ti), dev(w), precision=precision).cpu().numpy()
    assert forced.swc_winograd2x2_conv_last_form().decode() == form
    exact = winograd2x2_conv(dev(tii), dev(wi), precision=precision).cpu().numpy()
    ep = winograd2x2_conv(dev(ti), dev(w), precision=precision, scale=dev(scale), shift=dev(shift), residual=dev(res),
                          residual_relu=True).cpu().numpy()
    buf = dev(res)
    winograd2x2_conv(dev(ti), dev(w), precision=precision, out=buf, residual=buf)   # residual aliasing the output
    if precision == "bf16":
        ti, w = oracle.round_bf16(ti), oracle.round_bf16(w)
    want = oracle.conv(ti, w, acc64=True)
    err = np.abs(tiles_of(got, nH, nW).astype(np.float64) - tiles_of(want, nH, nW))
    # the fp32 instructions' bound, and one more rounding a product for the products of pieces that are left out
    more = 1 + 1 / (w.shape[1] + 8)
    assert (err <= more * bound(ti, w)[:, None, :] + 2.0 ** -24 * np.abs(tiles_of(want, nH, nW))).all()
    assert np.array_equal(exact, oracle.conv(tii, wi))
    assert np.array_equal(ep, oracle.affine(got, scale, shift) + np.maximum(res, 0))
    assert np.array_equal(buf.cpu().numpy(), got + res)


def test_infinities_and_nan_stay_where_they_are_with_bf16_operands(forced):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(73)
    ti = torch.randn((16, 1, 8, 8, 96), device="cuda", generator=gen).relu_()
    w = torch.randn((16, 96, 64), device="cuda", generator=gen) * 0.05
    ti[3, 0, 2, 5, 40], ti[5, 0, 7, 7, 95], w[9, 70, 11] = float("inf"), float("nan"), float("-inf")
    out = {}
    for form in FORMS[:3] + ["direct32x64"]:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        out[form] = winograd2x2_conv(ti, w, precision="bf16")
    want = out.pop("direct32x64")
    finite = torch.isfinite(want)
    for form, got in out.items():
        assert torch.equal(torch.isnan(got), torch.isnan(want)), form
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]), form
        assert (got[finite] - want[finite]).abs().max() <= 1e-5 * want[finite].abs().max(), form


@pytest.mark.parametrize("C", [64, 72, 128, 256, 512])
@pytest.mark.parametrize("density", [0.1, 0.3, 1.0])
@pytest.mark.parametrize("magnitude", [(1.0, 0.05), (1e-6, 1e-5), (3e4, 20.0)])
def test_no_further_from_float64_than_the_fp32_instructions(forced, C, density, magnitude):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(72)
    ti = torch.randn((16, 4, 16, 16, C), device="cuda", generator=gen).relu_() * magnitude[0]
    w = torch.randn((16, C, 128), device="cuda", generator=gen)
    w *= magnitude[1] * (w.abs() >= w.abs().flatten()[::7].quantile(1 - density))     # the largest are kept
    p = torch.bmm(ti.reshape(16, -1, C).double(), w.double()).reshape(4, 4, -1, 128)
    rows = torch.stack([p[0] + p[1] + p[2], p[1] - p[2] - p[3]])
    want = torch.stack([rows[:, 0] + rows[:, 1] + rows[:, 2], rows[:, 1] - rows[:, 2] - rows[:, 3]], 1)   # [dy,dx,M,K]
    want = want.reshape(2, 2, 4, 16, 16, 128).permute(2, 3, 0, 4, 1, 5).reshape(4, 32, 32, 128)
    errors = {}
    for form in FORMS + ["direct16x64"]:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        errors[form] = ((winograd2x2_conv(ti, w).double() - want).norm() / want.norm()).item()
        assert forced.swc_winograd2x2_conv_last_form().decode() == form
    # with few products (64 channels at 10 %) the outputs' own nine-term sums make most of either's error: equal to 1 %
    assert all(errors[f] <= 1.01 * errors["direct16x64"] for f in FORMS), errors


def test_operands_left_to_the_fp32_instructions(forced):  # noqa: F811
    """Infinities, NaN, operands above 2^30, sums below 2^-75: the position is multiplied with the fp32 instructions, so the
    result is the one-position-per-wave fp32 kernel's, which sums in the same order."""
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(73)
    ti0 = torch.randn((16, 1, 8, 8, 96), device="cuda", generator=gen).relu_()
    w0 = torch.randn((16, 96, 64), device="cuda", generator=gen) * 0.05

    def case(name):
        ti, w = ti0.clone(), w0.clone()
        if name == "infinite":
            ti[3, 0, 2, 5, 40] = float("inf")
            w[9, 70, 11] = float("-inf")
        elif name == "nan":
            ti[5, 0, 7, 7, 95] = float("nan")
        elif name == "late outlier":
            ti[:, :, :, :, 64:] *= 1e12
        elif name == "large weights, tiny activations":
            w *= 1e34
            ti *= 1e-34
        elif name == "large activations, tiny weights":
            ti *= 1e34
            w *= 1e-34
        elif name == "tiny":
            ti *= 1e-20
            w *= 1e-10
        elif name == "next to infinity":
            ti[:, 0, 3, 3, 10], w[:, 10] = 3.4e38, 1e-30
        return ti, w

    for name in ("infinite", "nan", "late outlier", "large weights, tiny activations", "large activations, tiny weights", "tiny",
                 "next to infinity"):
        ti, w = case(name)
        out = {}
        for form in FORMS + ["direct32x64"]:
            assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
            out[form] = winograd2x2_conv(ti, w)
        want = out.pop("direct32x64")
        finite = torch.isfinite(want)
        for form, got in out.items():
            assert torch.equal(torch.isnan(got), torch.isnan(want)), (name, form)
            if name in ("infinite", "nan"):      # the other positions are not bit-equal
                inf = torch.isinf(want)
                assert torch.equal(got[inf], want[inf]), (name, form)
                assert (got[finite] - want[finite]).abs().max() <= 1e-5 * want[finite].abs().max(), (name, form)
            elif name == "next to infinity":     # nor are the tiles without that row
                rest = torch.ones_like(got, dtype=torch.bool)
                rest[0, 6:8, 6:8] = False
                assert torch.equal(got[~rest], want[~rest]), (name, form)
                assert (got[rest] - want[rest]).abs().max() <= 1e-5 * want[rest].abs().max(), (name, form)
            else:
                same = torch.equal(got, want)
                assert same, (name, form)


def test_blank_data_is_not_multiplied_twice(forced):  # noqa: F811
    """Zeros in the first channels, whole rows and columns of zeros: nothing to look at again, and the same values as without
    the blank parts around them."""
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(78)
    ti = torch.randn((16, 1, 8, 8, 128), device="cuda", generator=gen).relu_()
    w = torch.randn((16, 128, 64), device="cuda", generator=gen)
    ti[..., :64] = 0
    ti[:, :, 4:] = 0
    w[:, :, 10:30] = 0
    for form in FORMS:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        got = winograd2x2_conv(ti, w)
        assert (got[:, 8:] == 0).all() and (got[..., 10:30] == 0).all()
        alone = winograd2x2_conv(ti[..., 64:].contiguous(), w[:, 64:].contiguous())
        same = torch.equal(got, alone)
        assert same, form


def test_unaligned_output_or_residual_takes_another_kernel(forced):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(77)
    ti, w = torch.randn((16, 16, 7, 7, 512), device="cuda", generator=gen), torch.randn((16, 512, 512), device="cuda", generator=gen)
    want = winograd2x2_conv(ti, w, precision="bf16")
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert forced.swc_winograd2x2_conv_last_form() == b"split32"
    n = want.numel()
    off = torch.zeros(2 * n + 2, device="cuda")
    out, res = off[1:1 + n].view(want.shape), off[1 + n:1 + 2 * n].view(want.shape)
    for kw in ({"out": out}, {"residual": res}):
        got = winograd2x2_conv(ti, w, precision="bf16", **kw)
        assert not forced.swc_winograd2x2_conv_last_form().startswith(b"split")
        # fp32 sums of the same 512 products and nine terms in another order
        assert (got - want).norm() <= 1e-5 * want.norm()
