"""The convolution on the 16-bit matrix instructions (fp32 operands as pairs of f16 values, or bf16 operands): each tile
height forced at the edges of its tiles and steps, its error against float64 beside the fp32 instructions', and operands
that do not split."""
import numpy as np
import pytest
import torch

from test_gpu_direct import forced, tiles_of  # noqa: F401

pytestmark = pytest.mark.gpu

FORMS = ["split32", "split48", "split64"]
# (B, nH, nW, C, K): M = 1, 17, 33, 49, 65, 130 rows; C below, at and past a step of 32 indices; K below, at and past 64
SHAPES = [(1, 1, 1, 4, 4), (1, 1, 17, 36, 20), (3, 1, 11, 64, 68), (1, 7, 7, 100, 132), (1, 5, 13, 28, 64), (2, 5, 13, 160, 36)]


def bound(ti, w):
    """(C + 8) roundings of fp32 sums of at most half a unit, as for the fp32 instructions, and what a product loses:
    2^-22 of it per operand (a value is taken to 23 bits and a sign, half a unit of which is below that) and as much
    for the product of the low parts."""
    C = w.shape[1]
    mag = np.einsum("imc,ick->mk", np.abs(ti).reshape(16, -1, C).astype(np.float64), np.abs(w).astype(np.float64))
    return (C + 8 + 12) * 2.0 ** -24 * mag


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_split_forms(oracle, forced, form, shape, precision):  # noqa: F811
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
    if precision == "bf16":
        ti, w = oracle.round_bf16(ti), oracle.round_bf16(w)
    want = oracle.conv(ti, w, acc64=True)
    err = np.abs(tiles_of(got, nH, nW).astype(np.float64) - tiles_of(want, nH, nW))
    assert (err <= bound(ti, w)[:, None, :] + 2.0 ** -24 * np.abs(tiles_of(want, nH, nW))).all()
    assert np.array_equal(exact, oracle.conv(tii, wi))
    assert np.array_equal(ep, oracle.affine(got, scale, shift) + np.maximum(res, 0))


@pytest.mark.parametrize("C", [64, 72, 128, 256, 512])
@pytest.mark.parametrize("magnitude", [(1.0, 0.05), (1e-6, 1e-5), (3e4, 20.0)])
def test_no_further_from_float64_than_the_fp32_instructions(forced, C, magnitude):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(72)
    ti = torch.randn((16, 4, 16, 16, C), device="cuda", generator=gen).relu_() * magnitude[0]
    w = torch.randn((16, C, 128), device="cuda", generator=gen) * magnitude[1]
    p = torch.bmm(ti.reshape(16, -1, C).double(), w.double()).reshape(4, 4, -1, 128)
    rows = torch.stack([p[0] + p[1] + p[2], p[1] - p[2] - p[3]])
    want = torch.stack([rows[:, 0] + rows[:, 1] + rows[:, 2], rows[:, 1] - rows[:, 2] - rows[:, 3]], 1)   # [dy,dx,M,K]
    want = want.reshape(2, 2, 4, 16, 16, 128).permute(2, 3, 0, 4, 1, 5).reshape(4, 32, 32, 128)
    errors = {}
    for form in FORMS + ["ring32"]:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        errors[form] = ((winograd2x2_conv(ti, w).double() - want).norm() / want.norm()).item()
    assert all(errors[f] <= errors["ring32"] for f in FORMS), errors


def test_operands_that_do_not_split(forced):  # noqa: F811
    """Infinities, NaN, values beyond f16's range around the first step's, a first step of zeros, magnitudes out of the
    scale's range: the tile is multiplied with the fp32 instructions, so the result is the one-position-per-wave fp32
    kernel's, which sums in the same order."""
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
            ti[:, :, :, :, 64:] *= 1e6
        elif name == "zeros first":
            ti[..., :32] = 0
            ti *= 1e-12
        elif name == "zero weights first":
            w[:, :32] = 0
            w *= 1e-12
        elif name == "tiny":
            ti *= 1e-30
        elif name == "huge":
            w *= 1e30
        return ti, w

    for name in ("infinite", "nan", "late outlier", "zeros first", "zero weights first", "tiny", "huge"):
        ti, w = case(name)
        out = {}
        for form in ("split64", "split48", "split32", "direct32x64"):
            assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
            out[form] = winograd2x2_conv(ti, w)
        want = out.pop("direct32x64")
        finite = torch.isfinite(want)
        for form, got in out.items():
            assert torch.equal(torch.isnan(got), torch.isnan(want)), (name, form)
            if name in ("infinite", "nan"):      # the positions that split are not bit-equal
                inf = torch.isinf(want)
                assert torch.equal(got[inf], want[inf]), (name, form)
                assert (got[finite] - want[finite]).abs().max() <= 1e-5 * want[finite].abs().max(), (name, form)
            else:
                assert torch.equal(got, want), (name, form)


def test_rows_and_columns_of_any_size_beside_each_other(forced):  # noqa: F811
    """Rows of TI and columns of W from 1 down to 2^-20 of the largest keep the accuracy they have by themselves."""
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(74)
    ti = torch.randn((16, 1, 8, 8, 128), device="cuda", generator=gen)
    w = torch.randn((16, 128, 64), device="cuda", generator=gen)
    assert forced.swc_winograd2x2_conv_force_tiling(b"split64") == 0
    plain = winograd2x2_conv(ti, w)
    rows = 2.0 ** -torch.arange(64, device="cuda").remainder(21).float()     # powers of two: exact in fp32
    cols = 2.0 ** -torch.arange(64, device="cuda").remainder(19).float()
    got = winograd2x2_conv(ti * rows.reshape(1, 1, 8, 8, 1), w * cols)
    by = rows.reshape(1, 8, 1, 8, 1, 1).expand(1, 8, 2, 8, 2, 1).reshape(1, 16, 16, 1) * cols
    err = ((got / by - plain).reshape(256, 64).norm(dim=0) / plain.reshape(256, 64).norm(dim=0)).max()
    assert err <= 1e-6, err      # two correct fp32 results of 128 products and nine sums differ by about 2e-7
