"""The bf16-operand convolution with the positions split over eight waves: each tile height forced at the edges of its
tiles and steps."""
import numpy as np
import pytest
import torch

from test_gpu_direct import bound, forced, tiles_of  # noqa: F401

pytestmark = pytest.mark.gpu

FORMS = ["split32", "split48", "split64"]
# (B, nH, nW, C, K): M = 1, 17, 33, 49, 65, 130, 255 rows; C below, at and past a step of 32 indices; K below, at and past 64;
# the last one has more columns than rows (column tiles are numbered the other way round)
SHAPES = [(1, 1, 1, 4, 4), (1, 1, 17, 36, 20), (3, 1, 11, 64, 68), (1, 7, 7, 100, 132), (1, 5, 13, 28, 64), (2, 5, 13, 160, 36), (1, 15, 17, 64, 132),
          (1, 7, 10, 64, 200)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
def test_split_forms(oracle, forced, form, shape):  # noqa: F811
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
    got = winograd2x2_conv(dev(ti), dev(w), precision="bf16").cpu().numpy()
    assert forced.swc_winograd2x2_conv_last_form().decode() == form
    exact = winograd2x2_conv(dev(tii), dev(wi), precision="bf16").cpu().numpy()
    ep = winograd2x2_conv(dev(ti), dev(w), precision="bf16", scale=dev(scale), shift=dev(shift), residual=dev(res),
                          residual_relu=True).cpu().numpy()
    buf = dev(res)
    winograd2x2_conv(dev(ti), dev(w), precision="bf16", out=buf, residual=buf)   # residual aliasing the output
    ti, w = oracle.round_bf16(ti), oracle.round_bf16(w)
    want = oracle.conv(ti, w, acc64=True)
    err = np.abs(tiles_of(got, nH, nW).astype(np.float64) - tiles_of(want, nH, nW))
    assert (err <= bound(ti, w)[:, None, :] + 2.0 ** -24 * np.abs(tiles_of(want, nH, nW))).all()
    assert np.array_equal(exact, oracle.conv(tii, wi))
    assert np.array_equal(ep, oracle.affine(got, scale, shift) + np.maximum(res, 0))
    assert np.array_equal(buf.cpu().numpy(), got + res)


def test_infinities_and_nan_stay_where_they_are(forced):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(73)
    ti = torch.randn((16, 1, 8, 8, 96), device="cuda", generator=gen).relu_()
    w = torch.randn((16, 96, 64), device="cuda", generator=gen) * 0.05
    ti[3, 0, 2, 5, 40], ti[5, 0, 7, 7, 95], w[9, 70, 11] = float("inf"), float("nan"), float("-inf")
    out = {}
    for form in FORMS + ["direct32x64"]:
        assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
        out[form] = winograd2x2_conv(ti, w, precision="bf16")
    want = out.pop("direct32x64")
    finite = torch.isfinite(want)
    for form, got in out.items():
        assert torch.equal(torch.isnan(got), torch.isnan(want)), form
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]), form
        assert (got[finite] - want[finite]).abs().max() <= 1e-5 * want[finite].abs().max(), form


def test_forced_on_fp32_operands_they_are_refused(forced):  # noqa: F811
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    ti, w = torch.ones((16, 1, 8, 8, 64), device="cuda"), torch.ones((16, 64, 64), device="cuda")
    assert forced.swc_winograd2x2_conv_force_tiling(b"split64") == 0
    winograd2x2_conv(ti, w)
    assert forced.swc_winograd2x2_conv_last_form() == b"whole" and forced.swc_winograd2x2_conv_last_kernel() == b"sync"


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
