"""The small-grid form of the convolution (sixteen waves per workgroup, one per position): each tile shape forced at the
edges of its tiles and of its blocks of reduction indices, and what the launcher picks by itself."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

FORMS = ["direct16x16", "direct16x32", "direct16x64", "direct32x64"]
# (B, nH, nW, C, K): M = 1, 15, 16, 17, 33, 49 rows; C below, at and past a block of 16, 32 or 64 indices; K below, at and
# past a tile, and no multiple of 16
SHAPES = [(1, 1, 1, 4, 4), (1, 3, 5, 16, 16), (1, 4, 4, 32, 64), (1, 1, 17, 36, 20), (3, 1, 11, 64, 68), (1, 7, 7, 100, 132),
          (2, 5, 5, 132, 36)]


def bound(ti, w):
    """What fp32 sums of C products and then nine of them may be off by: (C + 8) roundings of at most half a unit,
    each of a partial sum no larger than the sum of all magnitudes."""
    C = w.shape[1]
    mag = np.einsum("imc,ick->mk", np.abs(ti).reshape(16, -1, C).astype(np.float64), np.abs(w).astype(np.float64))
    return (C + 8) * 2.0 ** -24 * mag      # per tile row and column: all 16 positions, an output has nine


def tiles_of(y, nH, nW):                    # [B,2nH,2nW,K] -> [M,4,K]
    B, _, _, K = y.shape
    return y.reshape(B, nH, 2, nW, 2, K).transpose(0, 1, 3, 2, 4, 5).reshape(B * nH * nW, 4, K)


@pytest.fixture
def forced():
    import swc_hip
    L = swc_hip.lib()
    yield L
    assert L.swc_winograd2x2_conv_force_tiling(None) == 0


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_direct_forms(oracle, forced, form, shape, precision):
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    B, nH, nW, C, K = shape
    rng = np.random.default_rng(61)
    ti = np.maximum(rng.standard_normal((16, B, nH, nW, C)), 0).astype(np.float32)
    w = (rng.standard_normal((16, C, K)) * 0.05).astype(np.float32)
    tii = rng.integers(-4, 5, size=ti.shape).astype(np.float32)
    wi = rng.integers(-4, 5, size=w.shape).astype(np.float32)
    scale, shift = rng.standard_normal(K).astype(np.float32), rng.standard_normal(K).astype(np.float32)
    res = rng.standard_normal((B, 2 * nH, 2 * nW, K)).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()
    assert forced.swc_winograd2x2_conv_force_tiling(form.encode()) == 0
    got = winograd2x2_conv(dev(ti), dev(w), precision=precision).cpu().numpy()
    assert forced.swc_winograd2x2_conv_last_form().decode() == forced.swc_winograd2x2_conv_last_kernel().decode() == form
    exact = winograd2x2_conv(dev(tii), dev(wi), precision=precision).cpu().numpy()
    ep = winograd2x2_conv(dev(ti), dev(w), precision=precision, scale=dev(scale), shift=dev(shift), residual=dev(res),
                          residual_relu=True).cpu().numpy()
    buf = dev(res)
    winograd2x2_conv(dev(ti), dev(w), precision=precision, out=buf, residual=buf)   # residual aliasing the output
    off = torch.zeros(2 * res.size + 2, device="cuda")                              # output and residual 4 bytes past a line
    out, shifted = off[1:1 + res.size].view(res.shape), off[1 + res.size:1 + 2 * res.size].view(res.shape)
    shifted.copy_(dev(res))
    winograd2x2_conv(dev(ti), dev(w), precision=precision, out=out, residual=shifted)
    assert forced.swc_winograd2x2_conv_last_form().decode() == form
    assert np.array_equal(buf.cpu().numpy(), got + res) and np.array_equal(out.cpu().numpy(), got + res)
    if precision == "bf16":
        ti, w = oracle.round_bf16(ti), oracle.round_bf16(w)
    want = oracle.conv(ti, w, acc64=True)
    err = np.abs(tiles_of(got, nH, nW).astype(np.float64) - tiles_of(want, nH, nW))
    assert (err <= bound(ti, w)[:, None, :] + 2.0 ** -24 * np.abs(tiles_of(want, nH, nW))).all()
    assert np.array_equal(exact, oracle.conv(tii, wi))
    assert np.array_equal(ep, oracle.affine(got, scale, shift) + np.maximum(res, 0))


@pytest.mark.parametrize("C", [32, 36, 40, 60, 64, 96, 100, 124, 128, 176])
def test_bf16_single_tiles_with_every_end_of_a_block(forced, C):
    # Blocks of 32 indices that are turned round in LDS, and blocks of 64 that are not where C ends in the second half of one.  Whole
    # numbers are exact in bf16 and in any order of the sums.
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    gen = torch.Generator(device="cuda").manual_seed(63)
    ti = torch.randint(-4, 5, (16, 1, 7, 11, C), device="cuda", generator=gen).float()
    w = torch.randint(-4, 5, (16, C, 36), device="cuda", generator=gen).float()
    assert forced.swc_winograd2x2_conv_force_tiling(b"direct16x16") == 0
    got = winograd2x2_conv(ti, w, "bf16")
    assert forced.swc_winograd2x2_conv_last_form() == b"direct16x16"
    p = torch.matmul(ti.reshape(16, -1, C).double().cpu(), w.double().cpu()).reshape(4, 4, 7, 11, 36)
    a = torch.tensor([[1, 1, 1, 0], [0, 1, -1, -1]], dtype=torch.float64)
    want = torch.einsum("ai,bj,ijhwk->hawbk", a, a, p).reshape(1, 14, 22, 36)
    assert torch.equal(got.cpu().double(), want)


@pytest.mark.parametrize("shape,precision,want", [
    ((1, 8, 8, 64, 64), "fp32", "direct16x16"),       # 16 tiles of 16x16
    ((5, 14, 16, 96, 72), "fp32", "direct16x32"),     # 350 tiles of 16x16, 210 of 16x32
    ((16, 7, 7, 256, 256), "fp32", "direct16x64"),
    ((63, 14, 14, 36, 120), "fp32", "direct32x64"),   # below 64 channels
    ((16, 7, 7, 512, 512), "fp32", "split32"),        # 200 tiles of 32x64
    ((64, 7, 7, 256, 256), "fp32", "split64"),        # 196 tiles of 64x64
    ((128, 7, 7, 256, 256), "fp32", "split64+48"),    # 392: one round, the rest in 184 lower ones
    ((49, 30, 27, 96, 36), "fp32", "split64+32"),     # 621: two rounds, and 6922 rows in lower tiles
    ((64, 14, 14, 128, 128), "fp32", "whole"),        # 392 too, but 128 channels: wide48 is as fast
    ((64, 28, 28, 64, 64), "fp32", "whole"),          # 64 channels and more than a round
    ((16, 7, 7, 512, 512), "bf16", "split32"),
    ((64, 7, 7, 256, 256), "bf16", "split64"),        # 196 tiles of 64x64
    ((64, 14, 14, 128, 128), "bf16", "whole"),        # 392
    ((64, 14, 14, 32, 64), "bf16", "whole"),          # below 64 channels the ring takes less
    # channels that are no multiple of 32, which no ring kernel takes: a round behind the first counts as what it takes
    ((18, 16, 16, 72, 384), "bf16", "direct32x64"),   # 4 rounds, 16x64 tiles would be 7
    ((1, 5483, 1, 208, 256), "bf16", "direct32x64"),  # 3 and 6
    ((1, 2427, 1, 100, 96), "bf16", "split32"),       # 1 round, 16x32 tiles 2
    ((1, 14094, 1, 72, 128), "bf16", "direct32x64"),  # 4 and 7
])
def test_the_launcher_picks_the_smallest_tile_that_needs_one_round(forced, shape, precision, want):
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the picks are those of 256 CUs")
    B, nH, nW, C, K = shape
    winograd2x2_conv(torch.ones((16, B, nH, nW, C), device="cuda"), torch.ones((16, C, K), device="cuda"), precision=precision)
    assert forced.swc_winograd2x2_conv_last_form().decode() == want


def test_odd_columns_and_unaligned_weights_take_single_columns(oracle, forced):
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    rng = np.random.default_rng(62)
    ti = np.maximum(rng.standard_normal((16, 1, 5, 9, 20)), 0).astype(np.float32)
    for K, off in ((7, 0), (16, 1)):
        w = (rng.standard_normal((16, 20, K)) * 0.05).astype(np.float32)
        buf = torch.zeros(w.size + 4, device="cuda")
        wd = buf[off:off + w.size].view(w.shape)
        wd.copy_(torch.from_numpy(w))
        got = winograd2x2_conv(torch.from_numpy(ti).cuda(), wd).cpu().numpy()
        assert forced.swc_winograd2x2_conv_last_form() == b"direct16x16"
        want = oracle.conv(ti, w, acc64=True)
        err = np.abs(tiles_of(got, 5, 9).astype(np.float64) - tiles_of(want, 5, 9))
        assert (err <= bound(ti, w)[:, None, :] + 2.0 ** -24 * np.abs(tiles_of(want, 5, 9))).all()


def test_the_form_is_that_of_the_last_call(forced):
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    ti, w = torch.zeros((16, 1, 8, 8, 64), device="cuda"), torch.zeros((16, 64, 64), device="cuda")
    winograd2x2_conv(ti, w)
    assert forced.swc_winograd2x2_conv_last_form() == forced.swc_winograd2x2_conv_last_kernel() == b"direct16x16"
    winograd2x2_conv(ti.bfloat16(), w)
    assert forced.swc_winograd2x2_conv_last_form() == b"whole" and forced.swc_winograd2x2_conv_last_kernel().startswith(b"stored-")
