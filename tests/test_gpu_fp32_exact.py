"""The fp32 convolution computes with fp32 operands whatever the values around them are, on every kernel the launcher picks:
scaling by powers of two commutes with it bit for bit, and what fp32 represents exactly comes out exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (B, nH, nW, C, K) and what runs on 256 CUs
SHAPES = [((1, 8, 8, 64, 64), "direct16x16"), ((16, 7, 7, 256, 256), "direct16x64"), ((63, 14, 14, 36, 120), "direct32x64"),
          ((18, 19, 24, 32, 32), "ring32"), ((64, 14, 14, 48, 64), "ring16"), ((32, 28, 28, 64, 64), "tall16"),
          ((96, 22, 8, 64, 32), "short16"), ((15, 12, 23, 64, 384), "wide48"), ((64, 14, 14, 64, 64), "wide48x64"),
          ((16, 7, 7, 512, 512), "split32"), ((41, 18, 12, 64, 32), "split48"), ((64, 7, 7, 256, 256), "split64"),
          ((49, 30, 27, 96, 36), "split64+32"), ((128, 7, 7, 256, 256), "split64+48"), ((2, 4, 4, 5, 7), "sync")]


def ran():
    import swc_hip
    return swc_hip.lib().swc_winograd2x2_conv_last_kernel().decode()


def conv(ti, w):
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    return winograd2x2_conv(ti, w)


@pytest.mark.parametrize("shape,kernel", SHAPES)
@pytest.mark.parametrize("positive", [False, True])
def test_scaling_by_powers_of_two_commutes(shape, kernel, positive):
    """Rows of TI and columns of W down to 2^-50 of the others beside them, and channels whose activations and weights
    compensate each other: each product and sum is the unscaled one times a power of two, so nothing may round differently.
    (Over 2^30 the split forms multiply with the fp32 instructions, whose sums are those of the direct form.)"""
    B, nH, nW, C, K = shape
    gen = torch.Generator(device="cuda").manual_seed(75)
    ti = torch.randn((16, B, nH, nW, C), device="cuda", generator=gen)
    w = torch.randn((16, C, K), device="cuda", generator=gen)
    if positive:
        ti, w = ti.abs_(), w.abs_()
    else:
        ti.relu_()
    plain = conv(ti, w)
    got_kernel = ran()
    powers = torch.tensor([0, 0, -24, 0, -28, -34, 0, -44, -46, 0, -50], device="cuda")
    pick = lambda n: 2.0 ** powers[torch.arange(n, device="cuda") % len(powers)].double()   # noqa: E731
    rows = pick(B * nH * nW).float()
    by_pixel = rows.reshape(B, nH, 1, nW, 1, 1).expand(B, nH, 2, nW, 2, 1).reshape(B, 2 * nH, 2 * nW, 1)
    by_rows = torch.equal(conv(ti * rows.reshape(1, B, nH, nW, 1), w), plain * by_pixel)
    cols = pick(K).float()
    by_columns = torch.equal(conv(ti, w * cols), plain * cols)
    wide = torch.arange(C, device="cuda") * 7 % 81 - 40
    channels = (2.0 ** (wide / 2).round().double()).float()
    by_channels = torch.equal(conv(ti * channels, w / channels.reshape(C, 1)), plain)
    channels = (2.0 ** wide.double()).float()
    far = conv(ti * channels, w / channels.reshape(C, 1))
    if got_kernel.startswith("split"):
        import swc_hip
        assert swc_hip.lib().swc_winograd2x2_conv_force_tiling(b"direct32x64") == 0
        try:
            plain = conv(ti, w)
        finally:
            assert swc_hip.lib().swc_winograd2x2_conv_force_tiling(None) == 0
    by_channels_far = torch.equal(far, plain)
    assert by_rows and by_columns and by_channels and by_channels_far, (by_rows, by_columns, by_channels, by_channels_far)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert got_kernel == kernel


@pytest.mark.parametrize("shape,kernel", SHAPES)
def test_all_24_bits_of_an_operand_count(shape, kernel):
    B, nH, nW, C, K = shape
    gen = torch.Generator(device="cuda").manual_seed(76)

    def one_channel(ti_bits, w_bits):
        ti, w = torch.zeros((16, B, nH, nW, C), device="cuda"), torch.zeros((16, C, K), device="cuda")
        lo, hi = 2 ** (ti_bits - 1), 2 ** ti_bits
        a = torch.randint(lo, hi, (B, nH, nW), device="cuda", generator=gen) | 1
        b = torch.randint(2 ** (w_bits - 1), 2 ** w_bits, (K,), device="cuda", generator=gen) | 1
        ti[5, ..., 1], w[5, 1] = a.float(), b.float()
        y = conv(ti, w)
        want = (a.double().unsqueeze(-1) * b.double()).float()     # position 5 enters all four outputs with a plus
        for dy in (0, 1):
            for dx in (0, 1):
                same = torch.equal(y[:, dy::2, dx::2], want)
                assert same, (ti_bits, w_bits)

    one_channel(24, 1)      # weights of 1: the activations come back
    one_channel(1, 24)
    one_channel(12, 12)     # products of 24 bits
