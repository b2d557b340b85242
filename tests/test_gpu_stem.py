"""conv1 + pool1 of the model in one kernel, against float64."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def expected(image, w):
    import resnet18_var
    x = image.permute(0, 3, 1, 2)
    x = F.conv2d(F.pad(x, resnet18_var._same_pad(x, 7, 2)), w, stride=2)
    return resnet18_var._max_pool_same(x).permute(0, 2, 3, 1)


# one pixel; below, at and past a tile of 7x7 pooled pixels (28 of the image); odd sides (the padding moves to the other
# side); more tiles than CUs (ones fetched ahead)
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 5, 7), (1, 28, 28), (3, 29, 31), (2, 27, 57), (1, 56, 58), (2, 225, 226), (8, 224, 224)])
@pytest.mark.parametrize("scale", [1.0, 255.0, 1e-6])
def test_against_float64(shape, scale):
    import resnet18_var
    gen = torch.Generator().manual_seed(81)
    image = torch.randn(shape + (3,), generator=gen) * scale
    w = torch.randn((64, 3, 7, 7), generator=gen) * torch.logspace(-4, 0, 64).reshape(64, 1, 1, 1)
    got = resnet18_var.stem_conv_pool(image.cuda(), w.cuda()).cpu()
    want = expected(image.double(), w.double())
    assert got.shape == want.shape
    # 147 products: fp32 sums of them in any order are within 147 half units of the sum of magnitudes, a product within one
    # more; typical errors are far smaller, so the norm is held to 1e-6
    mag = expected_magnitude(image, w)
    assert ((got - want).abs() <= (147 + 1 + 4) * 2.0 ** -24 * mag).all()
    assert (got - want).norm() <= 1e-6 * want.norm()
    ints = torch.randint(-8, 9, shape + (3,), generator=gen).float()
    wi = torch.randint(-4, 5, w.shape, generator=gen).float()
    assert torch.equal(resnet18_var.stem_conv_pool(ints.cuda(), wi.cuda()).cpu(), expected(ints, wi))


def expected_magnitude(image, w):
    return expected(image.double().abs(), w.double().abs())   # a pooled value's sums are no larger than the largest


def test_values_that_do_not_split():
    import resnet18_var
    gen = torch.Generator().manual_seed(82)
    image = torch.randn((2, 64, 64, 3), generator=gen)
    w = torch.randn((64, 3, 7, 7), generator=gen) * 0.1
    image[0, 10, 11, 1] = float("inf")
    image[0, 50, 40, 0] = float("nan")
    image[1, 5:9] *= 1e36
    got, want = resnet18_var.stem_conv_pool(image.cuda(), w.cuda()).cpu(), expected(image, w)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf])
    ok = torch.isfinite(want)
    assert ((got - want)[ok].abs() <= 2 * 147 * 2.0 ** -24 * expected_magnitude(torch.nan_to_num(image, posinf=0.0), w)[ok]).all()
    w[3] *= 1e-30                                            # a channel of tiny weights
    got, want = resnet18_var.stem_conv_pool(image[1:].cuda(), w.cuda()).cpu()[..., 3], expected(image[1:].double(), w.double())[..., 3]
    assert ((got - want).abs() <= 147 * 2.0 ** -24 * expected_magnitude(image[1:], w)[..., 3]).all()


def test_spreads_beyond_the_exponents_that_pieces_are_shifted_by():
    """Within a channel's weights beyond 2^80, within a tile beyond 2^138: fp32 vector arithmetic, each pixel as good as alone."""
    import resnet18_var
    gen = torch.Generator().manual_seed(85)
    image, w = torch.randn((1, 64, 64, 3), generator=gen), torch.randn((64, 3, 7, 7), generator=gen) * 0.1
    bound = 2 * (147 + 4) * 2.0 ** -24
    spread = w.clone()
    spread[7, :, :3] *= 1e-28
    wide = image.clone()
    wide[0, :20] *= 1e22
    wide[0, 30:] *= 1e-22
    for im, wt in ((image, spread), (wide, w), (wide, spread)):
        got = resnet18_var.stem_conv_pool(im.cuda(), wt.cuda()).cpu()
        want = expected(im.double(), wt.double())
        assert ((got - want).abs() <= bound * expected_magnitude(im, wt)).all()


@pytest.mark.parametrize("bright", [24, 28, 34, 46, 60, 100])
@pytest.mark.parametrize("positive", [False, True])
def test_a_pixel_changes_only_what_sees_it(bright, positive):
    """One value 2^bright times the others: every pooled pixel that does not see it comes out bit for bit as without it."""
    import resnet18_var
    gen = torch.Generator().manual_seed(83)
    image, w = torch.randn((1, 90, 61, 3), generator=gen), torch.randn((64, 3, 7, 7), generator=gen) * 0.1
    if positive:
        image, w = image.abs(), w.abs()
    seen = torch.zeros_like(image)
    image[0, 40, 33, 1], seen[0, 40, 33, 1] = 0.0, 1.0
    without = resnet18_var.stem_conv_pool(image.cuda(), w.cuda()).cpu()
    image[0, 40, 33, 1] = 2.0 ** bright
    got = resnet18_var.stem_conv_pool(image.cuda(), w.cuda()).cpu()
    sees = expected(seen, torch.ones_like(w)) > 0
    same = torch.equal(got[~sees], without[~sees])
    assert same
    assert (got != without)[sees].any()


def test_all_24_bits_count_and_powers_of_two_commute():
    import resnet18_var
    gen = torch.Generator().manual_seed(84)
    run = lambda image, w: resnet18_var.stem_conv_pool(image.cuda(), w.cuda()).cpu()   # noqa: E731
    # single products: pixels far enough apart that a window holds one, one tap per channel
    for image_bits, w_bits in ((24, 1), (1, 24), (12, 12)):
        image, w = torch.zeros((1, 96, 96, 3)), torch.zeros((64, 3, 7, 7))
        image[0, ::16, ::16, 1] = (torch.randint(2 ** (image_bits - 1), 2 ** image_bits, (6, 6), generator=gen) | 1).float()
        w[:, 1, 3, 3] = (torch.randint(2 ** (w_bits - 1), 2 ** w_bits, (64,), generator=gen) | 1).float()
        same = torch.equal(run(image, w), expected(image.double(), w.double()).float())
        assert same, (image_bits, w_bits)
    # tiles of any magnitude, channels of any magnitude
    image, w = torch.randn((2, 64, 80, 3), generator=gen), torch.randn((64, 3, 7, 7), generator=gen)
    plain = run(image, w)
    for image_exp, w_exp in ((40, -60), (-60, 30), (0, -100), (-100, 60), (90, 20)):
        wide = w.clone()
        wide[5] *= 2.0 ** w_exp
        got = run(image * 2.0 ** image_exp, wide)
        want = plain * 2.0 ** image_exp
        want[..., 5] *= 2.0 ** w_exp
        same = torch.equal(got, want)
        assert same, (image_exp, w_exp)


def test_the_model_takes_it_and_the_library_path_agrees():
    import resnet18_var
    torch.manual_seed(3)
    model = resnet18_var.ResNet18Var().cuda()
    image = torch.randn((2, 64, 96, 3), device="cuda")
    assert resnet18_var._is_stem(model.conv1, image)
    assert not resnet18_var._is_stem(model.conv1, image.double())
    fused = model(image)
    strided = model(torch.cat([image, image], 3)[..., :3])
    seen = []
    model.conv1.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    plain = model(image)
    assert seen and torch.equal(strided, fused)
    assert (fused - plain).norm() <= 2e-6 * plain.norm()     # two fp32 sums of 147 products, through eight units


def test_whoever_watches_or_replaces_conv1_still_does():
    import resnet18_var
    from torch.utils.flop_counter import FlopCounterMode
    torch.manual_seed(3)
    model = resnet18_var.ResNet18Var().cuda()
    image = torch.randn((1, 32, 32, 3), device="cuda")
    seen = []
    watch = lambda m, i, *o: seen.append(m)   # noqa: E731
    for register in (torch.nn.modules.module.register_module_forward_hook, torch.nn.modules.module.register_module_forward_pre_hook,
                     model.conv1.register_forward_hook, model.conv1.register_forward_pre_hook):
        handle = register(watch)
        model(image)
        handle.remove()
        assert model.conv1 in seen, register
        del seen[:]
    own = model.conv1.forward
    model.conv1.forward = lambda x: (seen.append(model.conv1), own(x))[1]
    model(image)
    assert seen
    del model.conv1.forward
    counter = FlopCounterMode(display=False)
    with counter:
        model(image)
    assert counter.get_total_flops() >= 2 * 16 * 16 * 147 * 64
    assert resnet18_var._is_stem(model.conv1, image)


def test_images_the_kernel_does_not_take_go_to_the_layers():
    import resnet18_var
    import swc_hip
    model = resnet18_var.ResNet18Var().cuda()
    w = model.conv1.weight
    for H, W in ((1 << 20, 1), (1, 1 << 20)):
        image = torch.zeros((1, H, W, 3), device="cuda")
        assert not resnet18_var._is_stem(model.conv1, image)
        with pytest.raises(swc_hip.SwcError):
            resnet18_var.stem_conv_pool(image, w)
    image = torch.complex(torch.zeros(1, 32, 32, 3), torch.randn(1, 32, 32, 3)).cuda().conj().imag   # negated lazily
    assert image.is_neg() and not resnet18_var._is_stem(model.conv1, image)
