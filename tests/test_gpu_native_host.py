"""The native host side of the Python ops: the same values as the general path, which everything that is not a plain call takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(C=64, K=72, relu=False):
    gen = torch.Generator(device="cuda").manual_seed(91)
    rand = lambda *s: torch.randn(s, device="cuda", generator=gen)   # noqa: E731
    return {"x": rand(2, 7, 10, C), "ti": rand(16, 2, 4, 5, C), "w": rand(16, C, K), "a": rand(C), "b": rand(C), "scale": rand(K), "shift": rand(K),
            "res": rand(2, 8, 10, K)}


def calls(o, **kw):
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weights_bf16
    from winograd2x2_imTrans.winograd2x2_imTrans import winograd2x2_imTrans
    yield "transform", lambda **k: winograd2x2_imTrans(o["x"], **k), (16, 2, 4, 5, 64)
    yield "transform, relu, affine", lambda **k: winograd2x2_imTrans(o["x"], relu=True, scale=o["a"], shift=o["b"], **k), (16, 2, 4, 5, 64)
    yield "transform, bf16", lambda **k: winograd2x2_imTrans(o["x"], relu=True, out_dtype=torch.bfloat16, **k), (16, 2, 4, 5, 64)
    for precision in ("fp32", "bf16"):
        yield "conv " + precision, lambda **k: winograd2x2_conv(o["ti"], o["w"], precision=precision, **k), (2, 8, 10, 72)
        yield "conv epilogue " + precision, lambda **k: winograd2x2_conv(o["ti"], o["w"], precision=precision, scale=o["scale"], shift=o["shift"],
                                                                         residual=o["res"], residual_relu=True, **k), (2, 8, 10, 72)
    yield "stored", lambda **k: winograd2x2_conv(o["ti"].bfloat16(), winograd2x2_weights_bf16(o["w"]), residual=o["res"], **k), (2, 8, 10, 72)


def test_plain_calls_and_calls_with_out_agree():
    o = operands()
    for name, call, shape in calls(o):
        got = call()
        assert got.shape == shape and not got.requires_grad, name
        assert torch.equal(got, call(out=torch.empty_like(got))), name


def test_what_is_not_plain_takes_the_general_path():
    from torch.utils._python_dispatch import TorchDispatchMode
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv
    from winograd2x2_imTrans.winograd2x2_imTrans import winograd2x2_imTrans

    class Count(TorchDispatchMode):
        seen = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.seen += 1
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    o = operands()
    plain = winograd2x2_conv(winograd2x2_imTrans(o["x"]), o["w"])
    with Count():
        watched = winograd2x2_conv(winograd2x2_imTrans(o["x"]), o["w"])
    assert Count.seen >= 2 and torch.equal(watched, plain)
    strided = torch.empty((2, 10, 7, 64), device="cuda").transpose(1, 2).copy_(o["x"])
    assert torch.equal(winograd2x2_conv(winograd2x2_imTrans(strided), o["w"].transpose(1, 2).contiguous().transpose(1, 2)), plain)
    assert torch.equal(winograd2x2_conv(winograd2x2_imTrans(o["x"].as_subclass(Sub)), o["w"]), plain)
    x, w = o["x"].clone().requires_grad_(), o["w"].clone().requires_grad_()
    y = winograd2x2_conv(winograd2x2_imTrans(x), w)
    assert torch.equal(y, plain) and y.requires_grad
    with torch.no_grad():
        assert not winograd2x2_conv(winograd2x2_imTrans(x), w).requires_grad
    with torch.inference_mode():
        assert torch.equal(winograd2x2_conv(winograd2x2_imTrans(o["x"]), o["w"]), plain)
    # on a side stream that is busy and then writes what the ops read: launched on another, they would read zeros
    side, late = torch.cuda.Stream(), torch.zeros_like(o["x"])
    busy = torch.ones((4096, 4096), device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(20):
            busy = torch.mm(busy, busy).clamp_(max=1)
        late.copy_(o["x"])
        other = winograd2x2_conv(winograd2x2_imTrans(late), o["w"])
        last = winograd2x2_imTrans(other)
        other.zero_()   # and the convolution's output is not written to once more
    side.synchronize()
    assert torch.equal(last, winograd2x2_imTrans(plain)) and not other.any()
    for bad in (o["x"].double(), o["x"].cpu(), o["x"][0], "x"):
        with pytest.raises((TypeError, ValueError, RuntimeError)):
            winograd2x2_imTrans(bad)
    for bad in (o["w"][:, :60], o["w"][:15], o["w"].half(), o["w"].cpu(), None):
        with pytest.raises((TypeError, ValueError, RuntimeError)):
            winograd2x2_conv(o["ti"], bad)
    for bad in ({"scale": o["scale"]}, {"scale": o["scale"][:5], "shift": o["shift"]}, {"residual": o["res"][:1]}, {"residual_relu": True}):
        with pytest.raises((TypeError, ValueError)):
            winograd2x2_conv(o["ti"], o["w"], **bad)
    with pytest.raises(Exception):
        torch.func.vmap(lambda t: winograd2x2_imTrans(t))(o["x"].unsqueeze(0))


def test_arguments_that_raise_do_so_as_in_the_general_path():
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv, winograd2x2_weights_bf16
    from winograd2x2_imTrans.winograd2x2_imTrans import winograd2x2_imTrans, winograd2x2_imTrans_grad
    o = operands()
    neither = torch.ones(2)   # no truth value
    ti16, w16 = o["ti"].bfloat16(), winograd2x2_weights_bf16(o["w"])
    for call in (lambda: winograd2x2_imTrans(o["x"], relu=neither), lambda: winograd2x2_imTrans(o["x"], relu=neither, out_dtype=torch.bfloat16),
                 lambda: winograd2x2_conv(o["ti"], o["w"], residual=o["res"], residual_relu=neither),
                 lambda: winograd2x2_conv(ti16, w16, residual=o["res"], residual_relu=neither),
                 lambda: winograd2x2_conv(ti16, w16, workspace=neither)):
        with pytest.raises(RuntimeError, match="ambiguous"):
            call()
    for H, W in ((2 ** 70, 10), (7, -2 ** 70), (7, -1)):
        with pytest.raises(ValueError, match="do not tile"):
            winograd2x2_imTrans_grad(o["ti"], H, W)


def test_tangents_and_traces_go_through_the_models_pools():
    # Torch's operators carry a tangent on and are recorded by a trace; the library's kernels would do neither.
    import torch.autograd.forward_ad as fwd
    import resnet18_var
    gen = torch.Generator(device="cuda").manual_seed(92)
    x, t, other = (torch.randn((2, 7, 10, 64), device="cuda", generator=gen).permute(0, 3, 1, 2) for _ in range(3))
    plain = resnet18_var._max_pool_same(x)
    with fwd.dual_level():
        out = fwd.unpack_dual(resnet18_var._max_pool_same(fwd.make_dual(x, t)))
        assert torch.equal(out.primal, plain)
        pads = resnet18_var._same_pad(x, 3, 2)
        padded, at = torch.nn.functional.pad(x, pads, value=float("-inf")), torch.nn.functional.pad(t, pads)
        index = torch.nn.functional.max_pool2d(padded, 3, 2, return_indices=True)[1]
        assert torch.equal(out.tangent, at.flatten(2).gather(2, index.flatten(2)).view_as(plain))
    traced = torch.jit.trace(resnet18_var._max_pool_same, (x,))
    assert torch.equal(traced(other), resnet18_var._max_pool_same(other))


def test_gradients_through_both_paths():
    from winograd2x2_conv.winograd2x2_conv import winograd2x2_conv_grad
    from winograd2x2_imTrans.winograd2x2_imTrans import winograd2x2_imTrans_grad
    o = operands()
    g = torch.randn((2, 8, 10, 72), device="cuda")
    strided = g.transpose(1, 2).contiguous().transpose(1, 2)      # not contiguous
    for a, b in zip(winograd2x2_conv_grad(o["ti"], o["w"], g), winograd2x2_conv_grad(o["ti"], o["w"], strided)):
        assert torch.equal(a, b)
    strided = o["ti"].transpose(1, 2).contiguous().transpose(1, 2)
    for relu_input in (None, o["x"]):
        assert torch.equal(winograd2x2_imTrans_grad(o["ti"], 7, 10, relu_input=relu_input),
                           winograd2x2_imTrans_grad(strided, 7, 10, relu_input=relu_input))
    for bad in (g[:1], g[:, :6], g[..., :70]):
        with pytest.raises(Exception):
            winograd2x2_conv_grad(o["ti"], o["w"], bad)
    with pytest.raises(ValueError):
        winograd2x2_imTrans_grad(o["ti"], 9, 10)


def test_key_tells_writes_and_replacements():
    import swc_hip
    key = swc_hip.native().key
    w, m = torch.zeros(4, device="cuda"), torch.ones(4, device="cuda")
    k = key(w, m)
    assert key(w, m) == k and key(w.detach(), m) == k
    assert key(w, None) != k and key(w, m.clone()) != k and key(m, w) != k
    w.add_(1)
    assert key(w, m) != k
    with pytest.raises(TypeError):
        key(1)


@pytest.mark.gpu
@pytest.mark.parametrize("affine", [False, True])
@pytest.mark.parametrize("shape", [(1, 1, 1, 32, 1), (2, 7, 9, 64, 64), (1, 8, 8, 96, 65), (3, 5, 13, 128, 200), (1, 3, 3, 48, 20), (1, 2, 3, 4128, 8)])
def test_relu_pointwise_conv(shape, affine):
    # Tiles of 64 rows and columns and steps of 32 channels: below, at and beyond each; 48 channels, and 4128 with an affine, take
    # passes of their own.  Whole numbers up to 8*32*4128 < 2^24 are exact in any order of the sums.
    import resnet18_var
    B, H, W, C, K = shape
    gen = torch.Generator().manual_seed(5)
    x, w = (torch.randint(-4, 5, s, generator=gen).float() for s in ((B, H, W, C), (K, C)))
    a, b = (torch.randint(-2, 3, (C,), generator=gen).float() for _ in range(2))
    dev = torch.device("cuda:0")
    got = resnet18_var.relu_pointwise_conv(x.to(dev), w.to(dev), (a.to(dev), b.to(dev)) if affine else None).cpu()
    act = torch.relu(x.double() * a + b) if affine else torch.relu(x.double())
    assert torch.equal(got.double(), act @ w.double().t())
    # an infinity or NaN reaches its own pixel's sums and no other's
    for bad in (float("nan"), float("inf"), float("-inf")):
        y = x.clone()
        y[0, 0, 0, C // 2] = bad
        w1, a1, b1 = torch.ones_like(w), torch.ones_like(a), torch.zeros_like(b)
        got = resnet18_var.relu_pointwise_conv(y.to(dev), w1.to(dev), (a1.to(dev), b1.to(dev)) if affine else None).cpu()
        want = torch.relu(y) @ w1.t()
        assert torch.equal(torch.nan_to_num(got, 7.5, 9.5, 1.5), torch.nan_to_num(want, 7.5, 9.5, 1.5))


@pytest.mark.parametrize("affine", [False, True])
@pytest.mark.parametrize("shape", [(1, 1, 1, 32, 1), (2, 9, 11, 64, 64), (1, 8, 8, 96, 72), (1, 2, 3, 4128, 8)])
def test_relu_pointwise_conv_rounds_as_separate_passes(shape, affine):
    # The same bits as the BatchNorm's product and sum, the ReLU and the product one after the other, whichever way is taken: a model's
    # later layers turn a last bit into another bf16 rounding.
    import resnet18_var
    B, H, W, C, K = shape
    gen = torch.Generator(device="cuda").manual_seed(6)
    x, w = torch.randn((B, H, W, C), device="cuda", generator=gen), torch.randn((K, C), device="cuda", generator=gen)
    a, b = torch.rand(C, device="cuda", generator=gen) + 0.5, torch.randn(C, device="cuda", generator=gen) * 0.1
    got = resnet18_var.relu_pointwise_conv(x, w, (a, b) if affine else None)
    assert torch.equal(got, resnet18_var.pointwise_conv(torch.relu(torch.addcmul(b, x, a) if affine else x), w))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (2, 1, 5, 64), (1, 2, 2, 68), (3, 7, 10, 64), (2, 14, 9, 132), (1, 17, 16, 512), (2, 5, 6, 30)])
def test_model_pools(shape):
    # Odd and even sides (padding in front or not), sums shorter than, as long as and longer than their sixteen parts, channels that are
    # no whole workgroup, and 30 channels, which take torch's operators.  The mean adds n numbers: n * 2^-24 of their mean.
    import resnet18_var
    B, H, W, C = shape
    x = torch.randn(shape, generator=torch.Generator().manual_seed(7))
    nchw = x.permute(0, 3, 1, 2)
    dev = torch.device("cuda:0")
    pads = resnet18_var._same_pad(nchw, 3, 2)
    for bad in (None, float("nan"), float("inf"), float("-inf")):
        if bad is not None:
            x[0, H // 2, W // 2, C // 2] = bad
        got = resnet18_var._max_pool_same(nchw.to(dev)).cpu()
        want = torch.nn.functional.max_pool2d(torch.nn.functional.pad(nchw, pads, value=float("-inf")), 3, 2)
        assert torch.equal(torch.nan_to_num(got, 7.5), torch.nan_to_num(want, 7.5))
        mean = resnet18_var._native.relu_mean(x.to(dev))
        assert (mean is None) == (C % 4 != 0)
        if mean is not None:
            want = torch.relu(x.double()).mean(dim=(1, 2))
            assert torch.allclose(mean.cpu().double(), want, rtol=H * W * 2.0 ** -24 + 2.0 ** -23, atol=0, equal_nan=True)


@pytest.mark.parametrize("shape", [(2, 32, 32, 68), (1, 33, 32, 64), (1, 64, 64, 64)])
def test_relu_mean_up_to_its_longest_chain(shape):
    # 1024 pixels are sums of 64 terms in sixteen parts, four more additions and a division, all of one sign: 69 * 2^-24.  Beyond, the
    # library's reduction runs.
    import resnet18_var
    B, H, W, C = shape
    x = torch.randn(shape, generator=torch.Generator().manual_seed(9)) * torch.logspace(-3, 3, C)
    got = resnet18_var._native.relu_mean(x.cuda())
    assert (got is None) == (H * W > 1024)
    if got is not None:
        want = torch.relu(x.double()).mean(dim=(1, 2))
        assert ((got.cpu().double() - want).abs() <= 69 * 2.0 ** -24 * want).all()
