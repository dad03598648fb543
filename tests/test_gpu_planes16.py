"""The backward of 16-bit channel planes from what the forward left per pixel (csrc/planes16.hpp): LSR and Taylor cross
entropy against the same gradient in 64 bits and against the kernels that recompute. The first and last channel counts of both
forward forms, tiles that end inside a plane, planes shared out over blocks, views at other offsets into their lines."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}        # 8 and 11 significant bits: half a unit in the last of them
IGN = 255

# 16..32 channels and 33..256; a little more than 4096 pixels (the shortest planes), one and several tiles
SHAPES = [(2, 19, 65, 67), (1, 32, 65, 67), (1, 16, 63, 66), (2, 17, 1, 4097), (1, 24, 100, 131),
          (2, 33, 63, 66), (1, 256, 65, 66), (3, 40, 97, 66), (2, 150, 65, 65), (1, 255, 66, 67), (1, 36, 1, 9001)]


def inputs(shape, dtype, seed, offset=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n, c = shape[:2]
    store = torch.empty(offset + torch.Size(shape).numel(), device="cuda", dtype=dtype)
    x = store[offset:].view(shape)
    x.copy_(torch.randn(shape, device="cuda", generator=g) * 2)
    y = torch.randint(0, c, (n,) + shape[2:], device="cuda", generator=g)
    y[torch.rand(y.shape, device="cuda", generator=g) < 0.1] = IGN
    return x, y


def losses(kind, c):
    import pytorch_loss as pl
    if kind == "lsr":
        return lambda r: pl.LabelSmoothSoftmaxCEV3(lb_smooth=0.1, reduction=r, ignore_index=IGN)
    return lambda r: pl.TaylorCrossEntropyLossV3(n=int(kind[-1]), reduction=r, ignore_index=IGN)


def exact(kind, x, y):
    a = x.double().requires_grad_()
    if kind == "lsr":
        logp = a.log_softmax(1)
    else:
        t = [torch.ones_like(a)]
        for i in range(1, int(kind[-1]) + 1):
            t.append(t[-1] * a / i)
        f = sum(t)
        logp = f.log() - f.sum(1, keepdim=True).log()
    hot = torch.zeros_like(logp).scatter_(1, y.clamp(max=x.shape[1] - 1).unsqueeze(1), 1.0)
    w = 0.9 * hot + 0.1 / x.shape[1] * (1 - hot) if kind == "lsr" else hot
    keep = (y != IGN).unsqueeze(1)
    (-(w * logp * keep).sum() / keep.sum()).backward()
    return a.grad


def saved(kind, x):
    from pytorch_loss import _native
    entry = "plh_lsr_saves_lse_planes16" if kind == "lsr" else "plh_taylor_ce_saves_sums_planes16"
    return getattr(_native.load(), entry)(1 if x.dtype == torch.float16 else 2, x.shape[0], x.shape[1], x[0, 0].numel())


@pytest.mark.parametrize("kind", ["lsr", "taylor2", "taylor4"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_gradient(shape, dtype, kind):
    x, y = inputs(shape, dtype, 7)
    assert saved(kind, x) == 1
    make = losses(kind, shape[1])
    a = x.clone().requires_grad_()
    scale = 512.0 if dtype == torch.float16 else 1.0        # clear of the type's least values
    (make("mean")(a, y) * scale).backward()
    want = exact(kind, x, y) * scale
    # one rounding to the type, and sums in 32 bits (1e-6 of the largest, as the fp32 planes' test)
    assert ((a.grad.double() - want).abs() <= HALF_ULP[dtype] * want.abs() * 1.01 + 2e-6 * want.abs().max() + 2.0 ** -24).all()
    assert not a.grad[(y == IGN).unsqueeze(1).expand_as(x)].any()


@pytest.mark.parametrize("kind", ["lsr", "taylor4"])
@pytest.mark.parametrize("offset", [0, 1, 8, 64])
@pytest.mark.parametrize("shape", [(2, 19, 65, 67), (2, 40, 66, 65)], ids=str)
def test_views_and_labels_without_a_channel(shape, offset, kind):
    """A view whose gradient sits elsewhere in its line takes the kernels that recompute; labels outside the classes and NaN at
    ignored pixels are what they are there."""
    x, y = inputs(shape, torch.bfloat16, 11, offset)
    y[0, 0, :5] = shape[1] + 3
    x[(y == IGN).unsqueeze(1).expand_as(x)] = float("nan")
    make = losses(kind, shape[1])
    a = x.detach().requires_grad_()
    make("sum")(a, y).backward()
    b = x.clone().requires_grad_()
    make("none")(b, y).float().sum().backward()
    assert not torch.isnan(a.grad).any()
    assert ((a.grad.float() - b.grad.float()).abs() <= 2 * HALF_ULP[torch.bfloat16] * b.grad.float().abs() * 1.01 + 1e-6).all()


# planes of a multiple of 8 pixels off the lines; 12 planes per block and a last share of 6 (beyond 4096 blocks)
DIRECT = SHAPES + [(2, 19, 57, 72), (1, 200, 57, 72), (8, 150, 513, 513)]


# logits with a common offset, whose largest takes digits from anything added to it
@pytest.mark.parametrize("offset", [0.0, 1000.0, -300.0, 16000.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", DIRECT, ids=str)
def test_lsr_is_the_recomputed_gradient(shape, dtype, offset):
    """Bit for bit, at ignored pixels and labels without a channel too, and at the ends of the planes."""
    from pytorch_loss import _native
    x, y = inputs(shape, dtype, 13)
    boost = torch.rand(y.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(59)) * 12
    x.scatter_add_(1, y.clamp(max=shape[1] - 1).unsqueeze(1), boost.to(dtype).unsqueeze(1))
    x += offset
    y[0, 0, :5] = shape[1] + 3
    y[0, 0, 5:9] = -7
    x[:, :, -1, -1] = float("-inf")
    x[(y == IGN).unsqueeze(1).expand_as(x)] = float("nan")
    args = _native.lsr_args(x, y)
    loss, n_valid, lse = _native.lsr_forward_reduced_lse(x, y, IGN, 0.1, True, args=args)
    assert lse is not None
    up = torch.tensor(3.0 if dtype == torch.bfloat16 else 700.0, device="cuda")
    got = _native.lsr_backward_scaled_lse(lse, IGN, 0.1, up, n_valid, args)
    want = _native.lsr_backward_scaled(x, y, IGN, 0.1, up, n_valid, args=args)
    number = ~torch.isnan(want)
    assert torch.equal(torch.isnan(got), ~number) and torch.equal(got.view(torch.int16)[number], want.view(torch.int16)[number])


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", DIRECT, ids=str)
def test_taylor_from_its_sums(shape, dtype, order):
    """As test_gradient, whose sizes the module may have recomputed."""
    from pytorch_loss import _native
    x, y = inputs(shape, dtype, 7)
    args = _native.taylor_args(x, y)
    _, n_valid, sums = _native.taylor_ce_forward_reduced_sums(x, y, order, IGN, True, args=args)
    assert sums is not None
    scale = 512.0 if dtype == torch.float16 else 1.0
    got = _native.taylor_ce_backward_scaled_sums(sums, order, IGN, torch.tensor(scale, device="cuda"), n_valid, args)
    want = exact("taylor%d" % order, x, y) * scale
    assert ((got.double() - want).abs() <= HALF_ULP[dtype] * want.abs() * 1.01 + 2e-6 * want.abs().max() + 2.0 ** -24).all()
    assert not got[(y == IGN).unsqueeze(1).expand_as(x)].any()


@pytest.mark.parametrize("offset", [1, 8, 64])
@pytest.mark.parametrize("shape", [(2, 19, 65, 67), (2, 40, 66, 65)], ids=str)
def test_views_from_what_was_kept(shape, offset):
    """Views at other offsets into their lines, where the gradient may sit elsewhere in its own."""
    from pytorch_loss import _native
    x, y = inputs(shape, torch.bfloat16, 17, offset)
    up = torch.ones((), device="cuda")
    args = _native.lsr_args(x, y)
    _, n_valid, lse = _native.lsr_forward_reduced_lse(x, y, IGN, 0.1, True, args=args)
    got = _native.lsr_backward_scaled_lse(lse, IGN, 0.1, up, n_valid, args)
    assert torch.equal(got, _native.lsr_backward_scaled(x, y, IGN, 0.1, up, n_valid, args=args))
    args = _native.taylor_args(x, y)
    _, n_valid, sums = _native.taylor_ce_forward_reduced_sums(x, y, 4, IGN, True, args=args)
    got = _native.taylor_ce_backward_scaled_sums(sums, 4, IGN, up, n_valid, args).float()
    want = _native.taylor_ce_backward(x, y, 4, IGN, up, n_valid, args=args).float()
    assert ((got - want).abs() <= 2 * HALF_ULP[torch.bfloat16] * want.abs() * 1.01 + 1e-9).all()


@pytest.mark.parametrize("kind, shape, keeps", [("lsr", (2, 16, 257, 257), False), ("lsr", (8, 32, 513, 513), False), ("lsr", (4, 40, 129, 129), False),
                                                ("lsr", (2, 200, 257, 257), True), ("lsr", (8, 150, 513, 513), True), ("lsr", (16, 19, 769, 769), True),
                                                ("taylor4", (4, 150, 385, 385), False), ("taylor4", (3, 128, 257, 257), True),
                                                ("taylor4", (16, 19, 769, 769), True)], ids=str)
def test_modules_keep_what_pays(kind, shape, keeps):
    """A step that keeps something per pixel is up to twice as long where the caches hold the logits ((2,16,257,257): 25 -> 45 us)."""
    x = torch.zeros(shape, device="cuda", dtype=torch.bfloat16).requires_grad_()
    y = torch.zeros((shape[0],) + shape[2:], device="cuda", dtype=torch.int64)
    ctx = losses(kind, shape[1])("mean")(x, y).grad_fn
    assert ((ctx.variables if kind == "lsr" else ctx.vars)[-1] is not None) == keeps


def test_a_mask_is_refused():
    """The byte mask of a selection has no place in this backward: the call raises, and never returns an unmasked gradient."""
    from pytorch_loss import _native
    x, y = inputs((2, 19, 65, 67), torch.bfloat16, 5)
    args = _native.lsr_args(x, y)
    _, n_valid, lse = _native.lsr_forward_reduced_lse(x, y, IGN, 0.1, True, args=args)
    kept = (y != IGN).to(torch.uint8)
    up = torch.ones((), device="cuda")
    with pytest.raises(RuntimeError, match="mask"):
        _native.lsr_backward_scaled_lse(lse, IGN, 0.1, up, n_valid, args, kept=kept)
    assert _native.lsr_backward_scaled_lse(lse, IGN, 0.1, up, n_valid, args).shape == x.shape


def test_where_it_applies():
    from pytorch_loss import _native
    lib = _native.load()
    for entry in (lib.plh_lsr_saves_lse_planes16, lib.plh_taylor_ce_saves_sums_planes16):
        assert entry(2, 1, 19, 4097) == 1 and entry(2, 1, 19, 4160) == 0 and entry(2, 1, 32, 4097) == 1 and entry(2, 1, 15, 4097) == 0
        assert entry(2, 1, 33, 4097) == 1 and entry(1, 1, 256, 4098) == 1 and entry(2, 1, 257, 4097) == 0 and entry(2, 1, 33, 4096) == 0
        assert entry(2, 1, 40, 4095) == 0 and entry(0, 1, 40, 4097) == 0 and entry(2, 64, 40, 1) == 0
