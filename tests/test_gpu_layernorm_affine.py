"""The layer-norm module's kernels with weight and bias against the same module in 64 bits (its formulas in torch, on the
CPU): every slot count and form on both sides of its limits, loops of several pixel groups per block, and what the
gradients of weight and bias are when only some are asked for.
Outputs and grad_x as in test_gpu_layernorm; a sum over P pixels of fp32 terms t may be off by about
sqrt(P) * 2^-24 * max|t| (16-bit: one more rounding of the result)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pl():
    import pytorch_loss
    from pytorch_loss import _native
    _native.load()
    return pytorch_loss


# (N, C, H, W): one wave (C <= 32), four waves, eight waves with every slot count up to 128; ragged pixel counts, one pixel per
# lane, planes of odd length, more groups than blocks (the last two)
SHAPES = [(2, 1, 8, 8), (1, 5, 7, 7), (2, 8, 5, 13), (3, 12, 8, 9), (1, 20, 20, 20), (2, 32, 10, 33), (2, 33, 8, 8),
          (1, 64, 15, 20), (2, 65, 8, 16), (1, 100, 7, 11), (1, 160, 8, 8), (1, 256, 10, 13), (1, 384, 8, 8), (1, 512, 7, 7),
          (1, 600, 8, 8), (1, 768, 7, 10), (1, 1000, 8, 9), (2, 19, 65, 65), (2, 100, 64, 65), (1, 700, 65, 65),
          (5, 8, 513, 513), (5, 72, 256, 161)]


def ref64(x, w, b, g, eps):
    n, c = x.shape[:2]
    x3, g3 = x.double().reshape(n, c, -1), g.double().reshape(n, c, -1)
    w, b = w.double().reshape(1, c, 1), b.double().reshape(1, c, 1)
    mean = x3.mean(1, keepdim=True)
    v = x3.var(1, keepdim=True, unbiased=False) + eps
    y = (x3 - mean) * v.rsqrt()
    gx = -v.rsqrt() * (1 / c + (x3 - mean) * (x3 - 1 / c) * mean * v) * (g3 * w)       # csrc/layer_norm.cu:212-216
    return w * y + b, gx, g3 * y, g3


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
def test_module_matches_64_bits(pl, shape, dtype):
    gen = torch.Generator().manual_seed(sum(shape))
    n, c = shape[:2]
    x = (torch.randn(shape, generator=gen) * 1.5 + 0.3).to(dtype)
    g = torch.randn(shape, generator=gen).to(dtype)
    m = pl.LayerNormV3(c).to("cuda", dtype)
    with torch.no_grad():
        m.weight.copy_(1 + 0.2 * torch.randn((1, c, 1), generator=gen))
        m.bias.copy_(0.2 * torch.randn((1, c, 1), generator=gen))
    xt = x.cuda().requires_grad_()
    out = m(xt)
    out.backward(g.cuda())
    want, want_x, gy, g3 = ref64(x, m.weight.detach().cpu(), m.bias.detach().cpu(), g, 1e-6)
    step = {torch.float32: 0.0, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    assert out.dtype == dtype and xt.grad.dtype == dtype and m.weight.grad.dtype == dtype
    flat = lambda t: t.detach().cpu().double().reshape(n, c, -1)
    assert ((flat(out) - want).abs() <= 1e-5 + step * want.abs()).all()
    assert ((flat(xt.grad) - want_x).abs() <= 1e-5 * want_x.abs().max() + step * want_x.abs()).all()
    pixels = x.numel() // c
    for got, terms in ((m.weight.grad, gy), (m.bias.grad, g3)):
        assert got.shape == (1, c, 1)
        total = terms.sum((0, 2))
        bound = (8 + np.sqrt(pixels)) * 2.0 ** -24 * terms.abs().max() + step * total.abs() + 1e-30
        # the normalised value itself is good to about 1e-6
        bound = bound + (np.sqrt(pixels) * 1e-6 if terms is gy else 0.0)
        assert ((got.detach().cpu().double().reshape(c) - total).abs() <= bound).all()


def test_partial_gradients_and_fallbacks(pl):
    x = torch.randn(2, 16, 9, 10, device="cuda", requires_grad=True)
    m = pl.LayerNormV3(16).cuda()
    g = torch.randn(2, 16, 9, 10, device="cuda")
    m(x).backward(g)
    full = [t.grad.clone() for t in (x, m.weight, m.bias)]
    for frozen in (0, 1, 2):
        leaves = [t.detach().requires_grad_(i != frozen) for i, t in enumerate((x, m.weight, m.bias))]
        m2 = pl.LayerNormV3(16).cuda()
        m2.weight, m2.bias = torch.nn.Parameter(leaves[1], leaves[1].requires_grad), torch.nn.Parameter(leaves[2], leaves[2].requires_grad)
        m2(leaves[0]).backward(g)
        for i, (t, want) in enumerate(zip((leaves[0], m2.weight, m2.bias), full)):
            assert (t.grad is None) if i == frozen else torch.equal(t.grad, want)
    # create_graph: the gradient of weight stays differentiable with respect to the upstream gradient
    up = g.clone().requires_grad_()
    gw, = torch.autograd.grad(m(x), m.weight, up, create_graph=True)
    assert torch.allclose(gw, full[1], rtol=1e-4, atol=1e-4)
    gw.sum().backward()
    assert up.grad is not None and up.grad.abs().sum() > 0
    # fp32 parameters on a 16-bit tensor, one pixel per row, more channels than the kernels hold: torch's operations
    half = m(x.detach().bfloat16())
    assert half.dtype == torch.float32
    wide = pl.LayerNormV3(1100).cuda()
    assert wide(torch.randn(1, 1100, 8, 8, device="cuda")).shape == (1, 1100, 8, 8)
    assert m(torch.randn(4, 16, 1, 1, device="cuda")).shape == (4, 16, 1, 1)


def test_eps_zero_on_planes_of_odd_length(pl):
    """The last lane of an image holds fewer pixels than the others: its missing ones have no variance, and with eps = 0 no
    finite normalised value either. Bounds as above."""
    gen = torch.Generator().manual_seed(5)
    shape = (2, 19, 65, 65)
    x, g = torch.randn(shape, generator=gen), torch.randn(shape, generator=gen)
    m = pl.LayerNormV3(19, eps=0.0).cuda()
    xt = x.cuda().requires_grad_()
    m(xt).backward(g.cuda())
    _, _, gy, g3 = ref64(x, m.weight.detach().cpu(), m.bias.detach().cpu(), g, 0.0)
    for got, terms in ((m.weight.grad, gy), (m.bias.grad, g3)):
        pixels = 2 * 65 * 65
        bound = (8 + np.sqrt(pixels)) * 2.0 ** -24 * terms.abs().max() + np.sqrt(pixels) * 1e-6
        assert ((got.cpu().double().reshape(19) - terms.sum((0, 2))).abs() <= bound).all()


def test_what_torch_refuses_stays_refused(pl):
    """A weight changed in place between the passes, a second backward through freed buffers; forward mode through the weight
    alone keeps working, and parameters of another shape broadcast as torch broadcasts them."""
    x = torch.randn(2, 8, 9, 10, device="cuda", requires_grad=True)
    m = pl.LayerNormV3(8).cuda()
    out = m(x)
    with torch.no_grad():
        m.weight.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    out = m(x).sum()
    out.backward()
    with pytest.raises(RuntimeError, match="second time"):
        out.backward()
    from torch.autograd import forward_ad
    plain = pl.LayerNormV3(8, affine=False)(x.detach())
    weight, bias = m.weight.detach(), m.bias.detach()
    tangent = torch.randn_like(weight)
    with forward_ad.dual_level():
        del m.weight, m.bias
        m.weight, m.bias = forward_ad.make_dual(weight, tangent), bias
        got = forward_ad.unpack_dual(m(x.detach())).tangent
    assert torch.allclose(got, tangent.view(1, 8, 1, 1) * plain)
    square = torch.randn(1, 8, 2, 4, device="cuda")
    m.weight, m.bias = torch.arange(8.0, device="cuda"), torch.zeros(8, device="cuda")      # along the pixels
    want = (pl.LayerNormV3(8, affine=False)(square).view(1, 8, 8) * m.weight).view_as(square)
    assert torch.equal(m(square), want)


def test_input_changed_in_place_before_the_backward(pl):
    """The backward reads the input again: where the input takes part in the graph, a change of it before the backward is
    refused; where it does not (a buffer that is filled anew), the gradients of weight and bias are those of the values that
    the forward saw, bit for bit; so are all of them where the forward worked on a copy of a strided input."""
    gen = torch.Generator().manual_seed(11)
    shape = (2, 16, 9, 10)
    data, g = torch.randn(shape, generator=gen).cuda(), torch.randn(shape, generator=gen).cuda()
    m = pl.LayerNormV3(16).cuda()
    with torch.no_grad():
        m.weight.add_(0.1 * torch.randn(m.weight.shape, generator=gen).cuda())

    def grads(x, between):
        m.weight.grad = m.bias.grad = None
        out = m(x)
        between(x)
        out.backward(g)
        return [t.clone() for t in (m.weight.grad, m.bias.grad)]

    for fill in (lambda x: x.mul_(2).add_(1), lambda x: x.copy_(g), lambda x: x.relu_()):
        want = grads(data.clone(), lambda x: None)
        got = grads(data.clone(), fill)                                     # a buffer without gradient
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            grads(data.clone().requires_grad_() * 1, fill)                  # part of the graph
    x = data.clone().requires_grad_()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        grads(x, lambda x: x.detach().mul_(2))
    # a strided input: what the backward reads is a copy of its own
    wide = torch.randn((2, 32, 9, 10), generator=gen).cuda()
    leaf = wide.clone().requires_grad_()
    want = grads((leaf * 1)[:, ::2], lambda x: None) + [leaf.grad]
    leaf = wide.clone().requires_grad_()
    got = grads((leaf * 1)[:, ::2], lambda x: x.mul_(2)) + [leaf.grad]
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    assert torch.equal(got[2], want[2])
    # an in-place operation on the result, as an activation does, is nobody's loss
    x = data.clone().requires_grad_()
    out = m(x).relu_()
    out.backward(g)
    y = data.clone().requires_grad_()
    torch.relu(m(y)).backward(g)
    assert torch.equal(x.grad, y.grad)


@pytest.mark.parametrize("trained", ["neither", "weight", "bias"])
def test_frozen_input_computes_no_gradient_of_it(pl, trained):
    """Without a gradient of the input the backward allocates nothing of the input's size (peak: the upstream gradient times
    the normalised input, where the weight is trained)."""
    shape = (4, 64, 64, 64)
    x, g = torch.randn(shape, device="cuda"), torch.randn(shape, device="cuda")
    m = pl.LayerNormV3(64).cuda()
    m.weight.requires_grad_(trained == "weight")
    m.bias.requires_grad_(trained == "bias")
    out = m(x)
    assert out.requires_grad == (trained != "neither")
    if trained == "neither":
        return
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out.backward(g)
    peak = torch.cuda.max_memory_allocated() - before
    assert peak < (0.5 if trained == "bias" else 1.5) * x.numel() * 4
    assert x.grad is None
