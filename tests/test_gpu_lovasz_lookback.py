"""The decoupled look-back variant of the Lovasz sort passes (plh_lovasz_forward_lookback: tile descriptors and
chained waits instead of a histogram kernel and a row scan in front of every pass) must give the results of the
default route bit for bit: same keys, same stable order, same Jaccard differences, same loss (the default passes for few
classes, value buckets for many, one block per row up to 7680 pixels; see test_gpu_lovasz_buckets). And the default passes by
themselves, against the CPU oracle as well: every digit plan, rows of 16k staging regions, rows with nothing to sort."""
import numpy as np
import pytest
import torch

import oracle
from oracle import synth

from .test_gpu_parity import dev, seg_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def native():
    from pytorch_loss import _native
    _native.load()
    return _native


CASES = [
    # shape, logits scale, boost of the label's logit            what it exercises
    ((2, 5, 100, 100), 2.0, 0.0),          # several tiles per class, the last one ragged
    ((1, 4, 70, 64), 2.0, 0.0),            # a little over one tile
    ((2, 19, 64, 64), 2.0, 0.0),
    ((3, 7, 200, 300), 2.0, 0.0),          # 44 tiles per class: long chains of descriptors
    ((2, 400, 40, 50), 0.002, 0.0),        # near-uniform predictions: two passes per class
    ((2, 120, 40, 50), 0.3, 0.0),          # three passes
    ((2, 120, 40, 50), 1.0, 12.0),         # confident predictions: all four
    ((1, 3, 1024, 1100), 2.0, 0.0),        # rows of 1.1 M pixels: 275 tiles
]


@pytest.mark.parametrize("shape,scale,boost", CASES)
def test_look_back_variant_is_bit_identical(native, shape, scale, boost):
    n_cls = shape[1]
    y = synth.seg_labels(61, shape[:1] + shape[2:], n_cls, 255, 0.1)
    x = synth.normal(61, 1, shape, 0.0, scale)
    if boost:
        x = x + np.float32(boost) * np.moveaxis(np.eye(n_cls, dtype=np.float32)[np.where(y == 255, 0, y)], -1, 1)
    xt, yt = dev(x), dev(y)
    losses, jacc = native.lovasz_forward(xt, yt, 255)
    for _ in range(2):                                  # twice: tickets and descriptors are cleared per call
        losses_lb, jacc_lb = native.lovasz_forward(xt, yt, 255, look_back=True)
        assert not torch.isnan(losses_lb).any()
        assert torch.equal(losses_lb, losses)
        assert torch.equal(jacc_lb.view(torch.int32), jacc.view(torch.int32))
    l64, _ = oracle.lovasz_forward(x.astype(np.float64), y, 255)
    np.testing.assert_allclose(losses_lb.cpu().numpy(), l64, rtol=3e-4 if boost else 1e-5)


LONG = 2560 * 1024 + 1      # the shortest row that goes by passes whatever its classes
# shape, logits scale, boost of the label's logit, what the labels lack, the most passes that a class takes
RADIX = [
    ((1, 3, 100, 200), 0.1, -8.0, None, 2),         # a network that is wrong everywhere: errors above 0.99
    ((2, 4, 100, 100), 0.002, 0.0, None, 3),        # near-uniform
    ((2, 4, 100, 100), 1.0, 12.0, None, 4),         # confident
    ((2, 4, 100, 100), 2.0, 0.0, "classes", None),  # classes that no pixel has
    ((1, 3, 90, 100), 2.0, 0.0, "all", None),       # nothing but ignored pixels
    ((1, 3, 1, LONG), 0.1, -8.0, None, 2),
    ((1, 3, 1, LONG), 0.15, 0.0, None, 3),
    ((1, 3, 1, LONG), 1.0, 12.0, None, 4),
    ((1, 3, 1, LONG), 2.0, 0.0, "classes", None),
    ((1, 3, 1, LONG), 2.0, 0.0, "all", None),
]


@pytest.mark.parametrize("shape,scale,boost,lack,passes", RADIX)
def test_default_passes(native, shape, scale, boost, lack, passes):
    n_cls, pixels = shape[1], shape[0] * shape[2] * shape[3]
    assert native.load().plh_lovasz_workspace_bytes(1, n_cls, pixels) >= 16 * n_cls * pixels     # two key, two value buffers
    y = synth.seg_labels(67, shape[:1] + shape[2:], n_cls, 255, 0.1)
    if lack:
        y[:] = 255 if lack == "all" else np.where(y == 255, 255, y % 2)
    x = synth.normal(67, 1, shape, 0.0, scale)
    hot = np.moveaxis(np.arange(n_cls) == y[..., None], -1, 1)
    if boost:
        x = x + np.float32(boost) * hot
    if passes:
        # the width of each class's keys: up to its best classified positive's
        p = np.exp(x.astype(np.float64) - x.max(axis=1, keepdims=True))
        best = [np.float32(1.0 - (p / p.sum(axis=1, keepdims=True)).swapaxes(0, 1)[c][hot.swapaxes(0, 1)[c]].max()) for c in range(n_cls)]
        bits = [int(np.float32(1.0).view(np.uint32) - e.view(np.uint32)).bit_length() for e in best]
        assert all((2 if b <= 16 else 3 if b <= 24 else 4) == passes for b in bits), bits
    losses, jacc = native.lovasz_forward(dev(x), dev(y), 255)
    for _ in range(2):
        other, jacc_lb = native.lovasz_forward(dev(x), dev(y), 255, look_back=True)
        assert torch.equal(other, losses) and torch.equal(jacc_lb.view(torch.int32), jacc.view(torch.int32))
    jacc = jacc.cpu().numpy()
    l64, _ = oracle.lovasz_forward(x.astype(np.float64), y, 255)
    np.testing.assert_allclose(losses.cpu().numpy(), l64, rtol=3e-4 if boost > 0 else 1e-5)      # as above
    assert (jacc[:, y.reshape(-1) == 255] == 0).all()
    _, j32 = oracle.lovasz_forward(x, y, 255)
    # a last-bit difference of expf reorders neighbours, and moves the difference of a positive and another: of the few pixels
    # that have one so near, or, with millions of errors within 0.1 of each other (as dense as floats lie), of up to half of
    # them, two in five such pairs being mixed
    dense = passes == 3 and pixels == LONG
    assert (jacc.view(np.uint32) == j32.view(np.uint32)).mean() > (0.8 if dense else 0.99)
