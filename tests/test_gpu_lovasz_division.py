"""The Lovasz kernels' divisions, whose steps are written out, against IEEE division: probabilities down to the smallest subnormal,
and the Jaccard indices of rows of every route, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def native():
    from pytorch_loss import _native
    _native.load()
    return _native


def first_probability(native, t, k, n_cls):
    """softmax(t, 0 (k times), -inf, ...)[0] at every pixel as the backward sees it: with a Jaccard difference of 1 in class 0, none
    elsewhere and an upstream gradient of 1 for it, the gradient is p (1 - p), and 1 - p is 1."""
    x = torch.full((1, n_cls, t.numel(), 1), float("-inf"), device="cuda")
    x[0, 0, :, 0] = t
    x[0, 1:1 + k] = 0.0
    y = torch.full((1, t.numel(), 1), 1, device="cuda", dtype=torch.int64)
    jacc = torch.zeros((n_cls, t.numel()), device="cuda")
    jacc[0] = 1.0
    up = torch.zeros(n_cls, device="cuda")
    up[0] = 1.0
    return native.lovasz_backward(up, x, y, jacc, 255)[0, 0, :, 0].cpu().numpy()


@pytest.mark.parametrize("k", [2, 3, 7, 13, 18, 25, 31])
@pytest.mark.parametrize("n", [20000, 20001])
def test_smallest_probabilities(native, k, n):
    t = -torch.linspace(60.0, 104.0, n, device="cuda")
    e = first_probability(native, t, 1, 32)             # the sum is 1
    assert e[0] > 0 and (e[e > 0] < 2.0 ** -126).any()
    want = e / np.float32(k)
    units = np.abs(first_probability(native, t, k, 32).view(np.int32) - want.view(np.int32))
    # below 2^-126 a quotient can lie half-way between two numbers (k = 18: one in nine), and its last step rounds by the residual
    twice = e.astype(np.float64) / k * 2.0 ** 150
    assert (units <= (twice % 2 == 1)).all()


# one block's row, buckets of every table size up to the longest row, radix passes below and above that length
@pytest.mark.parametrize("n_cls, pixels, positives", [(2, 5, 0.5), (3, 7680, 0.3), (32, 20011, 0.5), (32, 300007, 0.9), (6, 2560 * 1024, 0.5),
                                                      (6, 2560 * 1024, 0.02), (2, 50021, 0.5), (2, 2560 * 1024 + 1, 0.5),
                                                      (2, 2 ** 24 - 1, 0.5), (2, 2 ** 24 - 1, 0.98)])
def test_jaccard_differences(native, n_cls, pixels, positives):
    """Class 0's errors fall from pixel to pixel, or stay where the keys do: ranks are pixel numbers. Runs of equal logits are all
    positive or all negative; neighbouring runs are 20 units and more apart in the error's last place."""
    rng = np.random.default_rng(pixels + n_cls)
    runs = min(pixels, 20000)
    run = np.arange(pixels, dtype=np.int64) * runs // pixels
    hot = rng.random(runs) < positives
    hot[0] = True
    hot = hot[run]
    logit = np.linspace(6.0, -6.0, runs, dtype=np.float32)[run]
    x = torch.full((1, n_cls, 1, pixels), float("-inf"), device="cuda")
    x[0, 0, 0] = torch.from_numpy(np.where(hot, -logit, logit)).cuda()
    x[0, 1] = 0.0
    y = torch.from_numpy(np.where(hot, 0, 1)).view(1, 1, pixels).cuda()
    _, jacc = native.lovasz_forward(x, y, 255)
    inter = (hot.sum() - np.cumsum(hot)).astype(np.float32)
    index = np.float32(1) - inter / (inter + np.arange(1, pixels + 1, dtype=np.float32))
    want = np.diff(index, prepend=np.float32(0))
    assert np.array_equal(jacc[0].cpu().numpy().view(np.int32), want.view(np.int32))
