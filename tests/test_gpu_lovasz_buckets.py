"""The Lovasz forward's sort by value buckets against the look-back variant, which sorts the same keys by radix passes: the
Jaccard differences have to be the same bit for bit (same ranks, equal keys in pixel order), and so do the losses: their terms
are exact in double and added in double, in an order of its own per path, so that the sums are some 2^-50 of their value
apart before they are rounded to float (equal for these inputs; for one in some 2^26 a rounding would fall between). Rows at the limits of the paths (one block, each number of buckets), values that crowd: ties,
clusters, one value only, rows without positives, and buckets that outgrow a block because the sampled bounds miss them."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def native():
    from pytorch_loss import _native
    _native.load()
    return _native


def labels(rng, shape, n_cls, ignored=0.1):
    y = rng.integers(0, n_cls, shape)
    y[rng.random(shape) < ignored] = 255
    return y


def compare(native, x, y):
    xt, yt = torch.as_tensor(x).cuda(), torch.as_tensor(y).cuda()
    want_l, want_j = native.lovasz_forward(xt, yt, 255, look_back=True)
    for _ in range(2):
        losses, jacc = native.lovasz_forward(xt, yt, 255)
        assert torch.equal(jacc.view(torch.int32), want_j.view(torch.int32))
        assert torch.equal(losses, want_l) and not torch.isnan(losses).any()
    return losses


def by_buckets(n_cls, pixels):
    """The route of a row, by its workspace: 10 bytes per key and tables (buckets), 16 and tables (radix passes)."""
    from pytorch_loss import _native
    return _native.load().plh_lovasz_workspace_bytes(1, n_cls, pixels) < 16 * n_cls * pixels


def test_which_rows_go_by_buckets(native):
    """Few classes of more pixels than one block holds went by buckets at first, up to three quarters slower than by radix
    passes where predictions are confident (2 classes of 262144 pixels: 102 -> 180 us)."""
    many = 2560 * 1024
    for n_cls, pixels, want in [(2, 7681, False), (2, 65536, False), (2, 262144, False), (2, many, False), (4, 263169, False),
                                (4, many, False), (8, 262144, False), (16, 65536, False), (19, 90300, False), (31, 65536, False),
                                (6, many, True), (8, 1048576, True), (16, 262144, True), (19, 4 * 512 * 1024, True),
                                (32, 65536, True), (150, 65536, True), (19, many + 1, False)]:
        assert by_buckets(n_cls, pixels) == want, (n_cls, pixels)


@pytest.mark.parametrize("boost", [0.0, 20.0])
@pytest.mark.parametrize("n_cls, pixels, want", [(12, 393216, True), (12, 393215, False), (12, 291272, False), (17, 170000, False),
                                                 (18, 131072, True), (18, 131071, False), (22, 131072, True), (22, 131071, False),
                                                 (11, 350000, False)])
def test_rows_of_a_single_image(native, n_cls, pixels, want, boost):
    """Where 12 classes and more begin to go by buckets: the same differences on both sides of the line. With 12 to 17 classes it
    lay at 5 2^23 = pixels x classes^2 at first, where a network that is sure by 17 loses a tenth (14 of 213996 170 -> 186 us)."""
    assert by_buckets(n_cls, pixels) == want
    rng = np.random.default_rng(pixels + n_cls)
    x = rng.standard_normal((1, n_cls, 1, pixels), dtype=np.float32) * 2
    y = labels(rng, (1, 1, pixels), n_cls)
    x += np.float32(boost) * (np.arange(n_cls)[None, :, None, None] == y[:, None])
    compare(native, x, y)


# pixels: one block's limit, 64 / 256 / 1024 buckets, the longest row that is cut into buckets and the first that is not
# classes: few (radix passes above one block's limit) and enough for buckets
@pytest.mark.parametrize("pixels", [1, 63, 512, 513, 7679, 7680, 7681, 8193, 20011, 2560 * 64, 2560 * 64 + 1, 2560 * 256 + 7])
@pytest.mark.parametrize("boost", [0.0, 10.0])
@pytest.mark.parametrize("n_cls", [3, 33])
def test_row_lengths(native, pixels, boost, n_cls):
    assert n_cls == 3 or pixels < 1000 or by_buckets(n_cls, pixels)
    rng = np.random.default_rng(pixels)
    x = rng.standard_normal((1, n_cls, 1, pixels), dtype=np.float32) * 2
    y = labels(rng, (1, 1, pixels), n_cls)
    x += np.float32(boost) * (np.arange(n_cls)[None, :, None, None] == y[:, None])
    losses = compare(native, x, y)
    if pixels < 10000 and not boost:
        want, _ = oracle.lovasz_forward(x.astype(np.float64), y, 255)
        np.testing.assert_allclose(losses.cpu().numpy(), want, rtol=1e-5)


@pytest.mark.parametrize("pixels", [1024 * 2560, 1024 * 2560 + 1])
@pytest.mark.parametrize("n_cls", [2, 6])
def test_longest_rows(native, pixels, n_cls):
    assert by_buckets(n_cls, pixels) == (n_cls == 6 and pixels == 1024 * 2560)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((1, n_cls, 1, pixels), device="cuda", generator=g)
    y = torch.randint(0, n_cls, (1, 1, pixels), device="cuda", generator=g)
    compare(native, x, y)


@pytest.mark.parametrize("pixels", [5000, 40000, 300000])
@pytest.mark.parametrize("kind", ["constant", "few values", "half steps", "cluster", "two clusters", "certain", "absent", "halves"])
@pytest.mark.parametrize("many", [False, True])
def test_crowded_values(native, pixels, kind, many):
    rng = np.random.default_rng(len(kind) + pixels)
    n_cls = 32 if many else (2 if kind in ("few values", "half steps") else 4)
    assert not many or by_buckets(n_cls, pixels)
    x = rng.standard_normal((1, n_cls, 1, pixels), dtype=np.float32)
    y = labels(rng, (1, 1, pixels), n_cls)
    if kind == "constant":              # every error the same
        x[:] = 0
    elif kind == "few values":          # ties by the thousand
        x = np.round(x)
    elif kind == "half steps":
        x = np.round(x * 64) / 64
    elif kind == "cluster":             # a new network: probabilities within 1e-5 of each other
        x *= np.float32(1e-5)
    elif kind == "two clusters":
        x = x * np.float32(1e-6) + np.float32(3) * (rng.random(x.shape) < 0.5)
    elif kind == "certain":             # probabilities of exactly 1, and the steps of 2^-24 below
        x += np.float32(17) * (np.arange(n_cls)[None, :, None, None] == y[:, None])
    elif kind == "halves":              # one value, 1/2, for the positives and the others of two classes; 0 for the others
        x[:] = -200
        x[:, :2] = 0
        y = np.where(y == 255, 255, y % 2)
    else:                               # classes that no pixel has
        y[:] = np.where(y == 255, 255, 1)
    compare(native, x.astype(np.float32), y)


def sampled(pixels):
    """The positions that the bucket bounds are chosen from (csrc/lovasz_buckets.hpp, bk_sample)."""
    i = np.arange(7680, dtype=np.uint64)
    h = (i * 0x9E3779B1) & 0xFFFFFFFF
    h = ((h ^ (h >> 15)) * 0x85EBCA6B) & 0xFFFFFFFF
    return i * pixels // 7680 + ((h * (pixels // 7680)) >> 32)


# most keys in one bucket: up to four times what a block holds, and more
@pytest.mark.parametrize("pixels", [20000, 70000, 500000])
@pytest.mark.parametrize("kind", ["spread", "one value", "both", "nested"])
@pytest.mark.parametrize("n_cls", [2, 32])
def test_buckets_that_the_sample_misses(native, pixels, kind, n_cls):
    assert n_cls == 2 or by_buckets(n_cls, pixels)
    rng = np.random.default_rng(pixels)
    d = rng.random(pixels) * (0.0 if kind == "one value" else 1e-2)
    if kind == "both":
        d[rng.random(pixels) < 0.5] = 5e-3
    if kind == "nested":                # a cluster in a cluster, and values that more keys share than a block holds
        d = 10.0 ** -rng.integers(0, 6, pixels) * rng.random(pixels)
        d[rng.random(pixels) < 0.3] = 0.25
    at = sampled(pixels).astype(np.int64)
    d[at] = 1 + rng.random(at.size)
    # the classes beyond the first two are absent, and hardly predicted
    x = np.stack([d, np.zeros(pixels)] + [np.full(pixels, -30.0)] * (n_cls - 2))[None, :, None, :].astype(np.float32)
    compare(native, x, labels(rng, (1, 1, pixels), 2))


# how many buckets the 64 neighbouring keys of a wave lie in: one (no vote), a few that all are met, many that few are met
@pytest.mark.parametrize("ways", [1, 2, 7, 16, 33, 64])
@pytest.mark.parametrize("pixels", [8192, 70001, 2560 * 256 + 4095])
def test_neighbours_in_few_buckets(native, ways, pixels):
    assert by_buckets(32, pixels)
    rng = np.random.default_rng(ways)
    per = -(-pixels // ways)
    order = np.sort(rng.standard_normal(per * ways).astype(np.float32) * 2)
    i = np.arange(pixels)
    x = rng.standard_normal((1, 32, 1, pixels), dtype=np.float32)
    x[0, 0, 0] = order[i % ways * per + i // ways]
    x[0, 1, 0] = np.where(rng.random(pixels) < 0.9, x[0, 0, 0], x[0, 1, 0])
    compare(native, x, labels(rng, (1, 1, pixels), 32))


@pytest.mark.parametrize("n_cls", [2, 19, 24, 32])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("plane", [(65, 67), (64, 65), (85, 121)])
def test_planes_of_odd_length(native, n_cls, dtype, plane):
    """Planes that start on element boundaries: the same as the pixels of four images side by side in one, whose planes start
    on the vector accesses' boundaries."""
    import pytorch_loss
    g = torch.Generator(device="cuda").manual_seed(n_cls + plane[0])
    x = (torch.randn((4, n_cls) + plane, device="cuda", generator=g) * 2).to(dtype)
    y = torch.randint(0, n_cls, (4,) + plane, device="cuda", generator=g)
    y[torch.rand(y.shape, device="cuda", generator=g) < 0.1] = 255
    side_x = x.flatten(2).transpose(0, 1).contiguous().unsqueeze(0)        # (1, C, 4, pixels of an image)
    side_y = y.flatten(1).unsqueeze(0)
    out = []
    for a, b in ((x, y), (side_x, side_y)):
        losses, jacc = native.lovasz_forward(a, b, 255)
        a = a.detach().requires_grad_()
        pytorch_loss.LovaszSoftmaxV3(ignore_index=255)(a, b).backward()
        out.append((losses, jacc, a.grad))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    assert torch.equal(out[0][2], out[1][2][0].transpose(0, 1).reshape(x.shape))


@pytest.mark.parametrize("pixels", [5000, 300000, 2560 * 1024, 2700000])
@pytest.mark.parametrize("gap", [18.5, 30.0])
@pytest.mark.parametrize("n_cls", [2, 32])
def test_small_losses_keep_their_digits(native, pixels, gap, n_cls):
    """A network that is all but certain: class losses down to 1e-14, whose terms are far below a loss's usual last bit. The
    errors follow from the logits (1 + exp(-gap) rounds to 1: the positives have none), the Jaccard differences from the
    forward, and the loss is the sum of their products. An error is good to some 2 units in its last place (expf), 3e-7."""
    rng = np.random.default_rng(pixels)
    y = rng.integers(0, 2, (1, 1, pixels))
    below = (gap + rng.integers(0, 64, pixels) / 64).astype(np.float32)
    x = np.full((1, n_cls, 1, pixels), -200.0, np.float32)          # classes that nothing predicts: exp(-200) is 0
    x[:, :2] = 0.0
    np.put_along_axis(x, 1 - y[:, None], -below[None, None, None, :], 1)
    xt, yt = torch.as_tensor(x).cuda(), torch.as_tensor(y).cuda()
    error = np.exp(-below.astype(np.float64))
    for look_back in (False, True):
        losses, jacc = native.lovasz_forward(xt, yt, 255, look_back=look_back)
        jacc = jacc[:2].cpu().numpy().astype(np.float64).reshape(2, pixels)
        for c in range(2):
            want = (error * jacc[c])[y.reshape(-1) != c].sum()
            assert abs(losses[c].item() - want) <= 1e-6 * want
