"""The division of whole numbers that the Lovasz bucket kernels write out (one residual, for unions of up to 2560 * 1024), and the one of
the radix passes (two residuals), in float32 on the CPU: the quotients nearest to half-way between two numbers, with the hardware's
reciprocal anywhere within a unit of the true one."""
import numpy as np
import pytest


def divide(a, b, y, residuals):
    """Fused multiply-adds rounded once: their products are exact in 64 significant bits, and what rounding the sum there first loses is far
    below the distance of any quotient here from half-way (1 / 2b of a unit)."""
    def fma(p, q, r):
        return (p.astype(np.longdouble) * q.astype(np.longdouble) + r).astype(np.float32)
    y = fma(fma(-b, y, np.float32(1)), y, y)
    q = a * y
    for _ in range(residuals):
        q = fma(fma(-b, q, a), y, q)
    return q


def near_half_way(rng, least, most, n):
    """Whole a <= b with a / b = (odd + eps / b) / 2^(25 + t) units: 1, 3 or 5 parts in 2b off."""
    out_a, out_b = [], []
    while sum(map(len, out_a)) < n:
        b = rng.integers(least, most, 4096, dtype=np.int64) | 1
        inverse = np.ones_like(b)
        for _ in range(6):
            inverse = inverse * (2 - b * inverse)           # modulo 2^64
        for t in range(4):
            for eps in (-5, -3, -1, 1, 3, 5):
                half = (-eps * inverse) & ((1 << (25 + t)) - 1)
                a = (half * b + eps) >> (25 + t)
                ok = (half >> 24 == 1) & (half & 1 == 1) & (a > 0) & (a <= b)
                out_a.append(a[ok])
                out_b.append(b[ok])
    return np.concatenate(out_a).astype(np.float32), np.concatenate(out_b).astype(np.float32)


# (unions from 2^23 on: a reciprocal a unit off fails the division operator's steps too, which are those of two residuals)
@pytest.mark.parametrize("least, most, residuals, off", [(1, 4096, 1, 1), (4096, 1 << 17, 1, 1), (1 << 17, 2560 * 1024, 1, 1),
                                                         (1 << 21, 2560 * 1024, 1, 1), (1 << 21, 2560 * 1024, 2, 1),
                                                         (2560 * 1024, 1 << 23, 2, 1), (1 << 23, 1 << 24, 2, 0)])
def test_quotients_near_half_way(least, most, residuals, off):
    a, b = near_half_way(np.random.default_rng(most), least, most, 200000)
    true = (1.0 / b.astype(np.float64)).astype(np.float32)
    for unit in range(-off, off + 1):
        y = (true.view(np.int32) + unit).view(np.float32)
        assert np.array_equal(divide(a, b, y, residuals), a / b), unit
