"""The device generators' last step, n / 1000 for n = -1000 .. 1000
(HashValue, csrc/pool_kernels.hip): its three operations, each correctly
rounded to float, give the correctly rounded quotient for every n."""
from fractions import Fraction

import numpy as np


def round_f32(x: Fraction) -> np.float32:
    """The float nearest to x (ties to even)."""
    near = np.float32(float(x))
    choices = [near, np.nextafter(near, np.float32(np.inf)), np.nextafter(near, np.float32(-np.inf))]
    return min(choices, key=lambda y: (abs(Fraction(float(y)) - x), int(y.view(np.uint32)) & 1))


def test_quotient_is_correctly_rounded():
    inv = Fraction(float(np.float32(0.001)))
    for n in range(-1000, 1001):
        q = Fraction(float(round_f32(n * inv)))
        rest = Fraction(float(round_f32(n - 1000 * q)))
        got = round_f32(rest * inv + q)
        assert got == round_f32(Fraction(n, 1000)) == np.float32(n) / np.float32(1000)
        # a planted slip, no correction, differs somewhere
    assert any(round_f32(n * inv) != np.float32(n) / np.float32(1000) for n in range(1, 1001))
