"""The rule by which the kernels of many rows take four planes' weights for fp16 numbers (may_round of lut_dequant_device.h, the form
that rounds every multiplier to a multiple of 2^-10 of the sum's binade), restated in numpy: what it takes for exact is exact."""
import itertools

import numpy as np
import pytest

PLANES = [  # scales of the four planes: both sides of the line
    (1024, 512, 256, 255), (1025, 513, 257, 252), (1025, 513, 257, 253), (1025, 513, 257, 255), (1025, 513, 257, 256), (1024, 512, 256, 257),
    (2046, 1, 1, 1), (2047, 1, 1, 2), (1, 2, 4, 2040), (0, 0, 3, 0), (0, 0, 0, 0), (5, 0, 1023, 0), (1.5, 0.75, 0.375, 1.125),
    (1 + 2 ** -10, 1, 2, 4), (4, 2, 1, 2 ** -8), (4, 2, 1, 2 ** -9), (2.0 ** -24, 2.0 ** -23, 3 * 2.0 ** -24, 0), (-1024, 511, -256, 255),
]
UNIFORM_SCALES = [  # alpha, q_bias: the planes are alpha / 2, / 4, / 8, / 16
    (16, 2032), (16, 2033), (16, 2034), (16, -2034), (-16, 2031), (2, 2.0 ** -9), (2, 2.0 ** -10), (2, 2.0 ** -11), (0, 3), (0, 0),
    (2.0 ** -14, 2.0 ** -10), (1.001953125, 0.25),
]


def entries(scales, uniform):
    """The sums that weights take, exact in fp64."""
    planes, q = (([scales[0] / 2 ** (b + 1) for b in range(4)], scales[1]) if uniform else (scales, 0.0))
    return [sum(s * float(np.float16(a) if not uniform else a) for s, a in zip(signs, planes)) + q for signs in itertools.product((-1, 1), repeat=4)]


def exact(sums):
    with np.errstate(over="ignore"):
        return all(float(np.float16(v)) == v for v in sums)


def may_round(multipliers):
    """may_round<4, UNI, false>, in 32 bits."""
    f = np.float32
    total = f(0)
    for v in multipliers:
        total = f(total + abs(f(v)))
    below = (total.view(np.uint32) & np.uint32(0x7f800000)).view(f)
    magic = f(max(below, f(2.0 ** -14)) * f(1.5 * 2 ** 13))
    if not total <= f(32768):
        return True
    return any(not f(f(f(v) + magic) - magic) == f(v) for v in multipliers)


@pytest.mark.parametrize("uniform", [False, True])
def test_nothing_inexact_is_taken_for_exact(uniform):
    rng = np.random.default_rng(7)
    taken = 0
    for i in range(6000):
        bits = rng.integers(1, 12)                     # of the multipliers, so that both answers occur
        if uniform:
            scales = tuple(float(np.float16(rng.integers(-2 ** bits, 2 ** bits) * 2.0 ** rng.integers(-20, 4))) for _ in range(2))
            multipliers = [scales[0] / 2 ** (b + 1) for b in range(4)] + [scales[1]]
        else:
            scales = tuple(float(np.float16(rng.integers(-2 ** bits, 2 ** bits) * 2.0 ** (rng.integers(-24, 4) if i % 2 else -12))) for _ in range(4))
            multipliers = scales
        if not may_round(multipliers):
            taken += 1
            assert exact(entries(scales, uniform)), scales
    assert 1000 < taken < 5000
    for scales in UNIFORM_SCALES if uniform else PLANES:
        multipliers = [scales[0] / 2 ** (b + 1) for b in range(4)] + [scales[1]] if uniform else scales
        assert may_round(multipliers) or exact(entries(scales, uniform)), scales


def test_the_line():
    """Sums of magnitudes under 2048 units are taken for exact, anything that needs a twelfth bit is not."""
    assert not may_round((1024, 512, 256, 255)) and not may_round((1025, 513, 257, 252)) and may_round((1025, 513, 257, 256))
    assert not may_round((2.0 ** -24, 2.0 ** -23, 3 * 2.0 ** -24, 0)) and may_round((2.0 ** -25, 0, 0, 0))
    assert not may_round((0, 0, 0, 0)) and may_round((float("inf"), 0, 0, 0)) and may_round((float("nan"), 0, 0, 0))
    assert may_round((30000, 2000, 800, 0)) and not may_round((16384, 8192, 4096, 2048))
