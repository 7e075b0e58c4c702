"""The coarsest AMG solve divides by a row's diagonal from its reciprocal: two
fma refinements of a * RN(1 / d).  This checks the method, not the kernel: restated
with exact rational arithmetic for the fmas, the quotient is the correctly
rounded one.  The device's quotients are compared with true ones, inside and
outside the method's range, in test_gpu_amg.py (test_coarsest_quotients)."""
import random
import struct
from fractions import Fraction


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def test_quotient_is_correctly_rounded():
    rng = random.Random(7)
    for t in range(20000):
        a, d = (rng.uniform(1, 2) * 2.0 ** rng.randint(-390, 390) * rng.choice((-1, 1))
                for _ in range(2))
        if t % 3 == 0:  # mantissas of ones: the hardest reciprocals
            d = struct.unpack("d", struct.pack("Q", struct.unpack("Q", struct.pack("d", d))[0]
                                               | ((1 << 52) - 1 - (1 << rng.randint(0, 6)))))[0]
        y = 1.0 / d
        q0 = a * y
        q1 = fma(fma(-d, q0, a), y, q0)
        assert fma(fma(-d, q1, a), y, q1) == a / d, (a, d)
