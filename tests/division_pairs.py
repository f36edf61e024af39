"""Quotients where the append's corrected product could miss the division's code.

With inv = RN(1 / b), q = RN(x inv), r = RN(x - q b), the corrected q' = RN(q + r inv) rounds
a value within 3 * 2^-24 steps of x / b (q is within 1.5 steps; inv and r within 2^-24 of
themselves), so that it can differ from RN(x / b) only where x / b lies that near a rounding
boundary of float32. Its code can then differ only where the boundary is the one above or below
a tie t 2^e of two codes (t odd). With 24-bit integers X 2^j = B M + d, M the boundary in half
steps (25 bits), that is |d| <= 6: for every t, side and d the pairs (X, B) follow from
B = -d / M mod 2^j."""

from fractions import Fraction

import numpy as np


def dangerous_pairs(odd, reach=8):
    """(t, x, b) as floats, x / b within ``reach`` (|d|) of the boundary beside a tie with
    significand t, for the odd numbers ``odd``; x and b in [1, 2)."""
    out = []
    for t in odd:
        for side in (-1, 1):
            bits = 26 if t == 1 and side < 0 else 25  # below a power of two the steps halve
            m = (t << (bits - t.bit_length())) + side
            for d in range(-reach, reach + 1):
                for j in range(23, 28):
                    mod = 1 << j
                    for b in range(-d * pow(m, -1, mod) % mod, 1 << 24, mod):
                        x, rest = divmod(b * m + d, mod)
                        if b >= 1 << 23 and rest == 0 and 1 << 23 <= x < 1 << 24:
                            out.append((t, x / 2.0 ** 23, b / 2.0 ** 23))
    return out


def nearest32(value):
    """A positive or negative rational rounded to float32 (half to even, no exponent limits)."""
    if value == 0:
        return Fraction(0)
    step = Fraction(2) ** (int(np.floor(np.log2(abs(float(value))))) - 23)
    while abs(value) / step >= 1 << 24:
        step *= 2
    while abs(value) / step < 1 << 23:
        step /= 2
    return round(value / step) * step  # Fraction's round is half to even


def corrected(x, b):
    inv = nearest32(1 / b)
    q = nearest32(x * inv)
    return nearest32(q + nearest32(x - q * b) * inv)
