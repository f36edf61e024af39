"""The append's corrected product against the division it replaces (common.h, quant_unit), in
exact rational arithmetic, at every pair of float32 numbers that could separate their codes."""

from fractions import Fraction

from tests.division_pairs import corrected, dangerous_pairs, nearest32


def test_corrected_product_gives_the_divisions_codes():
    # int8 ties are k + 1/2 (t < 254), FP8 ties have 5 or 4 significant bits
    pairs = dangerous_pairs(range(1, 255, 2))
    assert len(pairs) > 500
    for t, x, b in pairs:
        x, b = Fraction(x), Fraction(b)
        assert corrected(x, b) == nearest32(x / b), (t, x, b)


def test_pairs_are_where_the_plain_product_fails():
    """The enumeration is of the quotients that matter: among them x * RN(1 / b) does miss
    the division."""
    missed = sum(nearest32(Fraction(x) * nearest32(1 / Fraction(b))) !=
                 nearest32(Fraction(x) / Fraction(b)) for _, x, b in dangerous_pairs([3, 129, 253]))
    assert missed > 0
