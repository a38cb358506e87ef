"""The table-based double exponential of the verify kernels (exp_sum,
shared_amd/csrc/verify_kernel.hip) restated in exact arithmetic with one
rounding per operation: its table and constants are read from the source, its
error is within what the comment there states."""
import os
import random
import re
from decimal import Decimal, getcontext
from fractions import Fraction

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "shared_amd", "csrc",
                   "verify_kernel.hip")
getcontext().prec = 60
LN2 = Decimal(2).ln()


def _source():
    with open(SRC) as f:
        s = f.read()
    table = s[s.index("kExp2Tab[kExpTab] = {"):]
    table = table[:table.index("};")]
    return s, [(float.fromhex(a), float.fromhex(b)) for a, b in
               re.findall(r"\{(-?0x[0-9a-fp.+-]+), (-?0x[0-9a-fp.+-]+|0\.0)\}", table)]


def _fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))  # rounded once


def test_table_is_two_to_the_j_over_64():
    _, tab = _source()
    assert len(tab) == 64
    for j, (hi, lo) in enumerate(tab):
        exact = (LN2 * j / 64).exp()
        assert hi == float(exact)
        # what the high part leaves, to its own nearest double
        assert abs(Decimal(lo) - (exact - Decimal(hi))) <= abs(exact - Decimal(hi)) * Decimal(2) ** -53 + Decimal("1e-45")


def test_error_of_exp_sum():
    src, tab = _source()
    for constant in ("0x1.71547652b82fep+6", "0x1.a39ef35793c76p-39", "0x1.62e42fee00000p-7", "6755399441055744.0"):
        assert constant in src
    scale, ln2_lo, ln2_hi = (float.fromhex(c) for c in
                             ("0x1.71547652b82fep+6", "0x1.a39ef35793c76p-39", "0x1.62e42fee00000p-7"))

    def exp_sum(x):
        k = round(_fma(x, scale, 6755399441055744.0) - 6755399441055744.0)
        hi, lo = tab[k % 64]
        r = _fma(-k, ln2_lo, _fma(-k, ln2_hi, x))
        q = _fma(_fma(_fma(r, 1 / 120, 1 / 24), r, 1 / 6), r, 0.5)
        p = _fma(r * r, q, r)
        return (hi + _fma(hi, p, lo)), k // 64

    rng = random.Random(5)
    xs = [-rng.uniform(0, 700) for _ in range(2500)] + [-rng.uniform(0, 1) for _ in range(1000)]
    # around every boundary between table entries of the first octave and a far one
    for k in range(64):
        for base in (0, 300 * 64):
            m = -float(LN2 * (base + k) / 64 + LN2 / 128)
            xs += [m * (1 - 2e-15), m, m * (1 + 2e-15)]
    worst, total = 0.0, 0.0
    for x in xs:
        y, e = exp_sum(x)
        exact = Decimal(x).exp()
        scaled = exact * Decimal(2) ** -e
        ulp = Decimal(2) ** (-52 if scaled >= 1 else -53)
        err = float(abs(Decimal(y) - scaled) / ulp)
        worst, total = max(worst, err), total + err * err
    print(f"worst {worst:.3f} ulp, rms {(total / len(xs)) ** 0.5:.3f}")
    assert worst <= 0.82  # the comment's bound
    assert (total / len(xs)) ** 0.5 <= 0.33  # 0.296 over [-700, 0]; the boundaries and [-1, 0] are harder
