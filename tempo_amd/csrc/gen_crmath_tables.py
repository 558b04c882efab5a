"""Write tempo_crmath_tables.inc: the constants of the double-double
exp/log kernels in tempo_crmath.hpp, evaluated to 60 significant digits with
Python's decimal module and split into double-precision hi/lo parts.

    python tempo_amd/csrc/gen_crmath_tables.py
"""
import os
from decimal import Decimal, getcontext

getcontext().prec = 60
HERE = os.path.dirname(os.path.abspath(__file__))


def split(d):
    """d ~ hi + lo with hi = nearest double, lo = nearest double of the rest."""
    hi = float(d)
    lo = float(d - Decimal(hi))
    return hi, lo


def trunc_bits(x, bits):
    """x rounded toward zero to `bits` significant bits (so n*x is exact for small n)."""
    import math
    m, e = math.frexp(x)
    scale = 2 ** bits
    return math.ldexp(math.floor(m * scale) / scale, e)


def main():
    ln2 = Decimal(2).ln()
    ln10 = Decimal(10).ln()
    lines = ["// Generated by gen_crmath_tables.py -- do not edit.", ""]
    # 2^(j/64), j = 0..63, as (hi, lo) pairs, so that one 16-byte load fetches an entry
    lines.append("alignas(16) static constexpr double kExp2Tab[64][2] = {")
    for j in range(64):
        hi, lo = split((ln2 * j / 64).exp())
        lines.append(f"    {{{hi.hex()}, {lo.hex()}}},")
    lines.append("};")
    # Cody-Waite split of ln2/64: c1 has 32 significant bits (n*c1 exact for |n| < 2^21)
    l64 = ln2 / 64
    c1 = trunc_bits(float(l64), 32)
    rest = l64 - Decimal(c1)
    c2 = float(rest)
    c3 = float(rest - Decimal(c2))
    inv = float(64 / ln2)
    # ln2 = lh + ll with lh holding 40 significant bits (e*lh exact for |e| < 2^13)
    lh = trunc_bits(float(ln2), 40)
    ll = float(ln2 - Decimal(lh))
    ih, il = split(1 / ln10)
    th, tl = split(ln10)
    for name, v in (("kInvLn2x64", inv), ("kLn2o64C1", c1), ("kLn2o64C2", c2), ("kLn2o64C3", c3),
                    ("kLn2Hi", lh), ("kLn2Lo", ll), ("kInvLn10Hi", ih), ("kInvLn10Lo", il),
                    ("kLn10Hi", th), ("kLn10Lo", tl)):
        lines.append(f"static constexpr double {name} = {v.hex()};")
    with open(os.path.join(HERE, "tempo_crmath_tables.inc"), "w") as f:
        f.write("\n".join(lines) + "\n")


if __name__ == "__main__":
    main()
