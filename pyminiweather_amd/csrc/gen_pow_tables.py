"""Writes pmw_pow_tables.h: the tables of pmw_pow.h, computed with Python's
decimal module at 60 digits and rounded to doubles.

    python gen_pow_tables.py > pmw_pow_tables.h

* log: for j = 0..128, c_j = 1/(1 + j/128) rounded to 8 significant bits,
  so that r = m*c_j - 1 is exact in one fma for m within 1/256 of 1 + j/128;
  and -ln(c_j) as a double-double.
* exp: 2^(j/256), j = 0..255, as a double-double (pow_pos_fast takes every
  4th entry, 2^(j/64)).
* gamma: for j = 0..511, c_j = 1/(1 + (j + 1/2)/512) rounded to 10 bits, so
  that r = m*c_j - 1 is exact in one fma for m in [1 + j/512, 1 + (j+1)/512)
  (|r| <= 2^-9), c_j^-gamma as a double-double and c_j^(1-gamma); and for
  every biased exponent e of a double 2^((e-1023) gamma) as a double-double
  (up to the largest whose power stays finite, then one NaN) and
  2^((e-1023) (gamma-1)).
  gamma is the double nearest to the physical constant.
"""
import math
from decimal import Decimal, getcontext

getcontext().prec = 60
GAMMA = 1.40027894002789400278940027894  # as a double: the exponent the kernels use


def rn(d):
    return float(d)  # correctly rounded (float(Decimal) rounds to nearest)


def dd(d):
    h = rn(d)
    return h, rn(d - Decimal(h))


def round_bits(d, bits):
    """d (in (0.5, 1]) rounded to `bits` significant bits, as a Decimal."""
    scale = Decimal(2) ** bits
    return (d * scale).to_integral_value() / scale


def main():
    out = ["// generated by gen_pow_tables.py -- do not edit", "#pragma once", "",
           "namespace pmw {", "namespace powt {", ""]
    cs, lh, ll = [], [], []
    for j in range(129):
        c = round_bits(Decimal(1) / (1 + Decimal(j) / 128), 8)
        assert Decimal(rn(c)) == c
        h, l = dd(-c.ln())
        cs.append(rn(c)); lh.append(h); ll.append(l)
    th, tl = [], []
    for j in range(256):
        h, l = dd(Decimal(2) ** (Decimal(j) / 256))
        th.append(h); tl.append(l)

    gamma = Decimal(GAMMA)
    gm = []  # c, hi and lo of c^-gamma, c^(1-gamma)
    for j in range(512):
        c = round_bits(1 / (1 + (Decimal(j) + Decimal("0.5")) / 512), 10)
        for m in (1 + Decimal(j) / 512, 1 + Decimal(j + 1) / 512):
            assert abs(m * c - 1) <= Decimal(2) ** -9
        lc = c.ln()
        gm += [rn(c), *dd((-gamma * lc).exp()), rn(((1 - gamma) * lc).exp())]
    ln2 = Decimal(2).ln()
    ge, gd = [], []
    for e in range(2048):
        k = e - 1023
        if e <= 1023 + 731:  # 2^(731 gamma) is the last below 2^1024
            ge += dd((k * gamma * ln2).exp()) if e else (0.0, 0.0)
        gd.append(rn((k * (gamma - 1) * ln2).exp()))

    last = len(ge) // 2
    ge += (math.nan, math.nan)

    def num(v):
        return "__builtin_nan(\"\")" if math.isnan(v) else float.hex(v)

    def arr(name, vals, align=False):
        a = "alignas(32) " if align else ""
        out.append(f"{a}constexpr double {name}[{len(vals)}] = {{")
        for i in range(0, len(vals), 4 if align else 3):
            row = vals[i:i + (4 if align else 3)]
            out.append("    " + ", ".join(num(v) for v in row) + ",")
        out.append("};")
    arr("kLogC", cs)
    arr("kLogHi", lh)
    arr("kLogLo", ll)
    arr("kExpHi", th)
    arr("kExpLo", tl)
    arr("kGamC", gm, align=True)
    arr("kGamE", ge, align=True)
    arr("kGamD", gd, align=True)
    out.append(f"constexpr unsigned kGamELast = {last};")
    # ln2/N with 31 significant bits (k * hi exact for |k| < 2^22)
    for n in (64, 256):
        scaled = ln2 / n
        e = 0
        while scaled * Decimal(2) ** e < Decimal(2) ** 30:
            e += 1
        hi = (scaled * Decimal(2) ** e).to_integral_value() / Decimal(2) ** e
        out.append(f"constexpr double kLn2_{n}Hi = {float.hex(rn(hi))};")
        out.append(f"constexpr double kLn2_{n}Lo = {float.hex(rn(scaled - hi))};")
        out.append(f"constexpr double k{n}InvLn2 = {float.hex(rn(n / ln2))};")
    h = (ln2 * Decimal(2) ** 31).to_integral_value() / Decimal(2) ** 31
    out.append(f"constexpr double kLn2Hi = {float.hex(rn(h))};")
    out.append(f"constexpr double kLn2Lo = {float.hex(rn(ln2 - h))};")
    out += ["", "}  // namespace powt", "}  // namespace pmw", ""]
    print("\n".join(out))


if __name__ == "__main__":
    main()
