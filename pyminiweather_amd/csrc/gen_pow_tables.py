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
  (|r| <= 2^-9); for the sixteen binades from 2^-6, entry 512 o + j: the power
  (2^(o-6) / c_j)^gamma as a double and a float of its rest, and c_j as a float
  (kGamQ); and for other binades e, whose significands use the entries of binade
  (e+6) mod 16 - 6, 2^(16 (i-64) gamma) for i = 0.. as a double-double, times
  2^64 for i < 36 and 2^-64 for i >= 100, up to the last i with a finite power,
  then one NaN (kGamE).
* gamma - 1: c_j^(1-gamma) and c_j (kGamM), and for every biased exponent e of
  a double 2^((e-1023) (gamma-1)) (kGamD).
  gamma is the double nearest to the physical constant.
"""
import math
import struct
from decimal import Decimal, getcontext

getcontext().prec = 60
GAMMA = 1.40027894002789400278940027894  # as a double: the exponent the kernels use


def rn(d):
    return float(d)  # correctly rounded (float(Decimal) rounds to nearest)


def dd(d):
    h = rn(d)
    return h, rn(d - Decimal(h))


def f32(d):
    return struct.unpack("f", struct.pack("f", float(d)))[0]  # rounds to nearest


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
    ln2 = Decimal(2).ln()
    gq, gm = [], []
    for i in range(8192):
        o, j = divmod(i, 512)
        c = round_bits(1 / (1 + (Decimal(j) + Decimal("0.5")) / 512), 10)
        for m in (1 + Decimal(j) / 512, 1 + Decimal(j + 1) / 512):
            assert abs(m * c - 1) <= Decimal(2) ** -9
        lx = (o - 6) * ln2 - c.ln()
        h, l = dd((gamma * lx).exp())
        gq.append((h, f32(l), f32(c)))
        assert Decimal(f32(c)) == c
        if o == 0:
            gm += [rn(((1 - gamma) * c.ln()).exp()), rn(c)]
    ge, gd = [], []
    for i in range(111):
        lift = 64 if i < 36 else -64 if i >= 100 else 0  # clear of subnormals and overflow
        ge += dd(((16 * (i - 64) * gamma + lift) * ln2).exp())
    for e in range(2048):
        gd.append(rn(((e - 1023) * (gamma - 1) * ln2).exp()))

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
    out.append("struct alignas(16) GamQ {\n  double h;\n  float l, c;\n};")
    out.append(f"constexpr unsigned kGamEntries = {len(gq)};")
    out.append(f"constexpr GamQ kGamQ[{len(gq)}] = {{")
    out.extend("    {%s, %sf, %sf}," % tuple(float.hex(v) for v in q) for q in gq)
    out.append("};")
    arr("kGamM", gm, align=True)
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
