"""Generates pp_crmath_tables.h: the constants of the correctly rounded FP64
exp and log in pp_crmath.h, computed here with mpmath at 60 digits from their
definitions.

exp: x = k ln2/128 + r.  T[j] = 2^(j/128) as a double-double (hi, lo);
ln2/128 split as C1 (32 significant bits, so k*C1 is exact for |k| < 2^21),
C2, C3; the Taylor coefficients 1/k! as doubles (fast path) and as
double-doubles (slow path).

log: x = 2^e m with m in [0.75, 1.5), split into 96 intervals of width
1/128; interval j uses inv[j] = 1/(its centre) in double, rounded to 8
significant bits -- the device forms it with the same two operations -- and
L[j] = -log(inv[j]) as a double-double.  The two intervals around 1 use
inv = 1 and L = 0, so that log of x near 1 keeps its relative accuracy.
ln2 as a double-double (hi with 42 significant bits, so e*hi is exact), the
log1p coefficients (-1)^(k+1)/k as doubles and double-doubles.

    python pplacer_amd/csrc/gen_crmath_tables.py   # rewrites pp_crmath_tables.h
"""
import os

import mpmath as mp

mp.mp.dps = 60
HERE = os.path.dirname(os.path.abspath(__file__))


def rn(x):
    """x rounded to the nearest double (mpmath rounds to nearest, ties even)."""
    return float(mp.mpf(x))


def dd(x):
    hi = rn(x)
    lo = rn(mp.mpf(x) - mp.mpf(hi))
    return hi, lo


def round_bits(x, bits):
    """x rounded to `bits` significant bits (nearest)."""
    x = mp.mpf(x)
    if x == 0:
        return 0.0
    e = int(mp.floor(mp.log(abs(x), 2)))
    scale = mp.mpf(2) ** (bits - 1 - e)
    return float(mp.nint(x * scale) / scale)


def hexs(v):
    return float(v).hex()


def main():
    out = []
    w = out.append
    w("// Generated by gen_crmath_tables.py: constants of the correctly rounded")
    w("// FP64 exp and log (pp_crmath.h), computed with mpmath at 60 digits.")
    w("// The includer defines PP_CR_TAB (storage class of the arrays).")
    w("#pragma once")
    w("")
    ln2 = mp.log(2)
    # ---- exp
    c = ln2 / 128
    c1 = round_bits(c, 32)
    c2 = rn(c - c1)
    c3 = rn(c - c1 - c2)
    w("PP_CR_CST double pp_cr_exp_c[4] = {%s, %s, %s, %s};  // 128/ln2, ln2/128 = C1 + C2 + C3"
      % (hexs(rn(128 / ln2)), hexs(c1), hexs(c2), hexs(c3)))
    w("PP_CR_TAB double pp_cr_exp_t[256] = {  // 2^(j/128): hi, lo")
    for j in range(128):
        hi, lo = dd(mp.mpf(2) ** (mp.mpf(j) / 128))
        w("    %s, %s," % (hexs(hi), hexs(lo)))
    w("};")
    w("PP_CR_CST double pp_cr_exp_p[8] = {  // 1/k!, k = 0..7")
    w("    " + ", ".join(hexs(rn(1 / mp.factorial(k))) for k in range(8)) + ",")
    w("};")
    w("PP_CR_TAB double pp_cr_exp_pdd[28] = {  // 1/k!, k = 0..13: hi, lo")
    for k in range(14):
        hi, lo = dd(1 / mp.factorial(k))
        w("    %s, %s," % (hexs(hi), hexs(lo)))
    w("};")
    # ---- log
    ln2hi = round_bits(ln2, 42)
    ln2lo = rn(ln2 - ln2hi)
    ln2lo2 = rn(ln2 - ln2hi - ln2lo)
    w("PP_CR_CST double pp_cr_ln2[3] = {%s, %s, %s};  // ln2 = hi (42 bits) + lo + lo2"
      % (hexs(ln2hi), hexs(ln2lo), hexs(ln2lo2)))
    inv, Lhi, Llo = [], [], []
    umax = mp.mpf(0)
    for j in range(96):
        a = mp.mpf(3) / 4 + mp.mpf(j) / 128
        b = a + mp.mpf(1) / 128
        if j in (31, 32):  # [1 - 2^-7, 1 + 2^-7): no table step
            v = 1.0
        else:
            # the device's inv: 1/c in double (correctly rounded division),
            # then 8 significant bits (ties to even, as rint)
            c = 0.75 + (j + 0.5) * 0.0078125
            q = 1.0 / c
            v = round(q * 256.0) / 256.0 if q < 1.0 else round(q * 128.0) / 128.0
            assert v == round_bits(q, 8)
        inv.append(v)
        h, l = dd(-mp.log(mp.mpf(v)))
        Lhi.append(h)
        Llo.append(l)
        umax = max(umax, abs(a * mp.mpf(v) - 1), abs(b * mp.mpf(v) - 1))
    assert umax < mp.mpf(2) ** -6, umax
    w("// inv[j]: 1/(0.75 + (j + 0.5)/128) in double rounded to 8 significant bits, 1 for j = 31, 32;")
    w("// |m inv[j] - 1| < %.4g over every interval" % float(umax))
    w("PP_CR_TAB double pp_cr_log_l[192] = {  // -log(inv[j]): hi, lo")
    for j in range(96):
        w("    %s, %s," % (hexs(Lhi[j]), hexs(Llo[j])))
    w("};")
    w("PP_CR_CST double pp_cr_log_p[16] = {  // (-1)^(k+1)/k, k = 1..16")
    w("    " + ", ".join(hexs(rn(mp.mpf((-1) ** (k + 1)) / k)) for k in range(1, 17)) + ",")
    w("};")
    w("PP_CR_TAB double pp_cr_log_pdd[36] = {  // (-1)^(k+1)/k, k = 1..18: hi, lo")
    for k in range(1, 19):
        hi, lo = dd(mp.mpf((-1) ** (k + 1)) / k)
        w("    %s, %s," % (hexs(hi), hexs(lo)))
    w("};")
    with open(os.path.join(HERE, "pp_crmath_tables.h"), "w") as f:
        f.write("\n".join(out) + "\n")


if __name__ == "__main__":
    main()
