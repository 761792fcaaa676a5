"""Write moro_tail_f64.inc: the FP64 path kernels' inverse-normal tail.

The tail of the Beasley-Springer-Moro function (gaussians.h:47-87), a
polynomial in log(-log(v)) of the tail mass v = min(p, 1 - p) <= 0.08, is
smooth on every quarter of a binade of v.  Row r covers
v = (1 + q / 4 + [0, 1/4)) 2^e with r = 4 (e + 33) + q, e = -33 .. -4: the
upper 14 bits of the double less a constant.  Each row holds the twelve
coefficients, in d = v - (the row's midpoint), of the polynomial through
Chebyshev nodes of the row, formed in extended precision (64-bit mantissa)
and rounded once.  The subtraction is exact and the terms fall off by a
factor of 9 or more per order, so the result carries little more than the
rounding of its last multiply-add: within 2.0 half-ulps of the exact tail
(0.48 on average) over the Sobol words.  120 rows of 96 bytes; eighths of a
binade with ten coefficients are as accurate and take 19,200 bytes, sixteenths
with eight (2.7 half-ulps) 30,720.

    python compfinance_amd/csrc/gen_moro_tail_f64.py
"""
import os

import numpy as np

DEG = 11
PARTS = 4            # rows per binade: the top two mantissa bits
E_MIN, E_MAX = -33, -4
HERE = os.path.dirname(os.path.abspath(__file__))
LD = np.longdouble

C = ["0.3374754822726147", "0.9761690190917186", "0.1607979714918209", "0.0276438810333863", "0.0038405729373609",
     "0.0003951896511919", "0.0000321767881768", "0.0000002888167364", "0.0000003960315187"]


def tail(v):
    """Moro's tail in extended precision, its constants as doubles."""
    r = np.log(-np.log(np.asarray(v, dtype=LD)))
    p = np.full_like(r, LD(float(C[8])))
    for k in range(7, -1, -1):
        p = LD(float(C[k])) + r * p
    return p


def _monomials(y):
    """Monomial coefficients in t of the polynomial through the values y at
    the Chebyshev nodes t_j = cos(pi (j + 1/2) / n), extended precision."""
    n = len(y)
    th = [LD(j) + LD(0.5) for j in range(n)]
    pi = LD("3.14159265358979323846264338327950288")
    cheb = [LD(2 if k else 1) / LD(n) * sum(y[j] * np.cos(LD(k) * pi * th[j] / LD(n)) for j in range(n))
            for k in range(n)]
    out = [LD(0)] * n
    prev, cur = [LD(1)], [LD(0), LD(1)]
    polys = [prev, cur]
    for _ in range(2, n):
        nxt = [LD(0)] + [LD(2) * c for c in cur]
        for i, c in enumerate(prev):
            nxt[i] -= c
        prev, cur = cur, nxt
        polys.append(cur)
    for k in range(n):
        for i, c in enumerate(polys[k]):
            out[i] += cheb[k] * c
    return out


def table():
    n = DEG + 1
    pi = LD("3.14159265358979323846264338327950288")
    t = np.array([np.cos(pi * (LD(j) + LD(0.5)) / LD(n)) for j in range(n)])
    rows = []
    for e in range(E_MIN, E_MAX + 1):
        for q in range(PARTS):
            half = np.ldexp(LD(1), e - 3)                      # half the row's width
            mid = np.ldexp(LD(1) + (LD(q) + LD(0.5)) / LD(PARTS), e)
            c = _monomials(list(tail(mid + half * t)))
            rows.append([float(c[k] / half ** k) for k in range(n)])
    return np.array(rows)


def main():
    rows = table()
    lines = ["// Generated by gen_moro_tail_f64.py: %d rows (quarters of the binades" % len(rows),
             "// 2^%d .. 2^%d of the tail mass) of the coefficients of Moro's tail in the" % (E_MIN, E_MAX),
             "// distance to the row's midpoint."]
    for k, r in enumerate(rows):
        lines.append("    " + ", ".join("%.17e" % c for c in r) + ",  // row %d" % k)
    with open(os.path.join(HERE, "moro_tail_f64.inc"), "w") as f:
        f.write("\n".join(lines) + "\n")
    print("rows %d" % len(rows))


if __name__ == "__main__":
    main()
