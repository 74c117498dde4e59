#!/usr/bin/env python3
"""Generate the cardinal B-spline weight polynomials used by charge assignment.

The charge-assignment function of order p (cao = p) is the centred cardinal
B-spline B_p of support [-p/2, p/2], obtained by p-1 convolutions of the unit
box.  For a particle whose offset from its reference mesh point is
x in [-1/2, 1/2], the weight of stencil point j (j = 0 .. p-1) is

    W_j(x) = B_p(x - j + (p-1)/2)

which is one polynomial piece of B_p.  Every piece has rational coefficients
with the common denominator D_p = 2^(p-1) (p-1)!, so it is stored as integer
numerators and evaluated as Horner(numerators, x) / D_p.  The derivative
weights W'_j(x) are the derivatives of the same pieces.

The reference tabulates the same functions (window-functions.c:108-184 for
W, :46-106 for W') and evaluates them at the quantised offsets of
interpol.c:53-60; this script derives them from the definition instead of
copying them.

Usage:  python3 gen_bspline.py > bspline_coeffs.hpp
"""
import math
import sys
from fractions import Fraction as Fr

MAX_ORDER = 7


def _ev(c, t):
    s = Fr(0)
    for ck in reversed(c):
        s = s * t + ck
    return s


def _shift(c, a):
    """Coefficients of c(t + a) as a polynomial in t."""
    out = [Fr(0)] * len(c)
    for k, ck in enumerate(c):
        for j in range(k + 1):
            out[j] += ck * math.comb(k, j) * a ** (k - j)
    return out


def bspline_pieces(p):
    """Pieces of B_p: pieces[k] is the polynomial (in t) on [-p/2+k, -p/2+k+1]."""
    pieces = [[Fr(1)]]
    lo = Fr(-1, 2)
    for _ in range(2, p + 1):
        n = len(pieces)
        anti = [[Fr(0)] + [c[k] / (k + 1) for k in range(len(c))] for c in pieces]
        consts, acc = [], Fr(0)
        for k in range(n):
            a = lo + k
            consts.append(acc - _ev(anti[k], a))
            acc += _ev(anti[k], a + 1) - _ev(anti[k], a)
        total = acc

        def phi(k, shift):
            if k < 0:
                return [Fr(0)]
            if k >= n:
                return [total]
            c = list(anti[k])
            c[0] += consts[k]
            return _shift(c, shift)

        new = []
        for m in range(n + 1):
            up, dn = phi(m, Fr(1, 2)), phi(m - 1, Fr(-1, 2))
            width = max(len(up), len(dn))
            up += [Fr(0)] * (width - len(up))
            dn += [Fr(0)] * (width - len(dn))
            new.append([u - d for u, d in zip(up, dn)])
        pieces, lo = new, lo - Fr(1, 2)
    return pieces


def weight_polys(p):
    """W_j(x) for j = 0..p-1 as lists of Fraction coefficients (ascending powers)."""
    pieces = bspline_pieces(p)
    polys = []
    for j in range(p):
        c = _shift(pieces[p - 1 - j], Fr(p - 1, 2) - j)
        c += [Fr(0)] * (p - len(c))
        polys.append(c[:p])
    return polys


def denominator(p):
    return 2 ** (p - 1) * math.factorial(p - 1)


def integer_tables(p):
    D = denominator(p)
    w, dw, d2w = [], [], []
    for c in weight_polys(p):
        num = [ck * D for ck in c]
        assert all(v.denominator == 1 for v in num)
        w.append([int(v) for v in num])
        d = [num[k] * k for k in range(1, p)] + [Fr(0)]
        dw.append([int(v) for v in d])
        d2 = [num[k] * k * (k - 1) for k in range(2, p)] + [Fr(0), Fr(0)]
        d2w.append([int(v) for v in d2])
    return D, w, dw, d2w


def _horner(coeffs):
    """Horner expression in x for integer coefficients (ascending powers)
    times u."""
    expr = "T(u * %d)" % coeffs[-1]
    for c in reversed(coeffs[:-1]):
        expr = "T(u * %d) + x * (%s)" % (c, expr)
    return expr


def main(out=sys.stdout):
    out.write("/* Generated by gen_bspline.py -- do not edit.\n"
              " * Cardinal B-spline charge-assignment weights of order P (cao):\n"
              " *   w[j]  = W_j(x)  = B_P(x - j + (P-1)/2),  x in [-1/2, 1/2]\n"
              " *   dw[j] = W'_j(x),  d2w[j] = W''_j(x)\n"
              " * each times u D_P, D_P = 2^(P-1) (P-1)!: integer-coefficient Horner\n"
              " * polynomials.  u is 1 in FP64 and in FP32 one over the largest power of two\n"
              " * up to D_P, so that the coefficients are exact in both and FP32 sums of mesh\n"
              " * values times weights stay in the range of the mesh values (the scaled\n"
              " * coefficients in FP64 too: k_collect 1045 -> 1253 us at order 7, fewer of\n"
              " * them are inline constants).  The caller multiplies the product of three by\n"
              " * norm^3 (stencil_norm) in FP64, once per particle: a rounded FP32 1/D_P in\n"
              " * every weight scales all of them by the same error. */\n")
    out.write("#pragma once\n\nnamespace p3m {\n\n")
    out.write("template <int P, typename T> struct Bspline;\n\n")
    for p in range(1, MAX_ORDER + 1):
        D, w, dw, d2w = integer_tables(p)
        S = 2 ** (D.bit_length() - 1)
        out.write("template <typename T> struct Bspline<%d, T> {\n" % p)
        out.write("  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / %d;\n" % S)
        out.write("  static constexpr double norm = 1.0 / (u * %d);\n" % D)
        out.write("  __host__ __device__ static inline void w(T x, T *o) {\n")
        if p == 1:
            out.write("    (void)x;\n")
        for j in range(p):
            out.write("    o[%d] = (%s);\n" % (j, _horner(w[j])))
        out.write("  }\n")
        out.write("  __host__ __device__ static inline void dw(T x, T *o) {\n")
        if p <= 2:
            out.write("    (void)x;\n")
        for j in range(p):
            if p == 1:
                out.write("    o[%d] = T(0.0);\n" % j)
            else:
                out.write("    o[%d] = (%s);\n" % (j, _horner(dw[j][:p - 1])))
        out.write("  }\n")
        out.write("  __host__ __device__ static inline void d2w(T x, T *o) {\n")
        if p <= 3:
            out.write("    (void)x;\n")
        for j in range(p):
            if p <= 2:
                out.write("    o[%d] = T(0.0);\n" % j)
            else:
                out.write("    o[%d] = (%s);\n" % (j, _horner(d2w[j][:p - 2])))
        out.write("  }\n};\n\n")
    out.write("// the norm of a product of three weights\n"
              "template <int P, typename T> constexpr double stencil_norm =\n"
              "    Bspline<P, T>::norm * Bspline<P, T>::norm * Bspline<P, T>::norm;\n\n")
    out.write("}  // namespace p3m\n")


if __name__ == "__main__":
    main()
