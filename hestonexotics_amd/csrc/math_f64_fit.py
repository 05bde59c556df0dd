"""Coefficients of the FP64 kernel's exponential and logarithm (math_f64.hpp).

Interpolation at the Chebyshev nodes (in the node-transformed variable, within a factor 1 + 4/pi^2 ln n
of the best polynomial) of
    Q(r) = (e^r - 1 - r) / r^2            on |r| <= ln(2)/2 (1 + 2^-20), degree 9
    P(z) = (2 atanh(s) - 2 s) / (s z)     at z = s^2, s = (m - 1)/(m + 1), m in [sqrt(1/2), sqrt(2)], degree 6
in 80-bit arithmetic, from their Taylor series. Prints the coefficients, constant term first, and the
largest relative error of e^r and log(m) with the coefficients rounded to FP64.
"""
import numpy as np

L = np.longdouble


def interpolate(f, lo, hi, degree):
    k = np.arange(degree + 1, dtype=L)
    x = (lo + hi) / 2 + (hi - lo) / 2 * np.cos((2 * k + 1) * L(np.pi) / (2 * (degree + 1)))
    d = f(x)  # Newton's divided differences, expanded into powers
    for i in range(1, degree + 1):
        d[i:] = (d[i:] - d[i - 1:-1]) / (x[i:] - x[:-i])
    c = np.zeros(degree + 1, L)
    for i in range(degree, -1, -1):
        c[1:], c[0] = c[:-1] - x[i] * c[1:], d[i] - x[i] * c[0]
    return c


def series(coeffs, x):
    s = np.zeros_like(x)
    for c in reversed(coeffs):
        s = s * x + c
    return s


def exp_taylor():
    out, f = [], L(2)
    for i in range(26):
        out.append(1 / f)
        f *= L(i + 3)
    return out


def main():
    h = np.log(L(2)) / 2 * (1 + L(2) ** -20)
    q = interpolate(lambda r: series(exp_taylor(), r), -h, h, 9).astype(np.float64)
    r = np.linspace(-h, h, 20001, dtype=L)
    err = np.abs(r * r * (series(q.astype(L), r) - series(exp_taylor(), r)) / np.exp(r)).max()
    print("exp Q:", ", ".join(repr(float(v)) for v in q), " max relative error %.1e" % err)
    taylor = [L(2) / (2 * k + 3) for k in range(30)]
    smax = (np.sqrt(L(2)) - 1) / (np.sqrt(L(2)) + 1)
    p = interpolate(lambda z: series(taylor, z), L(0), smax * smax, 6).astype(np.float64)
    z = np.linspace(L(0), smax * smax, 20001, dtype=L)
    err = np.abs(z * (series(p.astype(L), z) - series(taylor, z)) / 2).max()
    print("log P:", ", ".join(repr(float(v)) for v in p), " max relative error %.1e" % err)


if __name__ == "__main__":
    main()
