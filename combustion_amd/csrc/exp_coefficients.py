"""Constants of the polynomials that the FP64 kernels inline, in 60-digit arithmetic.

exp64 of the straight-line kernels (hip_emit.cpp): e^x = 2^n e^r with n = rint(x / ln 2) and r = x - n ln 2 (Cody and
Waite's two-constant reduction: n ln2_hi is exact for |n| < 2^21 because ln2_hi keeps only the leading 32 bits of ln 2),
and e^r for |r| <= ln(2)/2 by a degree-10 polynomial: the Chebyshev interpolant of e^r on that interval (within a small
factor of the minimax error; its constant coefficient rounds to 1 in FP64, so e^0 = 1 exactly). Its worst relative error
is 4.3e-16 in FP64 Horner form (about two ulps; degree 11: 1.6e-16, one FMA more; degree 9: 1.9e-14 and a constant
coefficient off 1).

pow2_rows of kernels/rates_split.hip: the same of 2^r for |r| <= 1/2.

log_rows of kernels/rates_split.hip and log64 of the transport kernels (transport_split.hip, transport_pairs.hip):
log2 m = s P(s^2) with s = (m - 1)/(m + 1), for m in [sqrt(1/2), sqrt(2)): P(z) = 2 atanh(sqrt z) / (sqrt z ln 2) by its
Chebyshev interpolant of degree 7 on the interval of z (relative error 1.4e-17).

Prints the constants as C hex literals and each polynomial's worst relative error over a dense grid, evaluated in FP64
Horner form for the exponentials and exactly for the logarithm.

Run: python exp_coefficients.py
"""
import mpmath as mp

mp.mp.dps = 60
DEGREE = 10


def hexd(x):
    return float(x).hex()


def interpolant(f, low, high, degree):
    """Monomial coefficients of the Chebyshev interpolant of f on [low, high]."""
    n = degree + 1
    nodes = [(low + high) / 2 + (high - low) / 2 * mp.cos(mp.pi * (2 * k + 1) / (2 * n)) for k in range(n)]
    return list(mp.lu_solve(mp.matrix([[x ** j for j in range(n)] for x in nodes]), mp.matrix([f(x) for x in nodes])))


def exponential(base, a):
    c = [float(x) for x in interpolant(lambda x: base ** x, -a, a, DEGREE)]
    worst = 0
    for i in range(20001):
        r = float(-a + 2 * a * i / 20000)
        p = c[-1]
        for j in range(DEGREE - 1, -1, -1):
            p = p * r + c[j]  # FP64 Horner (rounding per step, as the kernel's FMAs at worst)
        worst = max(worst, abs((mp.mpf(p) - base ** mp.mpf(r)) / base ** mp.mpf(r)))
    return c, worst


def logarithm():
    P = lambda z: 2 / mp.log(2) * (mp.atanh(mp.sqrt(z)) / mp.sqrt(z) if z else 1)
    high = ((mp.sqrt(2) - 1) / (mp.sqrt(2) + 1)) ** 2
    c = [float(x) for x in interpolant(P, mp.mpf(0), high, 7)]
    exact = lambda z: sum(mp.mpf(x) * z ** j for j, x in enumerate(c))
    return c, max(abs(exact(high * i / 2000) / P(high * i / 2000) - 1) for i in range(2001))


def main():
    ln2 = mp.log(2)
    hi = mp.mpf(float(ln2))
    hi = mp.floor(hi * 2 ** 32) / 2 ** 32  # leading 32 bits
    print("ln2_hi", hexd(hi), "ln2_lo", hexd(ln2 - hi), "log2e", hexd(1 / ln2))
    for name, (c, worst) in (("e^r on [-ln2/2, ln2/2]", exponential(mp.e, ln2 / 2)), ("2^r on [-1/2, 1/2]", exponential(mp.mpf(2), mp.mpf(1) / 2)),
                             ("log2(m)/s in s^2", logarithm())):
        print(name, "c0..:", ", ".join(hexd(x) for x in c), "worst relative error %.3g" % worst)


if __name__ == "__main__":
    main()
