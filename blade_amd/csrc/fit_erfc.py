"""Fit the FP32 and FP64 erfc used by the nonbonded kernels.

erfc(x) = exp(-x^2) * erfcx(x), and erfcx is approximated on [0, XMAX] by a
polynomial in t = 1/(1 + P*x) (the substitution of Abramowitz & Stegun
7.1.26, refitted here to higher degree by a Chebyshev least-squares fit
against scipy's double-precision erfcx).  The FP64 form (energies) is a
polynomial in y = (x - A)/(x + A) on [0, XMAXD], the variable of Schonfelder's
Chebyshev expansions (Math. Comp. 32, 1978), fitted the same way: |y| < 1 and
its coefficients fall off, so Horner's rule keeps full precision.  Writes
erfc_coef.h beside this script.  Run:  python blade_amd/csrc/fit_erfc.py
"""
import os
import numpy as np
from numpy.polynomial import chebyshev as C
from scipy.special import erfcx

XMAX, P, DEG = 4.0, 0.4, 9
XMAXD, A, DEGD = 6.0, 3.0, 16


def fit():
    xs = np.linspace(0.0, XMAX, 40001)
    t = 1.0 / (1.0 + P * xs)
    tmin = 1.0 / (1.0 + P * XMAX)
    u = (t - tmin) / (1.0 - tmin) * 2.0 - 1.0
    cheb = C.chebfit(u, erfcx(xs), DEG)
    # back to a monomial polynomial in t
    inner = np.polynomial.Polynomial([-1.0 - 2.0 * tmin / (1.0 - tmin), 2.0 / (1.0 - tmin)])
    poly = np.polynomial.Polynomial(C.cheb2poly(cheb))(inner)
    return poly.coef, float(np.max(np.abs(poly(t) / erfcx(xs) - 1.0)))


def fit64():
    ymax = (XMAXD - A) / (XMAXD + A)
    th = np.cos(np.pi * (np.arange(4000) + 0.5) / 4000)
    y = 0.5 * (ymax + 1.0) * th + 0.5 * (ymax - 1.0)
    f = erfcx(A * (1.0 + y) / (1.0 - y))
    cheb = C.chebfit(th, f, DEGD, w=1.0 / f)
    inner = np.polynomial.Polynomial([(1.0 - ymax) / (1.0 + ymax), 2.0 / (1.0 + ymax)])
    poly = np.polynomial.Polynomial(C.cheb2poly(cheb))(inner)
    xs = np.linspace(0.0, XMAXD, 40001)
    return poly.coef, float(np.max(np.abs(poly((xs - A) / (xs + A)) / erfcx(xs) - 1.0)))


def main():
    coef, err = fit()
    coefd, errd = fit64()
    here = os.path.dirname(os.path.abspath(__file__))
    with open(os.path.join(here, "erfc_coef.h"), "w") as f:
        f.write("// Generated by fit_erfc.py: erfcx(x) ~ sum_k C[k] t^k, t = 1/(1+P x),\n")
        f.write(f"// x in [0,{XMAX}], max relative error of the fit {err:.2e} (exact arithmetic).\n")
        f.write("#pragma once\n")
        f.write(f"#define BM_ERFC_XMAX {XMAX:.1f}f\n#define BM_ERFC_P {P:.1f}f\n#define BM_ERFC_DEG {DEG}\n")
        f.write("static constexpr float bm_erfc_c[BM_ERFC_DEG + 1] = {\n")
        f.write(",\n".join(f"    {c:.9e}f" for c in coef))
        f.write("};\n")
        f.write("// FP64: erfcx(x) ~ sum_k C[k] y^k, y = (x-A)/(x+A), x in [0,%.1f], max relative\n" % XMAXD)
        f.write(f"// error {errd:.1e} (FP64 arithmetic).\n")
        f.write(f"#define BM_ERFCD_XMAX {XMAXD:.1f}\n#define BM_ERFCD_A {A:.1f}\n#define BM_ERFCD_DEG {DEGD}\n")
        f.write("#define BM_ERFCD_COEF \\\n")
        f.write(", \\\n".join(f"    {c:.17e}" for c in coefd) + "\n")
    print("max rel err", err, errd)


if __name__ == "__main__":
    main()
