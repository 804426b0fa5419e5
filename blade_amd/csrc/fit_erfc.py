"""Fit the FP32 erfc used by the nonbonded kernels.

erfc(x) = exp(-x^2) * erfcx(x), and erfcx is approximated on [0, XMAX] by a
polynomial in t = 1/(1 + P*x) (the substitution of Abramowitz & Stegun
7.1.26, refitted here to higher degree by a Chebyshev least-squares fit
against scipy's double-precision erfcx).  Writes erfc_coef.h beside this
script.  Run:  python blade_amd/csrc/fit_erfc.py
"""
import os
import numpy as np
from numpy.polynomial import chebyshev as C
from scipy.special import erfcx

XMAX, P, DEG = 4.0, 0.4, 9


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


def main():
    coef, err = fit()
    here = os.path.dirname(os.path.abspath(__file__))
    with open(os.path.join(here, "erfc_coef.h"), "w") as f:
        f.write("// Generated by fit_erfc.py: erfcx(x) ~ sum_k C[k] t^k, t = 1/(1+P x),\n")
        f.write(f"// x in [0,{XMAX}], max relative error of the fit {err:.2e} (exact arithmetic).\n")
        f.write("#pragma once\n")
        f.write(f"#define BM_ERFC_XMAX {XMAX:.1f}f\n#define BM_ERFC_P {P:.1f}f\n#define BM_ERFC_DEG {DEG}\n")
        f.write("static constexpr float bm_erfc_c[BM_ERFC_DEG + 1] = {\n")
        f.write(",\n".join(f"    {c:.9e}f" for c in coef))
        f.write("};\n")
    print("max rel err", err)


if __name__ == "__main__":
    main()
