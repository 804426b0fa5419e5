"""The FP64 erfc of the pair energies (coefficients of erfc_coef.h, exp by
range reduction and its Taylor series), restated here operation by operation
in double precision, against scipy."""
import os
import re

import numpy as np
from scipy.special import erfcx

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(HERE, "..", "blade_amd", "csrc", "erfc_coef.h")


def test_erfc64_fit():
    src = open(HEADER).read()
    a = float(re.search(r"BM_ERFCD_A\s+([\d.]+)", src).group(1))
    xmax = float(re.search(r"BM_ERFCD_XMAX\s+([\d.]+)", src).group(1))
    coef = [float(v) for v in re.findall(r"-?\d\.\d+e[+-]\d+(?=[, \n])", src.split("BM_ERFCD_COEF")[1])]
    assert len(coef) == int(re.search(r"BM_ERFCD_DEG\s+(\d+)", src).group(1)) + 1
    x = np.linspace(0.0, xmax, 60001)
    y = 1.0 - 2.0 * a / (x + a)
    p = np.zeros_like(x)
    for c in reversed(coef):
        p = p * y + c
    # the polynomial's own error is 7e-15; Horner's roundings at |y| <= 1
    # over coefficients summing below 1 add a few 1e-16 of erfcx(6) = 0.093
    assert np.max(np.abs(p / erfcx(x) - 1.0)) < 4e-14
    # exp(-x^2): |r| <= ln2/2, the series' next term is r^13/13! = 2e-16
    v = -x * x
    n = np.rint(v * 1.4426950408889634)
    hi = float(np.float32(0.693147182464599609375))
    r = (v - n * hi) + n * 1.904654299957767878541823e-09   # n*hi is exact: 24 + 6 bits
    e = np.zeros_like(x)
    f = 1.0
    term = [1.0]
    for k in range(1, 13):
        f *= k
        term.append(1.0 / f)
    for c in reversed(term):
        e = e * r + c
    assert np.max(np.abs(np.ldexp(e, n.astype(int)) / np.exp(v) - 1.0)) < 2e-15
