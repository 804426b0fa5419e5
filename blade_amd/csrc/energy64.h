// energy64.h - FP64 pair energies of energy steps (the pair kernel; compiled
// for the CPU by tests/test_erfc64.py).
//
// The total potential is a small difference of large pair sums, so the sum
// is built from FP64 pair energies.  They are formed without branches and
// without a division per pair, each with no larger an error than the plain
// form with IEEE division, square root and the library's erfc:
//   * r and 1/r from the hardware's approximation of 1/sqrt by a Newton
//     step and one correction each, within 0.51 ulp;
//   * division by constants of the system as a product and one correction;
//   * erfc by rows of 1/16 in its argument, each a Taylor series about the
//     row's middle.  Its error is below 2.5e-16 of erfc(x) to x = 6 (the
//     library's 4.5e-16); past that erfc is below 2.2e-17.  The library walks
//     through three ranges, of which a wave takes all, and a polynomial of
//     one range needs exp(-x^2) beside it, whose argument's rounding alone
//     costs 3e-15 at x = 4.
#pragma once

#include <cmath>

#ifdef __HIP__
#define BM_HD __host__ __device__ __forceinline__
#else
#define BM_HD inline
#endif

namespace blade {

// ---- erfc ----------------------------------------------------------------
// Terms of a row: the remainder (2 x h)^14 / 14! of erfc(x), h = 1/32, is
// 1.2e-17 at x = 6.  An even number: a row is read 16 bytes at a time.
constexpr int kErfcTerms = 14;
constexpr int kErfcPerUnit = 16;
constexpr int kErfcMaxRows = 27 * kErfcPerUnit;   // erfc(27) underflows

// rows for arguments up to xmax
inline int erfc_rows(double xmax) {
  const double r = std::floor(xmax * kErfcPerUnit) + 1;
  return r < 1 ? 1 : r < kErfcMaxRows ? (int)r : kErfcMaxRows;
}

// The table: derivatives of erfc about each row's middle x0 by the recurrence
// of g = erfc' = -2/sqrt(pi) exp(-x^2), whose series about x0 follows from
// g' = -2 x g.
inline void erfc_table(double *t, int rows) {
  for (int r = 0; r < rows; r++, t += kErfcTerms) {
    const long double x0 = (r + 0.5L) / kErfcPerUnit;
    long double before = 0.0L, g = -1.128379167095512573896158903121545172L * std::exp(-x0 * x0);
    t[0] = (double)std::erfc(x0);
    for (int k = 1; k < kErfcTerms; k++) {
      t[k] = (double)(g / k);
      const long double next = -2.0L * (x0 * g + before) / k;
      before = g;
      g = next;
    }
  }
}

// erfc(x), x >= 0, from the table's rows
BM_HD double erfc_d(const double *table, int rows, double x) {
  const unsigned last = rows - 1, at = (unsigned)(int)(x * kErfcPerUnit), r = at < last ? at : last;
  const double *c = table + r * kErfcTerms;
  const double d = x - (r + 0.5) * (1.0 / kErfcPerUnit);
  double p = c[kErfcTerms - 1];
#pragma unroll
  for (int k = kErfcTerms - 2; k >= 0; k--) p = fma(p, d, c[k]);
  return p;
}

// ---- 1/sqrt, division ----------------------------------------------------
// sqrt(x) and its reciprocal from an approximation y of 1/sqrt(x), x > 0: one
// Newton step takes a relative error of 2^-20 (the hardware's is below 2^-23)
// to 2^-39, and the correction of each result squares that
// (1/sqrt from the rounded root, so that the two belong together: the switched
// and shifted energies cancel)
BM_HD void sqrt_rsqrt(double x, double y, double &s, double &si) {
  y = fma(y, fma(-0.5 * x * y, y, 0.5), y);
  const double s0 = x * y;
  s = fma(fma(-s0, s0, x), 0.5 * y, s0);
  si = fma(fma(-s, y, 1.0), y, y);
}
// x / y given yi = 1 / y
BM_HD double div_by(double x, double y, double yi) {
  const double q = x * yi;
  return fma(fma(-y, q, x), yi, q);
}

// ---- pair energy ---------------------------------------------------------
// constants of a system's methods, formed on the host: as kernel arguments
// they are scalar operands, computed in the kernel they took up to 30 vector
// registers
struct EnConst {
  double rc, rs, beta, rcinv;
  double rc3i, rc6i, k6, k12, dv6, dv12;         // VFSWITCH
  double A, B, C, D, dvc, roff2;                 // FSWITCH
  double rul3, rul3i;                            // VSWITCH
  double rc2, rc2i;                              // FSHIFT
  double rc12, rc12i, rc18, rc18i, sh12, sh6;    // VSHIFT
};

inline EnConst make_energy_const(double rc, double rs, double beta) {
  EnConst c;
  c.rc = rc;
  c.rs = rs;
  c.beta = beta;
  c.rcinv = 1.0 / rc;
  const double rc3 = rc * rc * rc, rs3 = rs * rs * rs;
  c.rc3i = 1 / rc3;
  c.rc6i = 1 / (rc3 * rc3);
  c.k6 = rc3 / (rc3 - rs3);
  c.k12 = rc3 * rc3 / (rc3 * rc3 - rs3 * rs3);
  c.dv6 = 1 / (rc3 * rs3);
  c.dv12 = c.dv6 * c.dv6;
  const double roff2 = rc * rc, ron2 = rs * rs;
  const double rul3 = (roff2 - ron2) * (roff2 - ron2) * (roff2 - ron2), g = 1 / rul3;
  c.roff2 = roff2;
  c.rul3 = rul3;
  c.rul3i = g;
  c.A = roff2 * roff2 * (roff2 - 3 * ron2) * g;
  c.B = 6 * roff2 * ron2 * g;
  c.C = -(ron2 + roff2) * g;
  c.D = 2 * g / 5;
  c.dvc = 8 * (ron2 * roff2 * (rc - rs) - (roff2 * roff2 * rc - ron2 * ron2 * rs) / 5) * g;
  c.rc2 = roff2;
  c.rc2i = 1 / roff2;
  const double rc6 = rc * rc * rc * rc * rc * rc;
  c.rc12 = rc6 * rc6;
  c.rc12i = 1 / c.rc12;
  c.rc18 = c.rc12 * rc6;
  c.rc18i = 1 / c.rc18;
  c.sh12 = 3 / c.rc12;
  c.sh6 = 2 / rc6;
  return c;
}

// energy of a pair at effective distance r (rinv = 1/r); erfct: the erfc rows
// (PME)
template <int ELEC, int VDW>
BM_HD double pair_energy_sum(const EnConst &c, const double *erfct, int erfcrows, double qq, double c12, double c6,
                             double r, double rinv) {
  const double r2 = r * r;
  double e;
  if (ELEC == BM_PME) {
    e = qq * erfc_d(erfct, erfcrows, c.beta * r) * rinv;
  } else if (ELEC == BM_FSWITCH) {
    const double r3 = r2 * r, r5 = r3 * r2;
    const double in = rinv + c.dvc;
    const double out = c.A * (rinv - c.rcinv) + c.B * (c.rc - r) + c.C * (c.roff2 * c.rc - r3) +
                       c.D * (c.roff2 * c.roff2 * c.rc - r5);
    e = qq * (r <= c.rs ? in : out);
  } else {
    e = qq * (rinv - 2 * c.rcinv + div_by(r, c.rc2, c.rc2i));
  }
  const double rinv3 = rinv * rinv * rinv, rinv6 = rinv3 * rinv3;
  if (VDW == BM_VFSWITCH) {
    const bool in = r < c.rs;
    const double a3 = rinv3 - c.rc3i, a6 = rinv6 - c.rc6i;
    const double rep = in ? rinv6 * rinv6 - c.dv12 : c.k12 * a6 * a6;
    const double att = in ? rinv6 - c.dv6 : c.k6 * a3 * a3;
    e += c12 * rep - c6 * att;
  } else if (VDW == BM_VSWITCH) {
    const double rijl = c.rs * c.rs - r2, riju = c.roff2 - r2;
    const double sw = r < c.rs ? 1.0 : div_by(riju * riju * (riju - 3 * rijl), c.rul3, c.rul3i);
    e += sw * (c12 * rinv6 - c6) * rinv6;
  } else {
    const double r6 = r2 * r2 * r2;
    e += c12 * (rinv6 * rinv6 + div_by(2 * r6, c.rc18, c.rc18i) - c.sh12) -
         c6 * (rinv6 + div_by(r6, c.rc12, c.rc12i) - c.sh6);
  }
  return e;
}

}  // namespace blade
