// Errors of the FP64 pair energies (blade_amd/csrc/energy64.h) against long
// double, and those of the plain form: IEEE square root and division, the C
// library's erfc.  Run by test_erfc64.py.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../include/blade_mi355x.h"
#include "../blade_amd/csrc/energy64.h"

using namespace blade;
typedef long double real;

// the pair energy in the arithmetic of T
template <class T>
T plain(int elec, int vdw, T rc, T rs, T beta, T qq, T c12, T c6, T r) {
  const T rinv = 1 / r;
  T e;
  if (elec == BM_PME) {
    e = qq * std::erfc(beta * r) * rinv;
  } else if (elec == BM_FSWITCH) {
    const T roff2 = rc * rc, ron2 = rs * rs;
    const T ginv = 1 / ((roff2 - ron2) * (roff2 - ron2) * (roff2 - ron2));
    const T A = roff2 * roff2 * (roff2 - 3 * ron2) * ginv, B = 6 * roff2 * ron2 * ginv;
    const T C = -(ron2 + roff2) * ginv, D = 2 * ginv / 5;
    const T dvc = 8 * (ron2 * roff2 * (rc - rs) - (roff2 * roff2 * rc - ron2 * ron2 * rs) / 5) * ginv;
    const T r3 = r * r * r, r5 = r3 * r * r;
    e = r <= rs ? qq * (rinv + dvc)
                : qq * (A * (rinv - 1 / rc) + B * (rc - r) + C * (roff2 * rc - r3) + D * (roff2 * roff2 * rc - r5));
  } else {
    e = qq * (rinv - 2 / rc + r / (rc * rc));
  }
  const T rinv3 = rinv * rinv * rinv, rinv6 = rinv3 * rinv3;
  if (vdw == BM_VFSWITCH) {
    const T rc3 = rc * rc * rc, rs3 = rs * rs * rs;
    if (r < rs) {
      const T dv6 = 1 / (rc3 * rs3);
      e += c12 * (rinv6 * rinv6 - dv6 * dv6) - c6 * (rinv6 - dv6);
    } else {
      const T k6 = rc3 / (rc3 - rs3), k12 = rc3 * rc3 / (rc3 * rc3 - rs3 * rs3);
      const T a3 = rinv3 - 1 / rc3, a6 = rinv6 - 1 / (rc3 * rc3);
      e += c12 * k12 * a6 * a6 - c6 * k6 * a3 * a3;
    }
  } else if (vdw == BM_VSWITCH) {
    if (r < rs) {
      e += c12 * rinv6 * rinv6 - c6 * rinv6;
    } else {
      const T c2of = rc * rc, c2on = rs * rs, rul3 = (c2of - c2on) * (c2of - c2on) * (c2of - c2on);
      const T rijl = c2on - r * r, riju = c2of - r * r;
      e += riju * riju * (riju - 3 * rijl) / rul3 * (c12 * rinv6 - c6) * rinv6;
    }
  } else {
    const T r6 = r * r * r * r * r * r, rc6 = rc * rc * rc * rc * rc * rc;
    e += c12 * (rinv6 * rinv6 + 2 * r6 / (rc6 * rc6 * rc6) - 3 / (rc6 * rc6)) - c6 * (rinv6 + r6 / (rc6 * rc6) - 2 / rc6);
  }
  return e;
}

// a worse approximation of 1/sqrt(x) than the hardware's (2^-23): off by up to
// 2^-20
double seed(double x, double w) { return (1.0 + (2 * w - 1) * 0x1p-20) / std::sqrt(x); }

struct Err {
  double max = 0, sum2 = 0;
  long n = 0;
  void add(real v, real ref, real scale) {
    const double e = (double)std::fabs((v - ref) / scale);
    max = e > max ? e : max;
    sum2 += e * e;
    n++;
  }
  double rms() const { return std::sqrt(sum2 / n); }
};

template <int ELEC, int VDW>
void energies(double rc, double rs, double beta, std::mt19937_64 &rng, const std::vector<double> &table, int rows) {
  const EnConst c = make_energy_const(rc, rs, beta);
  std::uniform_real_distribution<double> u(0, 1);
  Err mine, ieee, qmine, qieee;
  for (int k = 0; k < 200000; k++) {
    // r^2 of a pair at uniform density from 1.5 A to the cutoff
    const double r0 = 1.5, w = u(rng), d2 = std::pow(r0 * r0 * r0 + w * (rc * rc * rc - r0 * r0 * r0), 2.0 / 3);
    if (!(d2 < rc * rc)) continue;
    const double q = 332.0716 * (u(rng) - 0.5), c12 = 6e5 * u(rng), c6 = 600 * u(rng);
    double r, ri;
    sqrt_rsqrt(d2, seed(d2, u(rng)), r, ri);
    const real R = std::sqrt((real)d2);
    // errors relative to the pair's 1/r, the size of what a sum cancels
    const real qref = plain<real>(ELEC, VDW, rc, rs, beta, q, 0, 0, R), ref = plain<real>(ELEC, VDW, rc, rs, beta, 0, c12, c6, R);
    const real qs = std::fabs(q) / R, ls = c12 / std::pow(R, (real)12) + c6 / std::pow(R, (real)6);
    const double rp = std::sqrt(d2);
    qmine.add(pair_energy_sum<ELEC, VDW>(c, table.data(), rows, q, 0, 0, r, ri), qref, qs);
    qieee.add(plain<double>(ELEC, VDW, rc, rs, beta, q, 0, 0, rp), qref, qs);
    mine.add(pair_energy_sum<ELEC, VDW>(c, table.data(), rows, 0, c12, c6, r, ri), ref, ls);
    ieee.add(plain<double>(ELEC, VDW, rc, rs, beta, 0, c12, c6, rp), ref, ls);
  }
  printf("energy %d %d %g %.4g %.4g %.4g %.4g %.4g %.4g %.4g %.4g\n", ELEC, VDW, rc, qmine.rms(), qieee.rms(), qmine.max,
         qieee.max, mine.rms(), ieee.rms(), mine.max, ieee.max);
}

int main() {
  std::mt19937_64 rng(11);
  std::uniform_real_distribution<double> u(0, 1);
  // erfc over the range of a system's arguments, and past it
  const int rows = erfc_rows(6.0);
  std::vector<double> t((size_t)kErfcTerms * kErfcMaxRows);
  erfc_table(t.data(), kErfcMaxRows);
  Err e, lib;
  for (int k = 0; k < 2000000; k++) {
    const double x = 6.0 * u(rng);
    e.add(erfc_d(t.data(), rows, x), std::erfc((real)x), std::erfc((real)x));
    lib.add(std::erfc(x), std::erfc((real)x), std::erfc((real)x));
  }
  printf("erfc %.4g %.4g %.4g %.4g\n", e.max, e.rms(), lib.max, lib.rms());
  double edge = 0, far = 0;
  for (int r = 0; r < rows; r++)
    for (int s = -1; s <= 1; s++) {
      const double x = s < 0 ? std::nextafter(r / 16.0, -1.0) : s > 0 ? std::nextafter(r / 16.0, 9.0) : r / 16.0;
      if (x >= 0) edge = std::fmax(edge, std::fabs(erfc_d(t.data(), rows, x) / (double)std::erfc((real)x) - 1));
    }
  for (double x = 6.0; x < 40; x += 0.0137) far = std::fmax(far, std::fabs(erfc_d(t.data(), kErfcMaxRows, x) - std::erfc(x)));
  printf("edges %.4g beyond %.4g\n", edge, far);
  // square root and its reciprocal
  Err s, si, sl, sil;
  for (int k = 0; k < 1000000; k++) {
    const double x = std::exp(12 * u(rng) - 6) ;
    double r, ri;
    sqrt_rsqrt(x, seed(x, u(rng)), r, ri);
    const real R = std::sqrt((real)x);
    s.add(r, R, R);
    si.add(ri, 1 / R, 1 / R);
    sl.add(std::sqrt(x), R, R);
    sil.add(1.0 / std::sqrt(x), 1 / R, 1 / R);
  }
  printf("sqrt %.4g %.4g rsqrt %.4g %.4g\n", s.max, sl.max, si.max, sil.max);
  const double sets[2][3] = {{12.0, 10.0, 0.32}, {9.0, 8.0, 0.34}};
  for (const double *p : sets) {
    const int n = erfc_rows(p[0] * p[2]);
    std::vector<double> tt((size_t)kErfcTerms * n);
    erfc_table(tt.data(), n);
    energies<BM_PME, BM_VFSWITCH>(p[0], p[1], p[2], rng, tt, n);
    energies<BM_FSWITCH, BM_VSWITCH>(p[0], p[1], p[2], rng, tt, n);
    energies<BM_FSHIFT, BM_VSHIFT>(p[0], p[1], p[2], rng, tt, n);
  }
}
