// spread.h - the PME charge spread of one brick (launched by pme.hip alone
// and by bonded.hip beside the bonded terms).
#pragma once

#include "device.h"

namespace blade {

// B-spline weights of order N: w[t] = M_N(frac+N-1-t) for grid point u0+t,
// dw[t] its derivative (M_{N-1}(x) - M_{N-1}(x-1)).
template <int N, class T>
__device__ __forceinline__ void bspline_w(T frac, T *w, T *dw) {
  T A[N];
  A[0] = T(1);
#pragma unroll
  for (int k = 1; k < N; k++) A[k] = T(0);
#pragma unroll
  for (int m = 2; m <= N; m++) {
    if (m == N) {
#pragma unroll
      for (int k = 0; k < N; k++) dw[N - 1 - k] = A[k] - (k ? A[k - 1] : T(0));
    }
    const T inv = T(1) / T(m - 1);
#pragma unroll
    for (int k = m - 1; k >= 0; k--) {
      T a = (frac + T(k)) * A[k];
      T b = k ? (T(m) - frac - T(k)) * A[k - 1] : T(0);
      A[k] = (a + b) * inv;
    }
  }
#pragma unroll
  for (int k = 0; k < N; k++) w[N - 1 - k] = A[k];
}

// grid index and fraction from the 32-bit fractional coordinate
template <class T>
__device__ __forceinline__ void grid_coord(unsigned u, int K, int &u0, T &frac) {
  unsigned long long p = (unsigned long long)u * (unsigned)K;
  u0 = (int)(p >> 32);
  frac = (T)((unsigned)(p & 0xFFFFFFFFull)) * (T(1) / T(4294967296.0));
}

// atoms per round of the spread: one wave per axis computes their weights
constexpr int kSpreadStage = 64;

// v * 2^32 rounded to the nearest integer (ties to even), as
// __double2ll_rn(v * 2^32) gives, for |v * 2^32| < 2^51: the sum with
// 1.5 * 2^52 is rounded to an integer by the addition itself, and its low
// mantissa bits are that integer plus a constant.
__device__ __forceinline__ long long fix_d_small(double v) {
  const double magic = 6755399441055744.0;   // 1.5 * 2^52
  return __double_as_longlong(fma(v, 4294967296.0, magic)) - __double_as_longlong(magic);
}

// One workgroup (256 threads) per brick, over the atoms binned in it and no
// others: their whole stencils go into the brick padded by order-1 points
// per axis, summed in LDS as 64-bit fixed point, and the padded brick is
// stored with plain stores (no global atomics, no clearing pass).  The
// FFT's first pass adds the bricks that overlap at a point (pme_charge), an
// exact integer sum.  Each round takes up to kSpreadStage atoms: three
// waves compute the FP64 B-spline weights, one axis each, then every thread
// takes (atom, x, y) stencil rows.  Against bricks that read every atom
// whose stencil could reach them (each atom's 176-byte spline record from
// HBM by up to eight bricks, the stencils clipped and their rows listed in
// LDS), each atom is read once, in 24 bytes, and each row visited once.
template <int N>
__device__ __forceinline__ void pme_spread_body(const Dev &d, int bid) {
  extern __shared__ long long acc[];
  __shared__ double s_w[3][N][kSpreadStage];   // the x weights times lambda*q
  __shared__ short s_off[3][kSpreadStage];     // first stencil point within the brick
  const int py = d.ppad[1], pz = d.ppad[2];
  for (int p = threadIdx.x; p < d.pvol; p += blockDim.x) acc[p] = 0;
  const int na = min(d.pbcount[bid], d.pcap);
  const int ax = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), al = threadIdx.x & 63;
  // (selects of values, not d.K[ax] nor what the compiler makes of selects of
  // its elements: a run-time index moves the whole Dev to scratch memory)
  const int K0 = __builtin_amdgcn_readfirstlane(d.K[0]), K1 = __builtin_amdgcn_readfirstlane(d.K[1]);
  const int K2 = __builtin_amdgcn_readfirstlane(d.K[2]), nb0 = __builtin_amdgcn_readfirstlane(d.pnb[0]);
  const int nb1 = __builtin_amdgcn_readfirstlane(d.pnb[1]), nb2 = __builtin_amdgcn_readfirstlane(d.pnb[2]);
  const int Kax = ax == 0 ? K0 : ax == 1 ? K1 : K2;
  const int nbax = ax == 0 ? nb0 : ax == 1 ? nb1 : nb2;
  const int bax = ax == 2 ? bid % nb2 : ax == 1 ? bid / nb2 % nb1 : bid / nb2 / nb1;
  const int lo = (bax * Kax) / nbax;
  for (int base = 0; base < na; base += kSpreadStage) {
    const int m = min(kSpreadStage, na - base);
    if (ax < 3 && al < m) {
      const long long e = (long long)bid * d.pcap + base + al;
      const uint4 u = d.pbpos[e];
      int u0;
      double fr, w[N], dw[N];
      grid_coord(ax == 0 ? u.x : ax == 1 ? u.y : u.z, Kax, u0, fr);
      bspline_w<N>(fr, w, dw);
      const double f = ax == 0 ? d.pblq[e] : 1.0;
#pragma unroll
      for (int t = 0; t < N; t++) s_w[ax][t][al] = w[t] * f;
      s_off[ax][al] = (short)(u0 - lo);
    }
    __syncthreads();
    for (int it = threadIdx.x; it < m * N * N; it += blockDim.x) {
      const int a = it / (N * N), xy = it % (N * N), x = xy / N, y = xy % N;
      const double wxy = s_w[0][x][a] * s_w[1][y][a];
      long long *row = acc + ((s_off[0][a] + x) * py + s_off[1][a] + y) * pz + s_off[2][a];
#pragma unroll
      for (int z = 0; z < N; z++)
        // |lambda q w w w| <= |q| < 2^19: within fix_d_small's range
        atomicAdd(reinterpret_cast<unsigned long long *>(row + z),
                  (unsigned long long)fix_d_small(wxy * s_w[2][z][a]));
    }
    __syncthreads();
  }
  if (na == 0) __syncthreads();
  long long *out = d.pgrid + (long long)bid * d.pvol;
  for (int p = threadIdx.x; p < d.pvol; p += blockDim.x) out[p] = acc[p];
}

}  // namespace blade
