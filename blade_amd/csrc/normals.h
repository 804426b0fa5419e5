// normals.h - the standard normals of a step (launched by update.hip alone
// and by bonded.hip beside the bonded terms).
#pragma once

#include "device.h"

namespace blade {

// standard normals of DOFs 2p and 2p+1 for (seed, step): the same rule as
// the oracle (one Philox block, Box-Muller cosine for the even DOF, sine for
// the odd one)
__device__ __forceinline__ double2 normal_pair(unsigned long long seed, unsigned long long step, unsigned long long p) {
#pragma clang fp contract(off)
  uint4 c = make_uint4((unsigned)p, (unsigned)step, (unsigned)(step >> 32), 0x4E524D4Cu);
  uint4 o = philox(c, make_uint2((unsigned)seed, (unsigned)(seed >> 32)));
  double u1 = ((double)((((unsigned long long)o.x) << 21) ^ (o.y >> 11)) + 0.5) * (1.0 / 9007199254740992.0);
  double u2 = ((double)((((unsigned long long)o.z) << 21) ^ (o.w >> 11)) + 0.5) * (1.0 / 9007199254740992.0);
  double rad = sqrt(-2.0 * log(u1));
  double sn, cs;
  sincospi(2.0 * u2, &sn, &cs);
  return make_double2(rad * cs, rad * sn);
}

__device__ __forceinline__ void upd_normals_body(const Dev &d, int bid) {
  const int p = bid * blockDim.x + threadIdx.x;
  const int N = 3 * d.n + d.nl;
  if (2 * p >= N) return;
  const double2 z = normal_pair(d.seed, (unsigned long long)(*d.step), (unsigned long long)p);
  d.xi[2 * p] = z.x;
  if (2 * p + 1 < N) d.xi[2 * p + 1] = z.y;
}

}  // namespace blade
