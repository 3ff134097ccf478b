// Sums over a 64-lane wavefront.
#pragma once
#include "common.hpp"

namespace dmrg {

// Sum over the wave, in every lane, by DPP adds (row shifts, then row
// broadcasts into the last lane): no trip through LDS.
template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  int p[2], q[2];
  __builtin_memcpy(p, &v, 8);
  q[0] = __builtin_amdgcn_update_dpp(0, p[0], CTRL, ROWS, 0xf, true);
  q[1] = __builtin_amdgcn_update_dpp(0, p[1], CTRL, ROWS, 0xf, true);
  double u;
  __builtin_memcpy(&u, q, 8);
  return v + u;
}
__device__ inline double read_lane(double v, int l) {
  int p[2];
  __builtin_memcpy(p, &v, 8);
  p[0] = __builtin_amdgcn_readlane(p[0], l);
  p[1] = __builtin_amdgcn_readlane(p[1], l);
  __builtin_memcpy(&v, p, 8);
  return v;
}
__device__ inline double wave_sum_all(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return read_lane(v, 63);
}
__device__ inline cdouble wave_sum_all(cdouble v) {
  return cdouble(wave_sum_all(v.x), wave_sum_all(v.y));
}
__device__ inline cdouble read_lane(cdouble v, int l) {
  return cdouble(read_lane(v.x, l), read_lane(v.y, l));
}

}  // namespace dmrg
