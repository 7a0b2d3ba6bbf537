// Wavefront reductions and broadcasts of doubles.
#pragma once
#include "gi_common.h"

namespace gi {

// maximum over the wavefront (NaN ignored), the same value in every lane: the
// rows of sixteen by row shifts, then the row totals by row broadcasts, lane 63
// last
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_max(double x) {
  const unsigned long long v = __builtin_bit_cast(unsigned long long, x);
  const int lo = __builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(v >> 32), (int)(v >> 32), CTRL, ROWS, 0xf, false);
  return fmax(x, __builtin_bit_cast(double, (unsigned long long)(unsigned)lo | ((unsigned long long)(unsigned)hi << 32)));
}
__device__ __forceinline__ double wave_max(double x) {
  x = dpp_max<0x111, 0xf>(x);   // row_shr:1, 2, 4, 8
  x = dpp_max<0x112, 0xf>(x);
  x = dpp_max<0x114, 0xf>(x);
  x = dpp_max<0x118, 0xf>(x);
  x = dpp_max<0x142, 0xa>(x);   // row_bcast:15 into rows 1 and 3
  x = dpp_max<0x143, 0xc>(x);   // row_bcast:31 into rows 2 and 3
  const unsigned long long v = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_readlane((int)v, 63), hi = __builtin_amdgcn_readlane((int)(v >> 32), 63);
  return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}
__device__ __forceinline__ double read_lane(double x, int lane) {   // lane uniform
  const unsigned long long v = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_readlane((int)v, lane), hi = __builtin_amdgcn_readlane((int)(v >> 32), lane);
  return __builtin_bit_cast(double, (unsigned long long)lo | ((unsigned long long)hi << 32));
}

}  // namespace gi
