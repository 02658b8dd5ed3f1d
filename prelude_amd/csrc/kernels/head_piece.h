// A head's row across neighbouring lanes of a wavefront, brought to unit RMS and turned in pairs by position.
#pragma once
#include "common.h"

namespace pa {

// The value of the lane `off` (a power of two below LANES) away within groups of LANES lanes, by the vector ALU's exchanges where it
// has them.  Four away in groups of sixteen or more: of a value that is the same eight lanes on, as within a sum.
template <int LANES>
__device__ __forceinline__ float from_lane_xor(float v, int off) {
  const unsigned u = __float_as_uint(v);
  const int lane = threadIdx.x % kWave;
  if (off == 32) {
    const auto both = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float(lane & 32 ? both[0] : both[1]);
  }
  if (off == 16) {
    const auto both = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __uint_as_float(lane & 16 ? both[0] : both[1]);
  }
  if (off == 8) return __int_as_float(__builtin_amdgcn_update_dpp(0, (int)u, 0x128, 0xf, 0xf, true));   // row_ror:8
  if (off == 4 && LANES >= 16) return __int_as_float(__builtin_amdgcn_update_dpp(0, (int)u, 0x124, 0xf, 0xf, true));   // row_ror:4
  if (off == 2) return __int_as_float(__builtin_amdgcn_update_dpp(0, (int)u, 0x4e, 0xf, 0xf, true));    // quad_perm [2, 3, 0, 1]
  if (off == 1) return __int_as_float(__builtin_amdgcn_update_dpp(0, (int)u, 0xb1, 0xf, 0xf, true));    // quad_perm [1, 0, 3, 2]
  return __shfl_xor(v, off, kWave);
}

// A lane's VEC neighbouring elements of a row of LPH lanes (c: which of them it is): times the row's 1 / sqrt(mean^2 + eps) and their
// weights w where `normed`, then turned with the elements half a row on by the angles whose cosines and sines cs and sn hold.
template <int LPH, int VEC>
__device__ __forceinline__ void norm_turn_piece(float (&x)[VEC], const float (&w)[VEC], const float (&cs)[VEC], const float (&sn)[VEC], bool normed,
                                                float eps, int c) {
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < VEC; ++e) ss += x[e] * x[e];
#pragma unroll
  for (int off = LPH / 2; off >= 1; off >>= 1) ss += from_lane_xor<LPH>(ss, off);
  const float inv = rsqrtf(ss / (float)(LPH * VEC) + eps);
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    if (normed) x[e] = x[e] * inv * w[e];
    const float partner = from_lane_xor<LPH>(x[e], LPH / 2);
    x[e] = c < LPH / 2 ? x[e] * cs[e] - partner * sn[e] : partner * sn[e] + x[e] * cs[e];
  }
}

}  // namespace pa
