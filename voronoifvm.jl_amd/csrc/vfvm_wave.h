// Sums within a wave of 64 lanes by register moves.
#pragma once

#include <hip/hip_runtime.h>

namespace vfvm {

// v plus the v of the lane that the DPP control CTRL selects in its row of 16
template <int CTRL>
__device__ __forceinline__ double add_dpp(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return v + __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, 0xf, 0xf, true),
                              __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}
// sum over each row of 16 lanes, the same value in its lanes
__device__ __forceinline__ double row_sum(double v) {
  v = add_dpp<0xB1>(v);    // lane ^ 1
  v = add_dpp<0x4E>(v);    // lane ^ 2
  v = add_dpp<0x141>(v);   // mirrored within 8 lanes
  return add_dpp<0x140>(v);  // mirrored within 16 lanes
}
// sum over the wave (all 64 lanes active), the same value in every lane.  The steps within a row
// of 16 lanes are register moves (a butterfly through LDS takes about 100 cycles per step).
__device__ __forceinline__ double wave_sum(double v) {
  v = row_sum(v);
  return (lane_value(v, 0) + lane_value(v, 16)) + (lane_value(v, 32) + lane_value(v, 48));
}

}  // namespace vfvm
