// Sums and exchanges of doubles between the lanes of a wave by DPP and lane-swap instructions
// (gfx950): no LDS traffic, and every lane ends with the same bits.
#pragma once

#include <hip/hip_runtime.h>

namespace dftbhip {

__device__ __forceinline__ double hilo(unsigned lo, unsigned hi) {
  return __hiloint2double((int)hi, (int)lo);
}

// sum over the 64 lanes, the same bits in every lane (each step adds a pair both ways round)
template <int Ctrl>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), Ctrl, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), Ctrl, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
constexpr int kRor8 = 0x128, kRor4 = 0x124, kRor2 = 0x122, kRor1 = 0x121;
constexpr int kHalfMirror = 0x141, kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;

// rows (16 lanes) r of a and b: even rows a_r + a_(r+1), odd rows b_(r-1) + b_r
__device__ __forceinline__ double swap16_add(double a, double b) {
  const auto l = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                  (unsigned)__double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                  (unsigned)__double2hiint(b), false, false);
  return hilo(l[0], h[0]) + hilo(l[1], h[1]);
}
// lanes < 32: a_l + a_(l+32); lanes >= 32: b_(l-32) + b_l
__device__ __forceinline__ double swap32_add(double a, double b) {
  const auto l = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                  (unsigned)__double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                  (unsigned)__double2hiint(b), false, false);
  return hilo(l[0], h[0]) + hilo(l[1], h[1]);
}
__device__ __forceinline__ double wave_total(double v) {
  v += dpp<kRor8>(v);
  v += dpp<kRor4>(v);
  v += dpp<kRor2>(v);
  v += dpp<kRor1>(v);
  v = swap16_add(v, v);
  return swap32_add(v, v);
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// sum over the eight lanes 8 r .. 8 r + 7
__device__ __forceinline__ double octet_sum(double v) {
  v += dpp<kHalfMirror>(v);
  v += dpp<kQuadXor1>(v);
  return v + dpp<kQuadXor2>(v);
}

}  // namespace dftbhip
