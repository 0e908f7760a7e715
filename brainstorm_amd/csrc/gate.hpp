// Shared by the kernels that select the largest scores of a row.
#pragma once

#include "common.hpp"

namespace brt {

// Scores as unsigned keys whose order is torch.topk's: larger key = ranked higher, NaN on top.
// 0 is below every real key and marks a column that is taken (or does not exist).
__device__ __forceinline__ uint32_t score_key(float f) {
  if (f != f) return 0xffffffffu;
  const uint32_t u = f == 0.0f ? 0u : __float_as_uint(f);  // -0 and +0 are one score
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);       // never 0: ~u of a number is >= 0x007fffff
}

template <int DT>
__device__ __forceinline__ float load_score(const void* p, size_t i) {
  if (DT == BRT_F32) return static_cast<const float*>(p)[i];
  return half_bits_to_float<DT>(static_cast<const uint16_t*>(p)[i]);
}

__device__ __forceinline__ float segment_sum(float v, int width) {
  return segment_all_reduce(v, width, [](float x, float y) { return x + y; });
}
__device__ __forceinline__ float segment_max(float v, int width) {
  return segment_all_reduce(v, width, [](float x, float y) { return fmaxf(x, y); });
}
__device__ __forceinline__ uint32_t segment_max(uint32_t v, int width) {
  return static_cast<uint32_t>(segment_all_reduce(static_cast<int>(v), width, [](int x, int y) {
    return static_cast<int>(max(static_cast<uint32_t>(x), static_cast<uint32_t>(y)));
  }));
}
// Maximum over the 64 lanes, in every lane as one scalar: lanes that a DPP step leaves out take 0, the least key.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
#define BRT_MAX_STEP(CTRL, ROWS)                                                                           \
  v = max(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, ROWS, 0xf, false)))
  BRT_MAX_STEP(0x111, 0xf);  // row_shr:1
  BRT_MAX_STEP(0x112, 0xf);  // row_shr:2
  BRT_MAX_STEP(0x114, 0xf);  // row_shr:4
  BRT_MAX_STEP(0x118, 0xf);  // row_shr:8
  BRT_MAX_STEP(0x142, 0xa);  // row_bcast:15 -> rows 1,3
  BRT_MAX_STEP(0x143, 0xc);  // row_bcast:31 -> rows 2,3
#undef BRT_MAX_STEP
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), kWave - 1));
}

}  // namespace brt
