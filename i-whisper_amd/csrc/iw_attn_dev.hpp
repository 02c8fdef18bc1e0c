// Device helpers shared by the prefill attention kernels: the score
// requantization and the index of the shift-exponential table.
#pragma once

#include "iw_common.hpp"
#include "iw_kernels.hpp"

namespace iw {

__device__ __forceinline__ int32_t qk_requant16(int32_t acc, uint32_t m, uint32_t s) {
  // (int32)(acc * m) modulo 2^32, Rshift, saturate to int16
  return clampi(rshift((int32_t)((uint32_t)acc * m), s), -32768, 32767);
}

// Median of three signed ints: clamp of x to [lo, hi] for lo <= hi, in one
// instruction where the bounds are not compile-time constants.
__device__ __forceinline__ int32_t med3i(int32_t x, int32_t lo, int32_t hi) {
  int32_t r;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
  return r;
}

// Table index of a raw score for a row maximum: min((rowmax + 1 - h16) mod
// 2^16, L) with L the last table entry.
//
// Where every key of a chunk counts in the row maximum and that is below
// 32767, rowmax + 1 - h16 lies in [1, 65535] and the index is
//   min(R - clamp16(h), L) = med3(R - h, min(R - 32767, L), min(R + 32768, L))
// with R = rowmax + 1 and h the unsaturated shift. R - h itself is one
// shift: with v = s * m, h = (v + half - [v < 0]) >> sh (floor), and
//   R - h = (R * 2^sh + 2^sh - 1 - half - v + [v < 0]) >> sh   (floor),
// which stays inside int32: |v| <= 2^21 * 255 < 2^29 and |R| <= 2^(29 - sh) + 2
// for sh <= 29. For sh >= 30 every h is 0 (|v| < 2^29 <= half), the same
// as m = 0 with sh = 0. [v < 0] = [s < 0] when m > 0; when m = 0 the term
// is below the rounding step either way (2^sh - half <= 2^sh - 1).
struct ScoreIndex {
  // general form (a shift >= 32 gives 0: multiplier 0 instead)
  int32_t m24;
  uint32_t sh, half, w, rmp1;
  // short form
  uint32_t fsh, fw;
  int32_t fnm, fK, flo, fhi;
  __device__ __forceinline__ ScoreIndex(const AttnArgs &a, int32_t rowmax) {
    m24 = a.qk_s >= 32 ? 0 : (int32_t)a.qk_m;
    sh = a.qk_s >= 32 ? 0u : a.qk_s;
    half = sh ? 1u << (sh - 1) : 0u;
    w = min(sh, 1u);
    rmp1 = (uint32_t)(uint16_t)(rowmax + 1);
    fsh = a.qk_s >= 30 ? 0u : a.qk_s;
    fnm = a.qk_s >= 30 ? 0 : -(int32_t)a.qk_m;
    fw = min(fsh, 1u);
    const int32_t R = rowmax + 1;
    fK = (int32_t)(((uint32_t)R << fsh) + ((1u << fsh) - 1u) - (fsh ? 1u << (fsh - 1) : 0u));
    flo = min(R - 32767, IW_SEXP_LUT - 1), fhi = min(R + 32768, IW_SEXP_LUT - 1);
  }
  // every key counts, row maximum below 32767
  __device__ __forceinline__ uint32_t full(int32_t s) const {
    const uint32_t y = (uint32_t)(__mul24(s, fnm) + fK) - (uint32_t)__builtin_amdgcn_sbfe(s, 31, fw);
    return (uint32_t)med3i((int32_t)y >> fsh, flo, fhi);
  }
  // requant (24-bit product: |score| < 2^21 and an 8-bit multiplier),
  // round-half-away shift, int16 saturation
  __device__ __forceinline__ uint32_t any(int32_t s) const {
    const int32_t v = __mul24(s, m24);
    const uint32_t tr = (uint32_t)v + half + (uint32_t)__builtin_amdgcn_sbfe(v, 31, w);
    const int32_t h16 = clampi((int32_t)tr >> sh, -32768, 32767);
    return min((rmp1 - (uint32_t)h16) & 0xffffu, (uint32_t)(IW_SEXP_LUT - 1));
  }
};

}  // namespace iw
