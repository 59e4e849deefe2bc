// fp32 activations as the uint4 projections read them: every value split exactly into three bf16
// terms (split3x8), laid out as the A operands of v_mfma_f32_32x32x16_bf16, with the sum of every
// 32 inputs. The kernel that makes the activations (a norm, the gated epilogue) writes them beside
// its fp32 output when a projection follows; split_planes makes them from a stored x.
//
// One row tile (32 rows) and group (64 inputs) takes 12 KiB: [term][k-step][lane][8] with lane =
// row % 32 + 32 h holding inputs 32 h + 8 step .. + 7, so a wavefront loads an operand as one
// contiguous KiB. Rows past the last one of a tile are never written; an MFMA
// keeps rows apart, and their results are never stored.
#pragma once

#include "common.h"

namespace tessery {

struct Planes {
  uint16_t* terms;  // [tile][group][3][4][64][8]
  float* sums;      // [tile][group][half][row % 32]
};

constexpr int kPlaneRows = 32;
constexpr int kPlaneTerm = 4 * 64 * 8, kPlaneGroup = 3 * kPlaneTerm, kPlaneSums = 64;

inline size_t planes_bytes(int rows, int k) {
  const size_t tiles = (static_cast<size_t>(rows) + kPlaneRows - 1) / kPlaneRows;
  return tiles * static_cast<size_t>(k / 64) * (kPlaneGroup * 2 + kPlaneSums * 4);
}

// The planes of [rows, k] activations at `base` (16-byte aligned, planes_bytes).
inline Planes planes_at(void* base, int rows, int k) {
  const size_t tiles = (static_cast<size_t>(rows) + kPlaneRows - 1) / kPlaneRows;
  auto terms = static_cast<uint16_t*>(base);
  return Planes{terms, reinterpret_cast<float*>(terms + tiles * static_cast<size_t>(k / 64) *
                                                            kPlaneGroup)};
}

struct Split3 {
  uint32_t t[3];  // the three bf16 terms, each in the upper half of its word
};
__device__ __forceinline__ Split3 split3(float x) {
  Split3 r;
  r.t[0] = __float_as_uint(x);
  const float r1 = x - __uint_as_float(r.t[0] & 0xffff0000u);
  r.t[1] = __float_as_uint(r1);
  r.t[2] = __float_as_uint(r1 - __uint_as_float(r.t[1] & 0xffff0000u));
  return r;
}
__device__ __forceinline__ uint32_t upper_pair(uint32_t first, uint32_t second) {
  return __builtin_amdgcn_perm(second, first, 0x07060302u);
}

// Columns col .. col + 3 of a row, from eight consecutive lanes that hold 32 aligned columns of
// it. Every writer adds a half group's sum in this order: 4 inputs, then lanes 1, 2 and 4 apart.
__device__ __forceinline__ void store_planes4(const Planes& p, int row, int col, int groups,
                                              floatx4 v) {
  // rounded values, not products to be contracted with what follows
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float x = v[j];
    asm("" : "+v"(x));
    v[j] = x;
  }
  const size_t at = static_cast<size_t>(row / kPlaneRows) * groups + (col >> 6);
  const int half = (col >> 5) & 1, lane = row % kPlaneRows + 32 * half;
  Split3 s[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) s[j] = split3(v[j]);
  uint16_t* const dst =
      p.terms + at * kPlaneGroup + ((col >> 3) & 3) * 512 + lane * 8 + (col & 4);
#pragma unroll
  for (int t = 0; t < 3; ++t)
    *reinterpret_cast<uint2v*>(dst + t * kPlaneTerm) =
        uint2v{upper_pair(s[0].t[t], s[1].t[t]), upper_pair(s[2].t[t], s[3].t[t])};
  float sum = (v[0] + v[1]) + (v[2] + v[3]);
  sum += __shfl_xor(sum, 1);
  sum += __shfl_xor(sum, 2);
  sum += __shfl_xor(sum, 4);
  if ((col & 31) == 0) p.sums[at * kPlaneSums + lane] = sum;
}

}  // namespace tessery
