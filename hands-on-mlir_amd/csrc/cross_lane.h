// Cross-lane reductions for 64-lane wavefronts on gfx950 that stay in the
// vector ALU: data-parallel-primitive (DPP) operands inside a row of 16 lanes,
// v_permlane16_swap / v_permlane32_swap between rows.  A __shfl_xor is an LDS
// round trip (ds_bpermute) of a hundred cycles or more; these are one
// instruction each.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hom {

// v + (v of the lane a DPP control selects); CTRL is the dpp_ctrl encoding.
template <int CTRL> __device__ __forceinline__ float addDpp(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(
                 0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// Sum over groups of N consecutive lanes (N = 4, 8 or 16, groups aligned to
// N), result in every lane of the group: quad permutes exchange lanes ^1 and
// ^2, the half-row and row mirrors pair each lane with one of the other quad /
// the other half of its row.
template <int N> __device__ __forceinline__ float sumAcrossLanes(float v) {
  static_assert(N == 4 || N == 8 || N == 16, "group size");
  v = addDpp<0xB1>(v); // quad_perm [1,0,3,2]
  v = addDpp<0x4E>(v); // quad_perm [2,3,0,1]
  if (N >= 8)
    v = addDpp<0x141>(v); // row_half_mirror
  if (N >= 16)
    v = addDpp<0x140>(v); // row_mirror
  return v;
}

// v_permlane32_swap exchanges the upper half of its first operand with the
// lower half of its second; given the same value twice it returns (lower-half
// values, upper-half values) in every lane pair (l, l ^ 32).
__device__ __forceinline__ float pairMax(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v),
                                                  __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float pairSum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v),
                                                  __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Two lanes l, l ^ 32 that each hold half of two 16-byte vectors (dwords even0, even1 of the
// one, odd0, odd1 of the other; the lower lane the lower half): the lower lane gets
// the even vector, the upper one the odd.
typedef uint32_t lanes4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ lanes4 joinHalves(uint32_t even0, uint32_t even1, uint32_t odd0,
                                             uint32_t odd1) {
  const auto a = __builtin_amdgcn_permlane32_swap(even0, odd0, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(even1, odd1, false, false);
  return lanes4{a[0], b[0], a[1], b[1]};
}
// The way back: a lane has the even (lower lane) or odd vector v and gets the dwords
// even0, even1, odd0, odd1 of its half.
__device__ __forceinline__ lanes4 splitHalves(lanes4 v) {
  const auto a = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
  return lanes4{a[0], b[0], a[1], b[1]};
}
// Rows of 16 lanes: the odd ones of a against the even ones of b (its own inverse).
typedef uint32_t lanes2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void swapRows(lanes4 &a, lanes4 &b) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const auto r = __builtin_amdgcn_permlane16_swap(a[i], b[i], false, false);
    a[i] = r[0];
    b[i] = r[1];
  }
}
// Lanes 8 .. 15 of a's rows against lanes 0 .. 7 of b's.
__device__ __forceinline__ void swapHalfRows(lanes4 &a, lanes4 &b) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int x = int(a[i]), y = int(b[i]); // (0x128: rotate a row of 16 lanes by 8)
    a[i] = uint32_t(__builtin_amdgcn_update_dpp(x, y, 0x128, 0xf, 0xc, false));
    b[i] = uint32_t(__builtin_amdgcn_update_dpp(y, x, 0x128, 0xf, 0x3, false));
  }
}
// v_permlane16_swap exchanges the odd rows of its first operand with the even
// rows of its second: the same value twice gives (even-row values, odd-row
// values) in every lane pair (l, l ^ 16).
__device__ __forceinline__ float rowPairSum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v),
                                                  __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Sum over the whole wavefront, result in every lane.
__device__ __forceinline__ float waveSum(float v) {
  return pairSum(rowPairSum(sumAcrossLanes<16>(v)));
}

} // namespace hom
