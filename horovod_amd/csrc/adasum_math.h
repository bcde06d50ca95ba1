// adasum_math.h -- the arithmetic of Adasum's pairwise combine (device code, not installed): sums over
// a workgroup, the coefficient formula, the scaled add.
#ifndef HVDHIP_ADASUM_MATH_H
#define HVDHIP_ADASUM_MATH_H

#include "internal.h"
#include "vecmem.h"

namespace hvdhip {

struct Triple {
  double d, a, b;
};

// x + (x of the lane that the DPP control CTRL names), for the rows in ROW_MASK; lanes without a
// source (or outside the mask) add zero.  Two 32-bit DPP moves and one add: data-parallel
// primitives move data between lanes inside the vector ALU, where a shuffle goes through the LDS
// crossbar and costs a memory-pipeline round trip per step.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_add(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  const int lo2 = __builtin_amdgcn_update_dpp(0, lo, CTRL, ROW_MASK, 0xf, false);
  const int hi2 = __builtin_amdgcn_update_dpp(0, hi, CTRL, ROW_MASK, 0xf, false);
  return x + __hiloint2double(hi2, lo2);
}

// Sum over each row of 16 lanes by a shifted-add scan; the totals arrive in lanes 15, 31, 47 and 63.
__device__ __forceinline__ double row_sum(double x) {
  x = dpp_add<0x111, 0xf>(x);  // row_shr:1
  x = dpp_add<0x112, 0xf>(x);  // row_shr:2
  x = dpp_add<0x114, 0xf>(x);  // row_shr:4
  return dpp_add<0x118, 0xf>(x);  // row_shr:8
}

// Sum over the 64 lanes of a wavefront in a fixed order; the total arrives in lane 63.  First the rows of 16
// lanes, then lane 15 of rows 0 and 2 into rows 1 and 3, then lane 31 into rows 2 and 3.
__device__ __forceinline__ double wave_sum(double x) {
  x = row_sum(x);
  x = dpp_add<0x142, 0xa>(x);  // row_bcast:15 into rows 1 and 3
  x = dpp_add<0x143, 0xc>(x);  // row_bcast:31 into rows 2 and 3
  return x;
}

// A lane's value in every lane.
__device__ __forceinline__ double lane_value(double x, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                          __builtin_amdgcn_readlane(__double2loint(x), lane));
}

__device__ __forceinline__ Triple wg_reduce(Triple t) {
  // wave64 sums, then the four wavefronts in order through LDS
  t.d = wave_sum(t.d);
  t.a = wave_sum(t.a);
  t.b = wave_sum(t.b);
  __shared__ double red[3][kWG / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 63) {
    red[0][wave] = t.d;
    red[1][wave] = t.a;
    red[2][wave] = t.b;
  }
  __syncthreads();
  Triple r = {0., 0., 0.};
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 0; w < kWG / 64; ++w) {
      r.d += red[0][w];
      r.a += red[1][w];
      r.b += red[2][w];
    }
  }
  return r;  // valid in thread 0
}

// Coefficients of adasum.h:397-404 from a layer's sums.
__device__ __forceinline__ void layer_coeffs(const Triple& r, double guard, double* ca, double* cb) {
  *ca = 1.;
  *cb = 1.;
  if (r.a >= guard) *ca = 1.0 - r.d / r.a * 0.5;
  if (r.b >= guard) *cb = 1.0 - r.d / r.b * 0.5;
}

// ScaledAdd<T>, adasum.h:429-435: acoeff * a[i] + bcoeff * b[i] with the operands widened to
// double: two rounded products, their rounded sum, then the conversion to T.  Contraction is
// switched off for this expression (device code contracts by default, and the rounded-operation
// intrinsics are plain operators to the compiler), so no product is fused into the sum.
template <typename T>
struct Axpby {
  static __device__ __forceinline__ T f(double ca, T a, double cb, T b) {
#pragma clang fp contract(off)
    const double pa = ca * (double)a, pb = cb * (double)b;
    return (T)(pa + pb);
  }
};
// ScaledAddfp16, adasum.h:482-500: float coefficients, t = ca*a rounded to fp32, r = fma(cb, b, t)
// rounded to fp32, then to half.  Both fp32 results are kept apart from what follows them: a fused
// mixed-precision product would take a +0 addend and lose the sign of a -0 product, and a fused
// fma-and-narrow rounds the exact sum once where fmadd_ps followed by cvtps_ph rounds twice
// (it differs from the reference in the last bit of some elements).  The widening of b folds
// into the fma, and pairs of results narrow with one packed conversion.
template <>
struct Axpby<half_t> {
  static __device__ __forceinline__ half_t f(double ca, half_t a, double cb, half_t b) {
    const float t = opaque(__fmul_rn((float)ca, (float)a));
    return (half_t)opaque(__fmaf_rn((float)cb, (float)b, t));
  }
};

}  // namespace hvdhip

#endif  // HVDHIP_ADASUM_MATH_H
