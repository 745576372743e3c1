// crm_round.hpp -- the three-term Adams-Bashforth sum with every rounding spelled out.
//
// at a + bt b + ct c is summed in FP64 as one product rounded by itself and two fused
// multiply-adds.  Left to the compiler, the product that stands alone changed with the
// arrangement of the surrounding loop, and so did the last bit of the velocities (in the mixed
// engine a last bit of the FP64 sum flips an FP32 rounding about once in 1e8 values, which the
// eddy viscosity then amplifies).  The order of each shape is the one its results have always
// had.  The same source builds for the host, so that a test can check every shape's order.
#pragma once

#if defined(__HIP__)
#define CRM_ROUND_HD __host__ __device__
#else
#define CRM_ROUND_HD
#endif

#ifndef CRM_NS
#define CRM_NS crm
#endif

namespace CRM_NS {

// the term whose product is rounded by itself
enum class AbAlone { A, B, C };
enum class AbField { U, V, W };

// columns: of an instance (nx ny); y3: 3D; fp64: the engine whose fields are FP64
constexpr AbAlone ab_alone(AbField f, int columns, bool y3, bool fp64) {
  if (columns == 64) return f != AbField::V ? AbAlone::C : fp64 ? AbAlone::A : AbAlone::B;
  return f == AbField::W && columns < 64 && !y3 ? AbAlone::A : AbAlone::B;
}

template <AbAlone ALONE>
CRM_ROUND_HD inline double ab_sum(double at, double a, double bt, double b, double ct, double c) {
#pragma clang fp contract(off)
  if constexpr (ALONE == AbAlone::A)
    return __builtin_fma(ct, c, __builtin_fma(bt, b, at * a));
  else if constexpr (ALONE == AbAlone::B)
    return __builtin_fma(ct, c, __builtin_fma(at, a, bt * b));
  else
    return __builtin_fma(at, a, __builtin_fma(bt, b, ct * c));
}

}  // namespace CRM_NS
