// Helpers of the triangular solves: 16 x 16 tiles in the accumulator layout of
// the 16x16 matrix instructions (lane l holds rows 4 (l / 16) + j, register j,
// of column l % 16), and division by a divisor used many times.
#pragma once

#include "device_common.h"

namespace aclblas {
namespace dev {

typedef float F32x4 __attribute__((ext_vector_type(4)));

// The value of lane group g (16 lanes) in every group.
template <int g>
__device__ __forceinline__ float GroupBroadcast(float v)
{
    const uint32_t u = __float_as_uint(v);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);  // {g0 g0 g2 g2}, {g1 g1 g3 g3}
    const uint32_t s = (g & 1) ? p[1] : p[0];
    const auto q = __builtin_amdgcn_permlane32_swap(s, s, false, false);
    return __uint_as_float((g & 2) ? q[1] : q[0]);
}

// x / u with r = 1 / u (correctly rounded): two residual corrections of x r.
// The first leaves the quotient within one ulp, from where one more with the
// rounded reciprocal gives the correctly rounded quotient (Markstein, IBM J.
// Res. Dev. 34, 1990) while no intermediate under- or overflows: Dividable.
__device__ __forceinline__ float DivideBy(float x, float u, float r)
{
    float q = x * r;
    q = fmaf(fmaf(-u, q, x), r, q);
    return fmaf(fmaf(-u, q, x), r, q);
}

// |v| in [2^-60, 2^60) (or +0 when ZERO): DivideBy is exact on such operands.
template <bool ZERO>
__device__ __forceinline__ bool Dividable(float v)
{
    const uint32_t u = __float_as_uint(v);
    const bool range = (u & 0x7FFFFFFFu) - ((127u - 60u) << 23) < (120u << 23);
    return range || (ZERO && u == 0u);
}

}  // namespace dev
}  // namespace aclblas
