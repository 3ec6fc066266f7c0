// lm_quotient.h — many values divided by one (device code, and plain C++ for the test that holds it to the division operator)
#pragma once
#include <math.h>

#ifdef __HIP__
#define ZG_ANYWHERE __host__ __device__ __forceinline__
#else
#define ZG_ANYWHERE inline
#endif

namespace zg {

// v / by, rounded as the division operator rounds it, from inv = 1.0f / by: Markstein's correction (P. W. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", 1990): the remainder of v * inv is exact in one fma, and one more rounds the quotient
// correctly.  Five operations where a division takes some twelve, four of them at a quarter of the rate.  A remainder that is not a number
// comes from an infinity or a zero divisor, whose quotient v * inv is already.  (Quotients below 2^-100 may differ in their last bit.)
ZG_ANYWHERE float quotient(float v, float by, float inv) {
    const float q = v * inv, rest = fmaf(-q, by, v);
    return rest == rest ? fmaf(rest, inv, q) : q;
}

}  // namespace zg
