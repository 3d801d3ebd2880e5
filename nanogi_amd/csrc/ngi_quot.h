// IEEE reciprocals and quotients of a ray's set-up in fused multiply-adds.
//
// rcp_newton: one Newton step makes any FP32 approximation within 1 ulp of
// 1 / d (the hardware's reciprocal) the correctly rounded one, but for the
// greatest significand (0x1.fffffe), whose approximation has to be the correct
// one already, as the hardware's is.  div_markstein:
// n / d from rd = 1 / d correctly rounded (P. Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", IBM J. Res.
// Dev. 34(1), 1990).  Both equal the IEEE division bit for bit where
// quot_exact says so: three and three instructions instead of ten each.
//
// The range, with |n| <= |d|: |d| >= 1e-20 keeps 1 / d far from overflow;
// |n| >= 2^-100 makes the residual n - q d exact; |d| < 2^26 keeps the quotient
// at 2^-126 or above.  A denormal quotient halfway between its neighbours
// rounds the wrong way: 0x1.508c0ap-87 / 0x1.3eep+51 is 0x1.0e4p-138, the steps
// give 0x1.0e2p-138.
// tests/quot_check.cpp compares both with the division over the range.
#pragma once

#include <math.h>

#include "ngi_common.h"

namespace ngi {

// r: 1 / d within 1 ulp.
NGI_HD float rcp_newton(float d, float r) { return fmaf(fmaf(-d, r, 1.0f), r, r); }

NGI_HD float div_markstein(float n, float d, float rd) {
    const float q = n * rd;
    return fmaf(fmaf(-d, q, n), rd, q);
}

// least: the smallest |n| of the quotients by d.
NGI_HD bool quot_exact(float least, float d) {
    const float a = fabsf(d);
    return least >= 7.8886091e-31f && a >= 1e-20f && a < 67108864.0f;   // 2^-100, guard_dir's bound, 2^26
}

}  // namespace ngi
