// Double-double arithmetic: sums for the refinement's residuals, products and
// quotients for the transforms' twiddles.
#pragma once

#include "tags_common.h"

namespace tags {

// Double-double accumulation for the refinement residuals: a sum kept as
// hi + lo with every product and addition error carried (Dekker/Knuth exact
// transformations: a b = p + fma(a, b, -p), s = hi + p + e by TwoSum), so that
// b - W x is accurate to about one FP64 rounding of its own size even where
// b and W x cancel. With FP64 residuals alone, refinement stops at a forward
// error of about cond(W) eps; with these it converges to working accuracy.
// Contraction is off here: a fused multiply-add in place of the separate
// product and sum would break the error terms.
struct DD {
    double hi, lo;
};
__device__ inline void dd_mac(DD& d, double a, double b)
{
#pragma clang fp contract(off)
    const double p = a * b;
    const double pe = fma(a, b, -p);
    const double s = d.hi + p;
    const double bb = s - d.hi;
    const double se = (d.hi - (s - bb)) + (p - bb);
    d.hi = s;
    d.lo += pe + se;
}
__device__ inline void dd_add(DD& d, double p)
{
#pragma clang fp contract(off)
    const double s = d.hi + p;
    const double bb = s - d.hi;
    const double se = (d.hi - (s - bb)) + (p - bb);
    d.hi = s;
    d.lo += se;
}
__device__ inline DD dd_plus(DD a, DD b)
{
#pragma clang fp contract(off)
    DD r = a;
    dd_add(r, b.hi);
    r.lo += b.lo;
    return r;
}
__device__ inline DD dd_shfl_xor(DD a, int o)
{
    return DD{__shfl_xor(a.hi, o), __shfl_xor(a.lo, o)};
}
// b - (hi + lo), rounded once
__device__ inline double dd_sub_from(double b, DD d)
{
#pragma clang fp contract(off)
    DD t{b, 0.0};
    dd_add(t, -d.hi);
    return t.hi + (t.lo - d.lo);
}

// Normalised values (|lo| at most half an ulp of hi)
__device__ inline DD dd_norm(double hi, double lo)
{
#pragma clang fp contract(off)
    const double s = hi + lo;
    return DD{s, lo - (s - hi)};
}
__device__ inline DD dd_mul(DD a, DD b)
{
#pragma clang fp contract(off)
    const double p = a.hi * b.hi;
    return dd_norm(p, fma(a.hi, b.hi, -p) + fma(a.hi, b.lo, a.lo * b.hi));
}
__device__ inline DD dd_div(DD a, double d)
{
#pragma clang fp contract(off)
    const double q = a.hi / d;
    return dd_norm(q, (fma(-q, d, a.hi) + a.lo) / d);
}
__device__ inline DD dd_sum(DD a, DD b)
{
#pragma clang fp contract(off)
    const DD s = dd_plus(a, b);
    return dd_norm(s.hi, s.lo);
}

}  // namespace tags
