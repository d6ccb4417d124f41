// rcp.hpp: reciprocals by the hardware's approximation (no HIP: host tests compile this file)
#pragma once

#include <math.h>

#if defined(__HIPCC__)
#define QIE_RCP_HD __host__ __device__
#else
#define QIE_RCP_HD
#endif

namespace qie {

// 1 / d from an approximation r within one ulp of it (v_rcp_f32): two Newton steps, the IEEE quotient for every d up to 2^126 whose mantissa is not
// all ones, where it may be an ulp off; one step leaves a dozen mantissas wrong.  Infinity, NaN and what lies beyond 2^126: r as it is.
QIE_RCP_HD inline float rcp_from(float d, float r) {
    const float once = fmaf(fmaf(-d, r, 1.0f), r, r), twice = fmaf(fmaf(-d, once, 1.0f), once, once);
    return d <= 0x1p126f ? twice : r;
}

}  // namespace qie
