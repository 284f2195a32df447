// Quotients of integer sums by one row's scale (the decode rule of the int8 family): arithmetic alone, so that it can be checked without a GPU.
#pragma once

#if defined(__HIP__)
#define TERNA_ROW_FUNCTION __device__
#else
#include <cmath>
#define TERNA_ROW_FUNCTION
#endif

namespace terna {

// The IEEE quotients: an estimate by the scale's reciprocal and one correction by its exact remainder (Markstein) for
// scales whose products and remainders are normal numbers -- every row's but one of absurd or no finite numbers -- three
// operations instead of a division's dozen.  (tests/row_quotient_check.cpp: all mantissas of a bf16 scale times all sums up to 2^22, the ends of the range.)
struct RowQuotient {
    float s, inverse;
    bool plain;
    TERNA_ROW_FUNCTION explicit RowQuotient(float scale) : s(scale), inverse(1.0f / scale), plain(scale >= 0x1p-60f && scale <= 0x1p60f) {}
    template <int F>
    TERNA_ROW_FUNCTION void of(float (&x)[F]) const
    {
        float q[F];
#pragma unroll
        for (int v = 0; v < F; ++v) {
            q[v] = x[v] * inverse;
            q[v] = fmaf(fmaf(-q[v], s, x[v]), inverse, q[v]);
        }
        if (!plain) {
#pragma unroll
            for (int v = 0; v < F; ++v) q[v] = x[v] / s;
        }
#pragma unroll
        for (int v = 0; v < F; ++v) x[v] = q[v];
    }
};

}  // namespace terna
