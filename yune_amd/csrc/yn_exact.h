// yn_exact.h — correctly rounded reciprocal and square root on the device,
// in fewer instructions than the compiler's.
//
// 1 / x and sqrt(x) must round as IEEE says, since the CPU oracle's do.  The
// compiler's sequences (division: 11 instructions and the waits its flag
// register asks for; square root: 16) also cover denormals, infinities and
// zeros.  Here an argument whose exponent keeps every intermediate normal
// takes the hardware's approximation and Newton's steps in FMAs (Markstein,
// IBM J. R&D 34, 1990), any other the compiler's sequence; a wave without
// such a lane skips it.  Compared with the compiler's results for all 2^32
// arguments on gfx950: equal for exponent fields 1..252 (x_rcp, either sign)
// and 25..254 (x_sqrt, positive), the ranges tested below.
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIPCC__)

namespace yune {

__device__ __forceinline__ float x_rcp(float x)
{
    float r;
    if (__builtin_expect((__float_as_uint(x) << 1) - (1u << 24) < (252u << 24), 1)) {
        r = __builtin_amdgcn_rcpf(x);
        r = fmaf(fmaf(-x, r, 1.0f), r, r);
    } else {
        r = 1.0f / x;
    }
    return r;
}

__device__ __forceinline__ float x_sqrt(float x)
{
    float s;
    if (__builtin_expect(__float_as_uint(x) - (25u << 23) < (230u << 23), 1)) {
        const float y = __builtin_amdgcn_rsqf(x);
        s = x * y;
        s = fmaf(fmaf(-s, s, x), 0.5f * y, s);
    } else {
        s = sqrtf(x);
    }
    return s;
}

// 1 / sqrt(x), both rounded.
__device__ __forceinline__ float x_rcp_sqrt(float x)
{
    float r;
    if (__builtin_expect(__float_as_uint(x) - (25u << 23) < (230u << 23), 1)) {
        const float y = __builtin_amdgcn_rsqf(x);
        float s = x * y;
        s = fmaf(fmaf(-s, s, x), 0.5f * y, s);      // exponent field 76..190
        r = __builtin_amdgcn_rcpf(s);
        r = fmaf(fmaf(-s, r, 1.0f), r, r);
    } else {
        r = 1.0f / sqrtf(x);
    }
    return r;
}

}  // namespace yune

#endif
