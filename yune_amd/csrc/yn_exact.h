// yn_exact.h — the correctly rounded reciprocal on the device, in fewer
// instructions than the compiler's division.
//
// 1 / x must round as IEEE says, since the oracle's does.  The compiler's
// division (11 instructions and the waits its flag register asks for) also
// covers denormals, infinities and zeros.  Here an argument whose exponent
// keeps every intermediate normal takes the hardware's approximation and one
// of Newton's steps in FMAs (Markstein, IBM J. R&D 34, 1990), any other the
// division; a wave without such a lane skips it.  Compared with the division
// for all 2^32 arguments on gfx950: equal.
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

}  // namespace yune

#endif
