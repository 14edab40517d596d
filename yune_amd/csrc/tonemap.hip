// tonemap.hip — kernels/post-proc/tonemap.cl on a device image.
//
// Bound by the double-precision arithmetic of a pixel's four x^(1/2.2), whose
// operations and order are fixed (yn_fmath.h).  1920x1080, Reinhard: 69.8 ->
// 42.9 us a call (2.1 TB/s of the 4.9 a copy reaches) by leaving out the four
// x^1, by one test for all special cases of a pixel, and by the shorter
// division below (3 us of it).
#define YNF_PLAIN_CONSTANTS     // one short kernel: its constants fit the scalar registers
#include "yn_internal_dev.h"
#include "yn_shade.h"

namespace yune {

// John Hable's filmic curve (tonemap.cl:49-58) on one channel: shoulder
// 0.15, linear 0.50 at angle 0.10, toe 0.20 with 0.02 / 0.30; no white-point
// division, as in the reference.
__device__ __forceinline__ float hable_curve(float x)
{
    const float sA = 0.15f, sB = 0.50f, sC = 0.10f, sD = 0.20f, sE = 0.02f, sF = 0.30f;
    return (x * (sA * x + sC * sB) + sD * sE) / (x * (sA * x + sB) + sD * sF) - sE / sF;
}

// x^g for g = 1/2.2f and a positive finite x, with ynf_powf's operations on
// the way it then takes (its result is inside float's range): the division
// of ynf_log, whose operands lie in [-0.3, 0.42] and [1.7, 2.42], by Newton's
// steps and Markstein's correction instead of the compiler's sequence, which
// also scales for ranges that do not occur.  (Same bits as ynf_powf for all
// 2^31 positive floats, and as n / d for 1.7e10 random m, on gfx950.)
__device__ __forceinline__ double div_near_one(double n, double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = fma(fma(-d, r, 1.0), r, r);
    r = fma(fma(-d, r, 1.0), r, r);
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
}

__device__ __forceinline__ float pow_gamma(float x)
{
    int e;
    const double m = ynf_log_split((double)x, &e);
    const double t = (double)(1 / 2.2f) * ynf_log_series(div_near_one(m - 1.0, m + 1.0), e);
    return (float)ynf_exp(t);
}

// x^1 by ynf_powf: x, or the default NaN (compared for all 2^32 floats).
__device__ __forceinline__ float pow_one(float x) { return x != x ? __builtin_nanf("") : x; }

// tonemap.cl:14-47, op 0: Reinhard with lum_white = 1 (identity up to
// rounding); op 1: the Hable curve the reference ships commented out
// (tonemap.cl:29).  The clamp is discarded as in the reference, then gamma
// 1/2.2.
__global__ __launch_bounds__(256) void k_tonemap(const float4* in, float4* out, int n, int op)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    f4 col = ld(in[i]);
    f4 ldr;
    if (op == 1) {
        ldr = mk(hable_curve(col.x), hable_curve(col.y), hable_curve(col.z), hable_curve(col.w));
    } else {
        float lum_world = 0.212671f * col.x + 0.715160f * col.y + 0.072169f * col.z + 0.001f;
        float lum_white = 1.0f;
        float lum_display = lum_world * (1 + lum_world / (lum_white * lum_white)) / (1 + lum_world);
        f4 sc = col / lum_world;
        ldr = mk(pow_one(sc.x), pow_one(sc.y), pow_one(sc.z), pow_one(sc.w)) * lum_display;
    }
    auto plain = [](float x) { return __float_as_uint(x) - 1u < 0x7f7fffffu; };     // positive and finite
    if (plain(ldr.x) && plain(ldr.y) && plain(ldr.z) && plain(ldr.w)) {
        out[i] = make_float4(pow_gamma(ldr.x), pow_gamma(ldr.y), pow_gamma(ldr.z), pow_gamma(ldr.w));
    } else {
        const float g = 1 / 2.2f;
        out[i] = make_float4(ynf_powf(ldr.x, g), ynf_powf(ldr.y, g), ynf_powf(ldr.z, g), ynf_powf(ldr.w, g));
    }
}

void launch_tonemap(const float4* in, float4* out, int n, int op, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_tonemap, dim3((n + 255) / 256), dim3(256), 0, s, in, out, n, op);
}

}  // namespace yune
