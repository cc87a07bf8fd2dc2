// Shared by the 16-bit convolution kernels: the exact float64 forms of the
// fixed-point multiplies, and the launcher of the LDS-resident byte split.
#pragma once

#include "qa_conv_mfma.h"

namespace qa {

// Most LDS bytes a work-group of the LDS-resident form takes (of a CU's 160
// KB; the rest is left to the runtime).
constexpr int64_t BSL_LDS_MAX = 152 * 1024;

// qa_conv_bs.hip: `b` in launch form, the byte split's own conditions met.
bool conv_bsl_applies(const ConvArgs& b);
int64_t bsl_lds(const ConvArgs& b, int wm);
// wm: 16-channel blocks a work-group (0: the library's choice)
bool launch_conv_bsl(const ConvArgs& b, bool narrow, int wm, hipStream_t st);

namespace {

// The 128-bit requantization of one value (out of line: the float64 form
// below hands it the rare values it cannot decide).
__device__ __noinline__ int64_t requant_exact(int64_t x, int64_t m, int64_t s,
                                              int64_t zp, int64_t lo,
                                              int64_t hi) {
    return qa_clip128(qa_mbqm_fast(x, m, s) + zp, lo, hi);
}

// Exact float64 forms of the fixed-point multiplies of the 16-bit epilogue
// (qa_mbqm: floor(x m 2^-ts + 1/2), ts = 31 + shift):
//  * requantize, |x| < 2^53, |m| < 2^31, 1 <= ts <= 120, clip bounds within
//    2^19: y = fma(x, m 2^-ts, 1/2 + zp) is one rounding of the exact value
//    (x and m 2^-ts are exact doubles), |error| <= 2^-52 |y|; below |y| =
//    2^20, floor(y) is the exact result unless frac(y) lies within 2^-30 of
//    0 or 1 (those values take requant_exact); above, the clip gives the
//    same bound either way.
//  * multiplies of a clipped value (|d| < 2^20) by |m| < 2^31 with 1 <= ts
//    <= 53 (the residual Add, the rescaled copy): d m is an exact double
//    below 2^51, and so is d m 2^-ts + 1/2, so floor gives the exact result.
struct MulD {
    double md;
    bool ok;
};
__device__ __forceinline__ MulD mul_d(int64_t m, int64_t shift, int64_t tmax) {
    const int64_t ts = 31 + shift;
    MulD r;
    r.ok = ts >= 1 && ts <= tmax && m > -((int64_t)1 << 31) &&
           m < ((int64_t)1 << 31);
    r.md = r.ok ? ldexp((double)m, -(int)ts) : 0.0;
    return r;
}
__device__ __forceinline__ double round_d(double d, double md) {
    return floor(fma(d, md, 0.5));
}
__device__ __forceinline__ double clamp_d(double v, int64_t lo, int64_t hi) {
    return fmin(fmax(v, (double)lo), (double)hi);
}

}  // namespace
}  // namespace qa
