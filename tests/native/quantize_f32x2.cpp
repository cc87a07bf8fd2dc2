// Host check of the two-float quantization (qa_round_f32x2): wherever it does
// not ask for the double form, clip(rounded + zp) must be the reference's
// clip(nearbyint(double(x) / scale) + zp) (qa_kernels.cpp:363-376). Scales
// over the form's whole range, values of every magnitude up to the largest
// float, quotients on and beside half-integers, infinities and NaN. Exit
// status 0 = equal.
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "qa_common.h"

int main(int argc, char** argv) {
    const long trials = argc > 1 ? atol(argv[1]) : 2000000;
    std::mt19937_64 g(777);
    long bad = 0, n = 0, slow_n = 0;
    auto check = [&](float x, double scale, int64_t zp, int64_t lo,
                     int64_t hi) {
        if (!qa_f32_form_ok(scale, zp, lo, hi)) return;
        const double inv = 1.0 / scale;
        const float invf = (float)inv, invlo = (float)(inv - (double)invf);
        bool slow = false;
        const float q = qa_round_f32x2(x, invf, invlo, &slow) + (float)zp;
        ++n;
        if (slow) {
            ++slow_n;
            return;
        }
        const double want = std::fmin(
            std::fmax(std::nearbyint((double)x / scale) + (double)zp,
                      (double)lo), (double)hi);
        // the kernel's med3; of a NaN it is anything but decided
        const bool same = q == q && want == want &&
                          (double)std::fmin(std::fmax(q, (float)lo),
                                            (float)hi) == want;
        if (!same && bad++ < 10)
            printf("mismatch x=%a scale=%a zp=%lld got=%a want=%a\n",
                   (double)x, scale, (long long)zp, (double)q, want);
    };
    struct Range {
        int64_t zp, lo, hi;
    };
    const Range ranges[] = {{0, -128, 127},   {130, 0, 255},
                            {255, 0, 255},    {0, -32768, 32767},
                            {65535, 0, 65535}, {0, 0, (1 << 19) - 1},
                            {1 << 22, (1 << 22) - 100, 1 << 22}};
    const double scales[] = {0x1p-60, 1e-12, 1e-4, 0.01, 0.037, 1.0,
                             3.7,     1e9,   0x1p60};
    const float xs[] = {0.f,      -0.f,     FLT_MIN,  0x1p-149f, 1e-30f,
                        1.3e37f,  1e37f,    1e38f,    3.4e38f,   FLT_MAX,
                        INFINITY, NAN,      0x1.fffffep+67f, 0x1p68f,
                        1e30f,    16777216.f};
    for (const Range& r : ranges)
        for (double s : scales)
            for (float x : xs)
                for (int sign = 0; sign < 2; ++sign)
                    check(sign ? -x : x, s, r.zp, r.lo, r.hi);
    for (long i = 0; i < trials; ++i) {
        const Range& r = ranges[g() % 7];
        const double s =
            g() % 4 ? scales[g() % 9]
                    : std::ldexp(1.0 + (double)(g() >> 12) * 0x1p-52,
                                 (int)(g() % 120) - 60);
        float x;
        if (g() % 2) {  // any bits
            const uint32_t b = (uint32_t)g();
            memcpy(&x, &b, 4);
        } else {  // a quotient on or beside a half-integer
            const double h =
                (double)((int64_t)(g() % (1 << 20)) - (1 << 19)) + 0.5;
            x = (float)(h * s);
            const int k = (int)(g() % 5) - 2;
            for (int j = 0; j < (k < 0 ? -k : k); ++j)
                x = std::nextafterf(x, k < 0 ? -INFINITY : INFINITY);
        }
        check(x, s, r.zp, r.lo, r.hi);
    }
    printf("checked %ld, double form %ld, mismatches %ld\n", n, slow_n, bad);
    return bad != 0;
}
