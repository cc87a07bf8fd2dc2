// 16-bit convolutions / GEMMs on the int8 matrix cores (the byte split of
// qa_conv_f64.hip) with the weights resident in LDS.
//
// A 16-bit product is four int8 ones, so such a layer does four times the
// MFMAs of its 8-bit form over twice the bytes; what bounded it was not
// that but re-reading both weight planes from L2 for every 16-pixel tile
// (half of the late layers' time), one tile a wave with nothing in flight
// across tiles, and an epilogue of 64-bit integer arithmetic and 2-byte
// stores. Here a work-group of 8 waves keeps its 16 WM channels' weights, all
// of K and both planes, in LDS in fragment order (one 1 KB direct load a
// fragment, read back as whole 1 KB rows without conflicts), and each wave
// walks 16-pixel tiles, the activations of the next D K-steps in flight
// across tile boundaries. The weights are the first MFMA operand: a lane
// ends with 4 consecutive channels of one pixel, and the sum of the pixel's
// bytes (against a row of ones) in a register of its own. The epilogue is
// float64 throughout: the four sums (each exact in int32) combine into the
// exact sum below 2^53 by fused multiply-adds, the requantization is one
// more (the bounds of mul_d), and 4 channels are stored, and their residual
// read, as 8 bytes. The table reads of all of a lane's values are issued
// together.
//
// YOLOv8n-cls int16, batch 64, 30 launches: 852 -> 500 us in all (stem 80
// -> 40, 3x3 32 -> 64 at 56x56 35 -> 18, 3x3 256 -> 256 at 7x7 37 -> 14, the
// 1280 -> 1000 head 31 -> 9). Left: the float64 epilogue, about 100 cycles a
// value and SIMD, and single waves waiting on their stores between tiles;
// 16 waves a work-group, or registers held to 4 waves a SIMD, were slower.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <type_traits>

#include "qa_conv_bs.h"

namespace qa {
namespace {

constexpr int BS_WAVES = 8;

struct BsChan {
    double mul;  // m 2^-(31 + shift)
    double add;  // (128 + x_add) W + bias
};

// Scalars of the epilogue in float64.
struct BsEpi {
    double c0, qlo, qhi;                              // 1/2 + zp, clip bounds
    double ra, rb, za, zb, asgn, azp, alo, ahi, rso;  // residual Add
    double r2, z2, zo2, lo2, hi2;                     // rescaled copy
};

constexpr int BIAS_LIM_LOG2 = 51;

// A 16-bit activation table for LDS (qa_plan_lut_i16): {base, entries with
// the format's tag, two groups}, then per group of 16 consecutive entries 8
// bytes: the first entry and the next group's first as uint16 above base, and
// 2 bits an entry, its difference (+ 2) from the rounded line between them.
// A smooth table (SiLU over 2^16 levels is within one step of those lines)
// then takes 32 KB instead of 256 KB; up to two groups that are not (where
// the clip cuts in) are named in the header, and their entries read from the
// table itself.
constexpr int LUTP_HEAD = 16;
// In the entries' word, above their 17 bits: the kernel reads a plan only
// when it is one, of a table as long as the descriptor's.
constexpr int LUTP_TAG = 0x51a80000;

__device__ __forceinline__ int lutp_get(const uint2* t, int base, int i) {
    const uint2 w = t[i >> 4];
    const int f = i & 15;
    const int k0 = (int)(w.x & 0xffffu), d = (int)(w.x >> 16) - k0;
    return base + k0 + ((d * f + 8) >> 4) + (int)(w.y >> (2 * f) & 3u) - 2;
}

__device__ __noinline__ int bs_exact(const int64_t* pre_p,
                                     const int64_t* mult,
                                     const int64_t* shift, int64_t c,
                                     double x, int64_t zp, int64_t lo,
                                     int64_t hi) {
    // (a bias past the limit is not part of x)
    const int64_t pre = pre_p ? pre_p[c] : 0;
    const int64_t lim = (int64_t)1 << BIAS_LIM_LOG2;
    const bool in = pre > -lim && pre < lim;
    return (int)qa_clip128(
        qa_mbqm_fast((int64_t)x + (in ? 0 : pre), mult[c], shift[c]) + zp, lo,
        hi);
}

// The residual Add and the rescaled copy of a table value past the float64
// forms' range, in 128 bits.
__device__ __noinline__ int bs_add_exact(int first, int second, int64_t za,
                                         int64_t ma, int64_t sa, int64_t zb,
                                         int64_t mb, int64_t sb, int64_t sign,
                                         int64_t zp, int64_t lo, int64_t hi) {
    return (int)qa_clip128(
        qa_mbqm_fast((int64_t)first - za, ma, sa) +
            (qa_i128)sign * qa_mbqm_fast((int64_t)second - zb, mb, sb) + zp,
        lo, hi);
}

__device__ __noinline__ int bs_copy_exact(int q, int64_t z, int64_t m,
                                          int64_t sh, int64_t zo, int64_t lo,
                                          int64_t hi) {
    return (int)qa_clip128(qa_mbqm_fast((int64_t)q - z, m, sh) + zo, lo, hi);
}

// D: K-steps in flight; a tile's steps are rounded up to whole turns of the
// ring with steps of zero activations (bs_depth picks D so that there are
// few), so that every load is unconditional and its wait exact.
// lutp: the table's LDS form is staged and read (a.plan).
template <int WM, int D, bool NARROW, bool RES, bool Y2>
__global__ __launch_bounds__(64 * BS_WAVES) void k_conv_bsl(ConvArgs a,
                                                            BsEpi e,
                                                            int lutp) {
    extern __shared__ int4 bs_dyn[];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15,
              kgl = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const XcdBlock blk = xcd_block(a.xcd_yfast != 0);
    const int g = (int)blk.z, co0 = (int)blk.y * (16 * WM);
    const int nsteps = a.KGp >> 2;
    // LDS: fragment (plane, block i, step s) of 1 KB at ((plane WM + i)
    // nsteps + s) KB; then the k-group table, then the channel constants
    int8_t* const s_w = (int8_t*)bs_dyn;
    int2* const s_kt = (int2*)(s_w + 2 * WM * nsteps * 1024);
    BsChan* const s_ch = (BsChan*)(s_kt + a.KGp);
    uint2* const s_lut = (uint2*)(s_ch + 16 * WM);

    {   // lane (row col, k-group kgl) of each fragment, straight into LDS
        const int8_t* src = a.ws + (int64_t)g * a.wp_gstride +
                            (int64_t)(co0 + col) * a.wp_rstride + 16 * kgl;
        const int64_t plane = (int64_t)a.G * a.wp_gstride;
        const int nf = 2 * WM * nsteps;
        for (int f = wave; f < nf; f += BS_WAVES) {
            const int pi = f / nsteps, s = f - pi * nsteps;
            const int8_t* p = src + (pi >= WM ? plane : 0) +
                              (int64_t)(pi >= WM ? pi - WM : pi) * 16 *
                                  a.wp_rstride +
                              64 * s;
            __builtin_amdgcn_global_load_lds(p, s_w + 1024 * f, 16, 0, 0);
        }
    }
    int4 lhead = int4{0, 0, -1, -1};
    if (lutp) {  // (the launcher found that many bytes readable there)
        const int8_t* src = (const int8_t*)a.plan + LUTP_HEAD;
        lhead = *(const int4*)a.plan;
        const int nc = (int)((a.lut_len + 15) / 16 + 1) / 2;  // of 16 bytes
        for (int c = tid; c < nc; c += 64 * BS_WAVES)
            ((int4*)s_lut)[c] = ((const int4*)src)[c];
        if (lhead.y != (LUTP_TAG | (int)a.lut_len)) lutp = 0;
    }
    // the element offset of a k-group's 16 channels from the tap's input
    // pixel (-1: no tap), its displacement dy << 16 | dx
    for (int kg = tid; kg < a.KGp; kg += 64 * BS_WAVES) {
        int2 t = {-1, 0};
        if (kg < a.KG) {
            const int tap = kg / a.CB, cb = kg - tap * a.CB;
            const int ky = tap / a.KW, kx = tap - ky * a.KW;
            t.x = (ky * a.DH * a.W + kx * a.DW) * (int)a.x_sp + 16 * cb;
            t.y = (ky * a.DH) << 16 | (kx * a.DW);
        }
        s_kt[kg] = t;
    }
    if (tid < 16 * WM) {
        const int c = min(co0 + tid, a.Cog - 1);
        const int64_t co = (int64_t)g * a.Cog + c;
        const int64_t pre = a.pre ? a.pre[co] : 0;
        const int64_t lim = (int64_t)1 << BIAS_LIM_LOG2;
        const bool in = pre > -lim && pre < lim;
        const MulD r = mul_d(a.mult[co], a.shift[co], 120);
        BsChan k;  // NaN: every value of the channel takes the 128-bit form
        k.mul = r.ok && in ? r.md : __builtin_nan("");
        k.add = (double)(a.ws_k[co] + (in ? pre : 0));
        s_ch[tid] = k;
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the direct loads landed
    __syncthreads();

    const int64_t ntiles = (a.M + 15) >> 4;
    const int64_t tstride = (int64_t)gridDim.x * BS_WAVES;
    int64_t tile = (int64_t)blk.x * BS_WAVES + wave;
    if (tile >= ntiles) return;
    // the stored zero point's bytes, as four copies
    const int pz = (int)(-a.x_add);
    const int ph = (int)(((uint32_t)(pz >> 8) & 255u) * 0x01010101u);
    const int pl = (int)((((uint32_t)pz & 255u) ^ 0x80u) * 0x01010101u);
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};

    constexpr int XW = NARROW ? 1 : 2;
    const int turns = (nsteps + D - 1) / D * D;
    PixPos fpos = pix_decode(a, tile * 16 + col);
    const int16_t* xb;
    int iy0, ix0, pb;
    auto origin = [&]() __attribute__((always_inline)) {
        const int n = fpos.n < a.N ? fpos.n : 0;  // past the end: image 0
        xb = (const int16_t*)a.x + (int64_t)n * a.x_sn + (int64_t)g * a.Cg;
        iy0 = fpos.oy * a.SH - a.PH;
        ix0 = fpos.ox * a.SW - a.PW;
        pb = (iy0 * a.W + ix0) * (int)a.x_sp;  // may be < 0
    };
    origin();
    int4 xr[D][XW];
    bool xin[D];
    auto fetch = [&](int4 (&x)[XW], bool& in, int s)
                     __attribute__((always_inline)) {
        const int2 t = s_kt[4 * min(s, nsteps - 1) + kgl];
        in = (t.x >= 0) &
             ((unsigned)(iy0 + (t.y >> 16)) < (unsigned)a.H) &
             ((unsigned)(ix0 + (t.y & 0xffff)) < (unsigned)a.W);
        // outside: the image's first pixel (in bounds, not used)
        const int16_t* p = xb + (in ? pb + t.x : 0);
        if constexpr (NARROW) {
            const int2 u = *(const int2*)p;
            x[0] = int4{u.x, u.y, 0, 0};
        } else {
            x[0] = *(const int4*)p;
            x[XW - 1] = *(const int4*)(p + 8);
        }
    };
    v4i hh[WM], md[WM], ll[WM], sh, sl;
    auto clear = [&]() __attribute__((always_inline)) {
        sh = sl = v4i{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < WM; ++i) hh[i] = md[i] = ll[i] = v4i{0, 0, 0, 0};
    };
    auto compute = [&](const int4 (&x)[XW], bool in, int s)
                       __attribute__((always_inline)) {
        // int16 channels 2j (low half) and 2j + 1 of dword j: the high
        // bytes are bytes 1 and 3 of each dword, the low bytes 0 and 2
        const int4 u = x[0], w = NARROW ? int4{0, 0, 0, 0} : x[XW - 1];
        v4i xh = {(int)__builtin_amdgcn_perm(u.y, u.x, 0x07050301u),
                  (int)__builtin_amdgcn_perm(u.w, u.z, 0x07050301u),
                  (int)__builtin_amdgcn_perm(w.y, w.x, 0x07050301u),
                  (int)__builtin_amdgcn_perm(w.w, w.z, 0x07050301u)};
        v4i xl = {(int)__builtin_amdgcn_perm(u.y, u.x, 0x06040200u),
                  (int)__builtin_amdgcn_perm(u.w, u.z, 0x06040200u),
                  (int)__builtin_amdgcn_perm(w.y, w.x, 0x06040200u),
                  (int)__builtin_amdgcn_perm(w.w, w.z, 0x06040200u)};
        xl ^= (int)0x80808080u;
        // (a rounding step's x is 0 in every product and sum)
        const bool real = s < nsteps;
        const int vh = real ? ph : 0, vl = real ? pl : 0;
        if (!(in & real)) {
            xh = v4i{vh, vh, vh, vh};
            xl = v4i{vl, vl, vl, vl};
        }
        const int8_t* f = s_w + 1024 * min(s, nsteps - 1) + 16 * lane;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const v4i wh = *(const v4i*)(f + 1024 * i * nsteps);
            const v4i wl = *(const v4i*)(f + 1024 * (WM + i) * nsteps);
            hh[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, xh, hh[i], 0, 0,
                                                          0);
            md[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, xh, md[i], 0, 0,
                                                          0);
            md[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wh, xl, md[i], 0, 0,
                                                          0);
            ll[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wl, xl, ll[i], 0, 0,
                                                          0);
        }
        sh = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xh, sh, 0, 0, 0);
        sl = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xl, sl, 0, 0, 0);
    };
    const int lmax = (int)a.lut_len - 1, loff = (int)a.lut_off;
    auto finish = [&]() __attribute__((always_inline)) {
        const int64_t p = tile * 16 + col;
        const bool pok = p < a.M;
        const int64_t pc = pok ? p : a.M - 1;
        // 128 U of the lane's pixel (every row of sh / sl holds it)
        const double u = 128.0 * fma((double)sh[0], 256.0, (double)sl[0]);
        int q[WM][4];
        int2 rv[RES ? WM : 1];
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const int cb = co0 + 16 * i + 4 * kgl;  // within the group
            const int64_t co = (int64_t)g * a.Cog + cb;
            if constexpr (RES) {
                const int16_t* r =
                    (const int16_t*)a.res + pc * a.res_pst + co;
                if (cb + 3 < a.Cog) {
                    rv[i] = *(const int2*)r;
                } else {
                    uint32_t w[2] = {0, 0};
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (cb + k < a.Cog)
                            w[k / 2] |= (uint32_t)(uint16_t)r[k]
                                        << (16 * (k & 1));
                    rv[i] = int2{(int)w[0], (int)w[1]};
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const BsChan k = s_ch[16 * i + 4 * kgl + r];
                // the exact sum, below 2^53: every step is exact
                const double x =
                    fma((double)hh[i][r], 65536.0,
                        fma((double)md[i][r], 256.0, (double)ll[i][r]) +
                            (u + k.add));
                const double y = fma(x, k.mul, e.c0);
                const double f = floor(y);
                const double fr = y - f;
                q[i][r] = (int)fmin(fmax(f, e.qlo), e.qhi);
                if (__builtin_expect(!(fr >= 0x1p-30 && fr <= 1.0 - 0x1p-30) &&
                                         !(fabs(y) >= 0x1p20),
                                     0))  // (also for a NaN)
                    q[i][r] = bs_exact(
                        a.pre, a.mult, a.shift,
                        (int64_t)g * a.Cog + min(cb + r, a.Cog - 1), x, a.zp,
                        a.qmin, a.qmax);
            }
        }
        if (lutp) {
            int ix[WM][4];
            bool odd = false;
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    ix[i][r] = min(max(q[i][r] - loff, 0), lmax);
                    q[i][r] = lutp_get(s_lut, lhead.x, ix[i][r]);
                    odd |= (ix[i][r] >> 4) == lhead.z;
                    odd |= (ix[i][r] >> 4) == lhead.w;
                }
            if (__builtin_expect(odd, 0)) {
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) q[i][r] = a.lut[ix[i][r]];
            }
        } else if (a.lut) {  // every table read of the lane in flight
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    q[i][r] = a.lut[min(max(q[i][r] - loff, 0), lmax)];
        }
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            const int cb = co0 + 16 * i + 4 * kgl;
            const int64_t co = (int64_t)g * a.Cog + cb;
            uint32_t wy[2] = {0, 0}, w2[2] = {0, 0};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int qv = q[i][r];
                if constexpr (RES) {
                    const uint32_t rw =
                        (uint32_t)(r < 2 ? rv[i].x : rv[i].y);
                    const int rs = (int)(int16_t)(rw >> (16 * (r & 1)));
                    if (__builtin_expect((unsigned)(qv + (1 << 19)) <
                                             (1u << 20),
                                         1)) {
                        const double v = (double)qv;
                        const double rd = (double)rs + e.rso;
                        const double first = a.res_first ? rd : v;
                        const double second = a.res_first ? v : rd;
                        const double t =
                            round_d(first - e.za, e.ra) +
                            e.asgn * round_d(second - e.zb, e.rb) + e.azp;
                        qv = (int)fmin(fmax(t, e.alo), e.ahi);
                    } else {
                        const int rq = rs + (int)a.res_so;
                        qv = bs_add_exact(a.res_first ? rq : qv,
                                          a.res_first ? qv : rq, a.za, a.ma,
                                          a.sa, a.zb, a.mb, a.sb, a.add_sign,
                                          a.add_zp, a.add_qmin, a.add_qmax);
                    }
                }
                wy[r / 2] |= ((uint32_t)(qv - (int)a.y_so) & 0xffffu)
                             << (16 * (r & 1));
                if constexpr (Y2) {
                    int c;
                    if (__builtin_expect((unsigned)(qv + (1 << 19)) <
                                             (1u << 20),
                                         1))
                        c = (int)fmin(
                            fmax(round_d((double)qv - e.z2, e.r2) + e.zo2,
                                 e.lo2),
                            e.hi2);
                    else
                        c = bs_copy_exact(qv, a.r2_zp_in, a.r2_m, a.r2_s,
                                          a.r2_zp_out, a.r2_qmin, a.r2_qmax);
                    w2[r / 2] |= ((uint32_t)(c - (int)a.y_so) & 0xffffu)
                                 << (16 * (r & 1));
                }
            }
            if (!pok) continue;
            auto put = [&](int16_t* d, const uint32_t* w)
                           __attribute__((always_inline)) {
                if (cb + 3 < a.Cog) {
                    *(int2*)d = int2{(int)w[0], (int)w[1]};
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (cb + k < a.Cog)
                            d[k] = (int16_t)(w[k / 2] >> (16 * (k & 1)));
                }
            };
            put((int16_t*)a.y + p * a.y_pst + co, wy);
            if constexpr (Y2) put((int16_t*)a.y2 + p * a.y2_pst + co, w2);
        }
    };
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(xr[d], xin[d], d);
    while (true) {
        clear();
        int c = 0;
        for (; c + D < turns; c += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                compute(xr[d], xin[d], c + d);
                fetch(xr[d], xin[d], c + d + D);
            }
        }
        // the tile's last turn: its slots refill from the wave's next tile
        // (past the last tile: image 0, in bounds, not used)
        pix_step(a, fpos);
        origin();
#pragma unroll
        for (int d = 0; d < D; ++d) {
            compute(xr[d], xin[d], c + d);
            fetch(xr[d], xin[d], d);
        }
        finish();
        tile += tstride;
        if (tile >= ntiles) return;
    }
}

// K-steps in flight: as many as divide the tile's steps, or 3.
int bs_depth(int nsteps) {
    return nsteps % 4 == 0 ? 4
           : nsteps % 3 == 0 ? 3
           : nsteps <= 2 ? nsteps
           : nsteps % 2 == 0 && nsteps < 14 ? 2
                                            : 3;
}

bool exact_mul(int64_t m, int64_t shift) {  // mul_d's range with tmax 53
    const int64_t ts = 31 + shift;
    return ts >= 1 && ts <= 53 && m > -((int64_t)1 << 31) &&
           m < ((int64_t)1 << 31);
}

// Whether the bytes at p, wherever a caller's plan came from, lie in one
// device allocation (a lookup in the runtime's map; memory it does not know
// is left alone). The kernel requests them together with the header that
// says whether they are a plan: a wait for it first costs 0.45 us a launch.
bool readable(const void* p, int64_t bytes) {
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) !=
        hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return (uintptr_t)p + bytes <= (uintptr_t)base + size;
}

double host_mul(int64_t m, int64_t shift) {
    return ldexp((double)m, -(int)(31 + shift));
}

}  // namespace

int64_t bsl_lds(const ConvArgs& b, int wm) {
    return (int64_t)2 * wm * (b.KGp / 4) * 1024 + b.KGp * 8 +
           16 * wm * (int64_t)sizeof(BsChan);
}

// int16 outputs, dense in 8-byte aligned 4-channel words, every scalar
// multiply of the epilogue inside its float64 form's range, and 16 channels'
// weights within LDS (K up to about 4,800 positions).
bool conv_bsl_applies(const ConvArgs& b) {
    const int64_t B19 = (int64_t)1 << 19;
    auto words = [&](const void* p, int64_t pst) {
        return !p || ((uintptr_t)p % 8 == 0 && pst % 4 == 0);
    };
    auto small = [&](int64_t v) { return v > -B19 && v < B19; };
    if (!(b.mode == EPI_QUANT && b.fastio && b.y_code == 2 && b.wide &&
          (b.G == 1 || b.Cog % 4 == 0) && words(b.y, b.y_pst) &&
          words(b.res, b.res_pst) && words(b.y2, b.y2_pst) &&
          small(b.qmin) && small(b.qmax) && b.qmin <= b.qmax &&
          small(b.zp) && small(b.y_so)))
        return false;
    if (b.lut &&
        !(b.lut_len > 0 && b.lut_len < (1 << 30) && small(b.lut_off)))
        return false;
    if (b.res && !(exact_mul(b.ma, b.sa) && exact_mul(b.mb, b.sb) &&
                   (b.add_sign == 1 || b.add_sign == -1) && small(b.za) &&
                   small(b.zb) && small(b.res_so) && small(b.add_zp) &&
                   small(b.add_qmin) && small(b.add_qmax) &&
                   b.add_qmin <= b.add_qmax))
        return false;
    if (b.y2 && !(exact_mul(b.r2_m, b.r2_s) && small(b.r2_zp_in) &&
                  small(b.r2_zp_out) && small(b.r2_qmin) &&
                  small(b.r2_qmax) && b.r2_qmin <= b.r2_qmax))
        return false;
    return ceil_div(b.Cog, 16) <= 65535 && b.G <= 65535 &&
           bsl_lds(b, 1) <= BSL_LDS_MAX;
}

bool launch_conv_bsl(const ConvArgs& b0, bool narrow, int wm,
                     hipStream_t st) {
    ConvArgs b = b0;
    const int64_t ntiles = ceil_div(b.M, 16);
    const int cus = cu_count();
    if (narrow) wm = 1;
    // the widest block (each activation fragment is split and read once a
    // block) that fits LDS and still gives every CU a work-group
    if (wm == 0) {
        wm = b.Cog > 32 ? 4 : b.Cog > 16 ? 2 : 1;
        while (wm > 1 && ceil_div(ntiles, BS_WAVES) *
                                 ceil_div(b.Cog, 16 * wm) * b.G <
                             cus)
            wm /= 2;
    }
    while (wm > 1 && bsl_lds(b, wm) > BSL_LDS_MAX) wm /= 2;
    int64_t lds = bsl_lds(b, wm);
    const int64_t gy = ceil_div(b.Cog, 16 * wm);
    BsEpi e;
    memset(&e, 0, sizeof(e));
    e.c0 = 0.5 + (double)b.zp;
    e.qlo = (double)b.qmin;
    e.qhi = (double)b.qmax;
    if (b.res) {
        e.ra = host_mul(b.ma, b.sa);
        e.rb = host_mul(b.mb, b.sb);
        e.za = (double)b.za;
        e.zb = (double)b.zb;
        e.asgn = (double)b.add_sign;
        e.azp = (double)b.add_zp;
        e.alo = (double)b.add_qmin;
        e.ahi = (double)b.add_qmax;
        e.rso = (double)b.res_so;
    }
    if (b.y2) {
        e.r2 = host_mul(b.r2_m, b.r2_s);
        e.z2 = (double)b.r2_zp_in;
        e.zo2 = (double)b.r2_zp_out;
        e.lo2 = (double)b.r2_qmin;
        e.hi2 = (double)b.r2_qmax;
    }
    // The table's LDS form: a 64-lane read of the 256 KB table takes the
    // L1 about 64 cycles (a line a lane), its LDS form about 16, for a
    // staging of up to 32 KB a work-group: worth it past about 4,000 values
    // a work-group (the YOLOv8n-cls layers up to 14x14).
    const int64_t nwg = std::min<int64_t>(
        ceil_div(ntiles, BS_WAVES) * gy * b.G, 2 * (int64_t)cus);
    const int64_t lutb = round_up(ceil_div(b.lut_len, 16) * 8, 16);
    const bool lutp = b.lut && b.plan && (uintptr_t)b.plan % 16 == 0 &&
                      b.lut_len <= 65536 && lds + lutb <= BSL_LDS_MAX &&
                      b.M * b.Cout >= 4096 * nwg &&
                      readable(b.plan, LUTP_HEAD + lutb);
    if (lutp) lds += lutb;
    // (see launch_kernel of the int8 form)
    b.xcd_yfast = 2 * (int64_t)b.N * b.H * b.W * b.Cg * b.G >=
                  2 * (int64_t)b.Cout * b.KGp * 16;
    auto run = [&](auto* k) {
        // as many work-groups as are resident, each walking its share
        const int64_t nres =
            resident_blocks((const void*)k, 64 * BS_WAVES, (int)lds);
        const int64_t cap = std::max<int64_t>(1, nres * cus / (gy * b.G));
        const int64_t gx = std::min(ceil_div(ntiles, BS_WAVES), cap);
        const int64_t stride = 16 * gx * BS_WAVES;
        const int64_t ohw = (int64_t)b.OH * b.OW;
        b.st_dn = (int32_t)(stride / ohw);
        b.st_doy = (int32_t)((stride % ohw) / b.OW);
        b.st_dox = (int32_t)((stride % ohw) % b.OW);
        k<<<dim3((unsigned)gx, (unsigned)gy, (unsigned)b.G), 64 * BS_WAVES,
            (size_t)lds, st>>>(b, e, lutp ? 1 : 0);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            set_hip_error("k_conv_bsl", err);
            return false;
        }
        return true;
    };
    auto forms = [&](auto w, auto dd, auto nr) {
        constexpr int W = decltype(w)::value, D = decltype(dd)::value;
        constexpr bool NR = decltype(nr)::value;
        if (b.res && b.y2) return run(&k_conv_bsl<W, D, NR, true, true>);
        if (b.res) return run(&k_conv_bsl<W, D, NR, true, false>);
        if (b.y2) return run(&k_conv_bsl<W, D, NR, false, true>);
        return run(&k_conv_bsl<W, D, NR, false, false>);
    };
    using std::integral_constant;
    auto depth = [&](auto w, auto nr) {
        switch (bs_depth(b.KGp / 4)) {
            case 1: return forms(w, integral_constant<int, 1>{}, nr);
            case 2: return forms(w, integral_constant<int, 2>{}, nr);
            case 3: return forms(w, integral_constant<int, 3>{}, nr);
            default: return forms(w, integral_constant<int, 4>{}, nr);
        }
    };
    if (narrow) return depth(integral_constant<int, 1>{}, std::true_type{});
    switch (wm) {
        case 1: return depth(integral_constant<int, 1>{}, std::false_type{});
        case 2: return depth(integral_constant<int, 2>{}, std::false_type{});
        default: return depth(integral_constant<int, 4>{}, std::false_type{});
    }
}

}  // namespace qa

using namespace qa;

QA_API int64_t qa_lut_i16_plan_bytes(int64_t lut_len) {
    if (lut_len < 1 || lut_len > 65536) return -1;
    return LUTP_HEAD + round_up(ceil_div(lut_len, 16) * 8, 16);
}

QA_API int qa_plan_lut_i16(const int32_t* lut, int64_t lut_len, void* plan) {
    const int64_t bytes = qa_lut_i16_plan_bytes(lut_len);
    if (!lut || !plan || bytes < 0) return -1;
    const auto mm = std::minmax_element(lut, lut + lut_len);
    const int64_t base = *mm.first;
    if ((int64_t)*mm.second - base > 65535) return 0;
    memset(plan, 0, (size_t)bytes);
    int32_t* head = (int32_t*)plan;
    head[0] = (int32_t)base;
    head[1] = LUTP_TAG | (int32_t)lut_len;
    head[2] = head[3] = -1;
    uint32_t* out = (uint32_t*)((char*)plan + LUTP_HEAD);
    int odd = 0;
    for (int64_t i = 0; i < lut_len; i += 16) {
        const int64_t k0 = lut[i] - base;
        const int64_t k1 = lut[std::min(i + 16, lut_len - 1)] - base;
        uint32_t bits = 0;
        bool fits = true;
        for (int64_t f = 0; f < 16 && i + f < lut_len; ++f) {
            const int64_t line = k0 + (((k1 - k0) * f + 8) >> 4);
            const int64_t r = lut[i + f] - base - line + 2;
            fits = fits && r >= 0 && r <= 3;
            bits |= (uint32_t)(r & 3) << (2 * f);
        }
        if (!fits) {
            if (odd == 2) return 0;
            head[2 + odd++] = (int32_t)(i / 16);
        }
        out[i / 8] = (uint32_t)(k0 | k1 << 16);
        out[i / 8 + 1] = bits;
    }
    return 1;
}
