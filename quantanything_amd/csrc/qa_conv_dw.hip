// Depthwise int8 convolutions (one input and one output channel a group) on
// the int8 matrix cores.
//
// A depthwise convolution is bound by its bytes (a read and a write a
// channel, KH*KW multiply-adds between them); a lane a channel with its own
// loads, unpacking and 64-bit multiplies is bound by instructions instead
// (32x128x56x56, 3x3: 479 us). Here 16 channels x 16 output pixels are one
// tile: v_mfma_i32_16x16x64_i8 takes 4 taps a step, its 64-byte K the 16
// channels of each, against weights that are zero off the diagonal, so a
// tile of a 3x3 kernel is three MFMAs, each lane's operand one 16-byte load
// of a tap's pixel (neighbouring taps and pixels meet in L1). The weights
// are the first operand: a lane holds one byte of its channel's row a step,
// expanded in registers, and ends with 4 consecutive channels of one pixel,
// which the table epilogue stores as one word. The 4 waves of a work-group
// take consecutive channel blocks of the same pixels (the pieces of one
// cache line), each wave a contiguous run of tiles with the next tile's
// loads in flight, and work-groups of one XCD consecutive runs (the rows of
// a window meet in its L2). The same layer: 24 us, its 150 thousand 64-line loads the bound.
//
// Weights: layout 2 of qa_pack_weights_i8 (a row of KH*KW bytes a channel,
// padded to 16; rows padded to 16).
#include <algorithm>

#include "qa_conv_mfma.h"

namespace qa {
namespace {

// S: steps of 4 taps; EPI: Q8_TABLE or Q8_GENERAL; RES / Y2: residual Add
// and rescaled copy of the table epilogue; RS: weights with an offset (8-bit
// types whose centred weights pass int8), which multiplies the sum of the
// channel's window, a second product against a diagonal of ones.
template <int S, int EPI, bool RES, bool Y2, bool RS>
__global__ __launch_bounds__(256) void k_conv_dw(ConvArgs a, int nch,
                                                 int per_wave) {
    constexpr bool TABLE = EPI == Q8_TABLE;
    __shared__ int s_tab[TABLE ? 768 : 1];
    const int lane = threadIdx.x & 63, col = lane & 15, kg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // contiguous work-groups on one XCD (see xcd_block)
    const uint32_t f = blockIdx.x, q8 = gridDim.x >> 3, r8 = gridDim.x & 7;
    const uint32_t xcd = f & 7;
    const int64_t wid =
        (int64_t)(xcd * q8 + min(xcd, r8) + (f >> 3)) * 4 + wave;
    const int chunk = (int)(wid % nch);
    const int64_t ntiles = (a.M + 15) >> 4;
    int64_t tile = wid / nch * per_wave;
    const int64_t tend = min(tile + per_wave, ntiles);
    const int ch = chunk * 16;

    // the lane's weight byte a step (row ch + col, tap 4 s + kg), in its
    // position of the diagonal
    const int8_t* wr = a.wp + (int64_t)(ch + col) * a.wp_rstride;
    const int taps = a.KH * a.KW;
    v4i wf[S], of[RS ? S : 1];
    int off[S], dydx[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int tap = 4 * s + kg;
        const bool real = tap < taps;
        const int b = real ? (int)(uint8_t)wr[real ? tap : 0]
                                 << (8 * (col & 3))
                           : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            wf[s][k] = (col >> 2) == k ? b : 0;
            if (RS)
                of[s][k] = real && (col >> 2) == k ? 1 << (8 * (col & 3)) : 0;
        }
        const int ky = real ? tap / a.KW : 0;
        const int kx = real ? tap - ky * a.KW : 0;
        const int dy = ky * a.DH, dx = kx * a.DW;
        dydx[s] = dy | dx << 16;
        off[s] = (dy * a.W + dx) * (int)a.x_sp;  // < 2^31 (dw_applies)
    }
    if (TABLE) {
        const int* tab = (const int*)((const char*)a.plan + PLAN_E);
#pragma unroll
        for (int j = 0; j < (RES ? 3 : 1); ++j)
            s_tab[threadIdx.x + 256 * j] = tab[threadIdx.x + 256 * j];
    }
    // the lane's 4 channels' constants
    const int cl = ch + 4 * kg;
    int cm[4] = {0}, ct[4] = {0}, cbo[4] = {0};
    int64_t cc[4] = {0};
    int pA = 0, pB = 0, pSH = 0;
    if (TABLE) {
        const int4 h = *(const int4*)a.plan;
        pA = h.x;
        pB = h.y;
        pSH = h.z;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = min(cl + r, a.Cout - 1);
            const int4 pc = ((const int4*)((const char*)a.plan + PLAN_CH))[c];
            cm[r] = pc.x;
            ct[r] = pc.y;
            cc[r] = plan_fold(
                (int64_t)(((uint64_t)(uint32_t)pc.w << 32) | (uint32_t)pc.z),
                a.corr ? (uint32_t)a.corr[c] : 0u, pc.x);
            if (RS) cbo[r] = a.boff[c];
        }
    }
    __syncthreads();
    if (tile >= tend) return;
    const int pv = splat4(a.pad_value);

    // fetch of one tile: S loads, from addresses inside the image; bit s of
    // *out: the tap lies outside
    PixPos pos = pix_decode(a, tile * 16 + col);
    auto fetch = [&](v4i* b, int* out) __attribute__((always_inline)) {
        const int n = pos.n < a.N ? pos.n : 0;  // past the end: image 0
        const int iy0 = pos.oy * a.SH - a.PH, ix0 = pos.ox * a.SW - a.PW;
        const int8_t* img = (const int8_t*)a.x + (int64_t)n * a.x_sn + ch;
        const int org = (iy0 * a.W + ix0) * (int)a.x_sp;
        *out = 0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const bool in =
                (unsigned)(iy0 + (dydx[s] & 0xffff)) < (unsigned)a.H &&
                (unsigned)(ix0 + (dydx[s] >> 16)) < (unsigned)a.W;
            if (!in) *out |= 1 << s;
            b[s] = *(const v4i*)(img + (in ? org + off[s] : 0));
        }
        pix_step(a, pos);
    };
    auto finish = [&](const v4i* b, int out) __attribute__((always_inline)) {
        const int64_t p = tile * 16 + col;
        const bool pok = p < a.M;
        uint32_t rv = 0;
        if (RES && pok) {
            const int8_t* pr = (const int8_t*)a.res + p * a.res_pst + cl;
            if (cl + 3 < a.Cout) {
                rv = *(const uint32_t*)pr;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (cl + r < a.Cout)
                        rv |= (uint32_t)(uint8_t)pr[r] << (8 * r);
            }
        }
        v4i acc{0, 0, 0, 0}, sum{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const v4i x = apply_pad<0>(b[s], out >> s & 1, pv);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[s], x, acc, 0, 0,
                                                        0);
            if (RS)
                sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(of[RS ? s : 0], x,
                                                            sum, 0, 0, 0);
        }
        if (!TABLE) {
            if (pok) {
#pragma unroll 1
                for (int r = 0; r < 4; ++r) {
                    const int v = r == 0   ? acc[0]
                                  : r == 1 ? acc[1]
                                  : r == 2 ? acc[2]
                                           : acc[3];
                    const int w = r == 0   ? sum[0]
                                  : r == 1 ? sum[1]
                                  : r == 2 ? sum[2]
                                           : sum[3];
                    if (cl + r < a.Cout)
                        store_general<EPI>(a, v, p, cl + r, w);
                }
            }
            return;
        }
        int e[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int w = RS ? acc[r] + cbo[r] * sum[r] : acc[r];
            const int i =
                med3_i32(plan_q0(w, cm[r], cc[r], ct[r]), pA, pB) - pA;
            if (RES) {
                const int t =
                    s_tab[256 + i] + s_tab[512 + ((rv >> (8 * r)) & 255)];
                e[r] = s_tab[med3_i32(t, 0, pSH)];
            } else {
                e[r] = s_tab[i];
            }
        }
        if (!pok) return;
        auto put = [&](int8_t* d, uint32_t w) __attribute__((always_inline)) {
            if (cl + 3 < a.Cout) {
                *(uint32_t*)d = w;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (cl + r < a.Cout) d[r] = (int8_t)(w >> (8 * r));
            }
        };
        put((int8_t*)a.y + p * a.y_pst + cl, pack_entries(e, 0));
        if (Y2)
            put((int8_t*)a.y2 + p * a.y2_pst + cl, pack_entries(e, 1));
    };
    v4i b0[S], b1[S];
    int o0, o1;
    fetch(b0, &o0);
    while (true) {
        if (tile + 1 < tend) fetch(b1, &o1);
        finish(b0, o0);
        if (++tile >= tend) return;
        if (tile + 1 < tend) fetch(b0, &o0);
        finish(b1, o1);
        if (++tile >= tend) return;
    }
}

}  // namespace

// Whether the depthwise kernel takes a layout-2 descriptor: up to 52 taps
// (the fragments are registers), 32-bit offsets inside an image.
bool conv_dw_applies(const ConvArgs& b) {
    return b.layout == 2 && b.Cg == 1 && b.Cog == 1 && b.G == b.Cout &&
           b.KH * (int64_t)b.KW <= 52 && b.x_code == 1 &&
           b.x_sc == 1 && (uintptr_t)b.x % 16 == 0 && b.x_sn % 16 == 0 &&
           b.x_sp % 16 == 0 && b.x_sp >= round_up(b.Cout, 16) &&
           (int64_t)(b.KH - 1) * b.DH < 32768 &&
           (int64_t)(b.KW - 1) * b.DW < 32768 &&
           ((int64_t)b.H + b.PH + b.KH * (int64_t)b.DH) *
                   ((int64_t)b.W + b.PW + b.KW * (int64_t)b.DW) * b.x_sp <
               ((int64_t)1 << 30) &&
           b.M < ((int64_t)1 << 31);
}

bool launch_conv_dw(const ConvArgs& a0, int epi, hipStream_t st) {
    ConvArgs a = a0;
    if (!conv_dw_applies(a) || (epi != Q8_TABLE && epi != Q8_GENERAL)) {
        set_error("launch_conv_dw", "depthwise convolution out of scope");
        return false;
    }
    const int nch = (int)ceil_div(a.Cout, 16);
    const int64_t ntiles = ceil_div(a.M, 16);
    // 16 waves a CU, each a run of tiles; single tiles when there are fewer
    const int64_t runs =
        std::max<int64_t>(1, (int64_t)cu_count() * 16 / nch);
    const int64_t per = ceil_div(ntiles, std::min(ntiles, runs));
    const int64_t waves = ceil_div(ntiles, per) * nch;
    // the next tile: 16 pixels on
    const int64_t ohw = (int64_t)a.OH * a.OW;
    a.st_dn = (int32_t)(16 / ohw);
    a.st_doy = (int32_t)((16 % ohw) / a.OW);
    a.st_dox = (int32_t)((16 % ohw) % a.OW);
    const dim3 grid((unsigned)ceil_div(waves, 4));
    auto launch = [&](auto steps, auto epic, auto res, auto y2, auto rs) {
        k_conv_dw<decltype(steps)::value, decltype(epic)::value,
                  decltype(res)::value, decltype(y2)::value,
                  decltype(rs)::value><<<grid, 256, 0, st>>>(a, nch, (int)per);
    };
    using T = std::true_type;
    using F = std::false_type;
    using TAB = std::integral_constant<int, Q8_TABLE>;
    using GEN = std::integral_constant<int, Q8_GENERAL>;
    auto go = [&](auto steps) {
        const int key = (a.res ? 4 : 0) | (a.y2 ? 2 : 0) | (a.rowsum ? 1 : 0);
        if (epi != Q8_TABLE) {
            a.rowsum ? launch(steps, GEN{}, F{}, F{}, T{})
                     : launch(steps, GEN{}, F{}, F{}, F{});
            return;
        }
        switch (key) {
            case 0: launch(steps, TAB{}, F{}, F{}, F{}); break;
            case 1: launch(steps, TAB{}, F{}, F{}, T{}); break;
            case 2: launch(steps, TAB{}, F{}, T{}, F{}); break;
            case 3: launch(steps, TAB{}, F{}, T{}, T{}); break;
            case 4: launch(steps, TAB{}, T{}, F{}, F{}); break;
            case 5: launch(steps, TAB{}, T{}, F{}, T{}); break;
            case 6: launch(steps, TAB{}, T{}, T{}, F{}); break;
            default: launch(steps, TAB{}, T{}, T{}, T{}); break;
        }
    };
    const int taps = a.KH * a.KW;
    if (taps <= 4)
        go(std::integral_constant<int, 1>{});
    else if (taps <= 12)
        go(std::integral_constant<int, 3>{});
    else if (taps <= 28)
        go(std::integral_constant<int, 7>{});
    else
        go(std::integral_constant<int, 13>{});
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_hip_error("k_conv_dw", e);
        return false;
    }
    return true;
}

}  // namespace qa
