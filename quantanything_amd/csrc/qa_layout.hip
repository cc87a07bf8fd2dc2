// Float32 NCHW on one side, quantized channels-last on the other: a graph
// input of more than 4 channels (or of 16-bit storage) quantized into the
// layout the convolutions read, and a channels-last graph output
// dequantized into the caller's NCHW floats.
//
// Both move 5 or 6 bytes a value and are bound by HBM, so they are shaped by
// their transactions: a work-group takes a tile of consecutive pixels (of
// all images in a row) and transposes it through 4 - 5 KB of LDS, so that
// the float side is read or written in runs of 256 bytes to 1 KB of a plane
// and the channels-last side in 16-byte chunks, consecutive lanes on
// consecutive chunks; every load of a thread is issued before its first
// use. 32x64x56x56 int8, 32 MB: 5.2 us in and 5.9 us out (6.2 and 5.4
// TB/s); a thread per pixel walking its channels one load at a time took
// 36.8 us in, a strided copy to NCHW and a second dequantizing launch 43.5
// us out; chunks of 4 pixels x 16 channels a thread without LDS 6.9 and
// 19.1 us (the 16-byte pieces of a line come from different waves).
#include <algorithm>
#include <type_traits>

#include "../../include/qa_hip.h"
#include "qa_common.h"

namespace qa {
namespace {

constexpr int kThreads = 256;

struct QuantTo {
    double scale, inv;
    float invf, invlo;
    int32_t f32ok;
    int64_t zp, qmin, qmax, so;
};

// q - so of one value; *slow as qa_quantize_f32x2 sets it.
__device__ __forceinline__ int quant_f32(const QuantTo& o, float f,
                                         bool* slow) {
    return qa_quantize_f32x2(f, o.invf, o.invlo, (int)o.zp, (int)o.qmin,
                             (int)o.qmax, slow) -
           (int)o.so;
}

__device__ __forceinline__ int quant_f64(const QuantTo& o, float f) {
    return (int)(qa_quantize_one_fast(f, o.scale, o.inv, o.zp, o.qmin,
                                      o.qmax) -
                 o.so);
}

// x float32 [N, C, HW] -> y [N * HW] pixels of y_sp elements (a multiple of
// 16 bytes), 0 in the channels C .. y_sp. A tile is 4096 / RB pixels x RB
// bytes of channels; a thread quantizes the 16 bytes of one pixel.
template <class T, int RB>
__global__ __launch_bounds__(kThreads) void k_quantize_tile(
    const float* __restrict__ x, int C, uint32_t HW, uint32_t pixels,
    T* __restrict__ y, int y_sp, QuantTo o) {
    constexpr int PX = 4096 / RB, CH = 16 / sizeof(T), CPR = RB / 16;
    constexpr int RS = RB / 4 + 1;  // LDS words a pixel: odd, so that lanes
                                    // on consecutive pixels spread over banks
    __shared__ uint32_t t[PX * RS];
    const int tid = threadIdx.x;
    const uint32_t p0 = blockIdx.x * PX;
    const int c0 = blockIdx.y * (int)(RB / sizeof(T));
    const int px = tid % PX, chunk = tid / PX;  // chunk: wave-uniform
    const int cb = c0 + chunk * CH;
    uint32_t w[4] = {0, 0, 0, 0};
    if (cb < C) {
        const uint32_t p = min(p0 + px, pixels - 1);
        const uint32_t n = p / HW;
        const float* s =
            x + ((int64_t)n * C + cb) * (int64_t)HW + (p - n * HW);
        const int last = min(CH - 1, C - 1 - cb);
        float f[CH];
#pragma unroll
        for (int k = 0; k < CH; ++k)  // (past C: the last plane, dropped)
            f[k] = s[(int64_t)min(k, last) * (int64_t)HW];
        constexpr int PW = 4 / sizeof(T);  // values a word
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            bool slow = !o.f32ok;
            int q[PW];
#pragma unroll
            for (int k = 0; k < PW; ++k)
                q[k] = quant_f32(o, f[PW * g + k], &slow);
            if (__builtin_expect(slow, 0)) {
#pragma unroll
                for (int k = 0; k < PW; ++k)
                    q[k] = quant_f64(o, f[PW * g + k]);
            }
#pragma unroll
            for (int k = 0; k < PW; ++k) {
                const uint32_t b =
                    (uint32_t)q[k] & (sizeof(T) == 1 ? 0xffu : 0xffffu);
                if (PW * g + k <= last) w[g] |= b << (8 * sizeof(T) * k);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) t[px * RS + 4 * chunk + k] = w[k];
    __syncthreads();
    const int sp = tid / CPR, sc = tid % CPR;  // the chunk this lane stores
    if (p0 + sp < pixels && c0 + sc * CH < y_sp) {
        const uint32_t* r = t + sp * RS + 4 * sc;
        *(uint4*)(y + (int64_t)(p0 + sp) * y_sp + c0 + sc * CH) =
            make_uint4(r[0], r[1], r[2], r[3]);
    }
}

// Any pixel stride or alignment: a thread quantizes PX pixels (4: the planes
// as float4, 4-channel pixels of 8 bytes) of CH channels.
template <class T, int CH, int PX>
__global__ __launch_bounds__(kThreads) void k_quantize_any(
    const float* __restrict__ x, int64_t C, int64_t HW, int64_t groups,
    int64_t nch, T* __restrict__ y, int64_t y_sp, QuantTo o) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
         i < groups * nch; i += (int64_t)gridDim.x * kThreads) {
        const int64_t chunk = i / groups;  // pixels fastest
        const int64_t p0 = (i - chunk * groups) * PX;
        const int64_t n = p0 / HW, p = p0 - n * HW, c0 = chunk * CH;
        float f[CH][PX];
#pragma unroll
        for (int k = 0; k < CH; ++k) {
            const float* s = x + (n * C + min(c0 + k, C - 1)) * HW + p;
            if (c0 + k >= C) continue;
            if constexpr (PX == 4) {
                const float4 v = *(const float4*)s;
                f[k][0] = v.x;
                f[k][1] = v.y;
                f[k][2] = v.z;
                f[k][3] = v.w;
            } else {
                f[k][0] = *s;
            }
        }
        T q[PX][CH];
#pragma unroll
        for (int j = 0; j < PX; ++j)
#pragma unroll
            for (int k = 0; k < CH; ++k) {
                q[j][k] = (T)0;
                if (c0 + k >= C) continue;
                bool slow = !o.f32ok;
                int v = quant_f32(o, f[k][j], &slow);
                if (__builtin_expect(slow, 0)) v = quant_f64(o, f[k][j]);
                q[j][k] = (T)v;
            }
        T* d = y + (n * HW + p) * y_sp + c0;
        if constexpr (PX == 4) {  // y_sp == CH: the pixels are contiguous
            typedef T vt __attribute__((ext_vector_type(2 * CH)));
#pragma unroll
            for (int j = 0; j < PX; j += 2) {
                vt v;
#pragma unroll
                for (int k = 0; k < 2 * CH; ++k) v[k] = q[j + k / CH][k % CH];
                *(vt*)(d + j * CH) = v;
            }
        } else {
#pragma unroll
            for (int k = 0; k < CH; ++k)
                if (c0 + k < y_sp) d[k] = q[0][k];
        }
    }
}

// x pixels of x_sp elements (image stride x_sn) -> y float32 [N, C, HW]:
// (float)((double)(stored + off) * scale). A tile is 256 pixels x 16 bytes
// of channels; VEC: 16-byte reads of whole chunks; V4: float4 stores (HW a
// multiple of 4), a wave writing 1 KB of a plane at a time.
template <class T, bool VEC, bool V4>
__global__ __launch_bounds__(kThreads) void k_dequantize_tile(
    const T* __restrict__ x, int64_t x_sn, int64_t x_sp, int C, uint32_t HW,
    uint32_t pixels, float* __restrict__ y, double scale, int64_t off) {
    constexpr int CH = 16 / sizeof(T);
    constexpr int PW = 4 / sizeof(T);  // channels a word
    __shared__ uint32_t t[256 * 5];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t p0 = blockIdx.x * 256;
    const int c0 = blockIdx.y * CH;
    {
        const uint32_t p = min(p0 + tid, pixels - 1);
        const uint32_t n = p / HW;
        const T* s = x + n * x_sn + (int64_t)(p - n * HW) * x_sp + c0;
        uint32_t w[4] = {0, 0, 0, 0};
        // (a view's last chunk may end the allocation: element loads)
        if (VEC && c0 + CH <= C) {
            const uint4 v = *(const uint4*)s;
            w[0] = v.x;
            w[1] = v.y;
            w[2] = v.z;
            w[3] = v.w;
        } else {
#pragma unroll
            for (int k = 0; k < CH; ++k) {
                const uint32_t b = (uint32_t)s[min(k, C - 1 - c0)] &
                                   (sizeof(T) == 1 ? 0xffu : 0xffffu);
                w[k / PW] |= b << (8 * sizeof(T) * (k % PW));
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) t[tid * 5 + k] = w[k];
    }
    __syncthreads();
    // wave w writes the channels of word w of its lanes' 4 pixels:
    // V4: pixels 4 lane .. + 3, else lane + 64 j
    const int ca = c0 + wave * PW;
    if (ca >= C) return;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        w[j] = t[(V4 ? 4 * lane + j : lane + 64 * j) * 5 + wave];
    auto value = [&](uint32_t v, int k) {
        return (float)((double)((int64_t)(T)(v >> (8 * sizeof(T) * k)) + off) *
                       scale);
    };
    if constexpr (V4) {
        const uint32_t p = p0 + 4 * lane;
        if (p >= pixels) return;
        const uint32_t n = p / HW;
        float* d = y + ((int64_t)n * C + ca) * (int64_t)HW + (p - n * HW);
#pragma unroll
        for (int k = 0; k < PW; ++k)
            if (ca + k < C)
                *(float4*)(d + (int64_t)k * HW) =
                    make_float4(value(w[0], k), value(w[1], k),
                                value(w[2], k), value(w[3], k));
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t p = p0 + lane + 64 * j;
            if (p >= pixels) return;
            const uint32_t n = p / HW;
            float* d = y + ((int64_t)n * C + ca) * (int64_t)HW + (p - n * HW);
#pragma unroll
            for (int k = 0; k < PW; ++k)
                if (ca + k < C) d[(int64_t)k * HW] = value(w[j], k);
        }
    }
}

bool launched(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_hip_error(what, e);
        return false;
    }
    return true;
}

// Tiles of pixels on grid axis x, of channels on y; pixels in 32 bits.
bool tile_grid_ok(int64_t pixels, int64_t ch_tiles) {
    return pixels < ((int64_t)1 << 31) - 4096 && ch_tiles <= 65535;
}

template <class T>
bool quantize_planes(const float* x, int64_t N, int64_t C, int64_t HW, T* y,
                     int64_t y_sp, const QuantTo& o, hipStream_t st) {
    const int64_t pixels = N * HW, row = y_sp * (int64_t)sizeof(T);
    if (row % 16 == 0 && (uintptr_t)y % 16 == 0 &&
        tile_grid_ok(pixels, ceil_div(row, 16))) {
        // the widest tile the pixel fills: 16, 32 or 64 bytes
        auto go = [&](auto rb) {
            constexpr int RB = decltype(rb)::value;
            const int64_t gx = ceil_div(pixels, 4096 / RB);
            const int64_t gy = ceil_div(row, RB);
            k_quantize_tile<T, RB>
                <<<dim3((unsigned)gx, (unsigned)gy), kThreads, 0, st>>>(
                    x, (int)C, (uint32_t)HW, (uint32_t)pixels, y, (int)y_sp,
                    o);
            return launched("qa_d_quantize_nhwc");
        };
        if (row == 16) return go(std::integral_constant<int, 16>{});
        if (row == 32) return go(std::integral_constant<int, 32>{});
        return go(std::integral_constant<int, 64>{});
    }
    // (four pixels a thread once single ones fill the chip: 3 channels of
    // 32x224x224 10.4 -> 7.3 us, but of 1x224x224 2.8 -> 3.3)
    const bool four = sizeof(T) == 2 && y_sp == 4 && HW % 4 == 0 &&
                      pixels >= (1 << 18) &&
                      ((uintptr_t)x | (uintptr_t)y) % 16 == 0;
    const int64_t groups = four ? pixels / 4 : pixels;
    const int64_t nch = ceil_div(y_sp, 4);
    const unsigned g = grid_1d(groups * nch, kThreads, 1 << 20);
    if (four)
        k_quantize_any<T, 4, 4><<<g, kThreads, 0, st>>>(x, C, HW, groups, nch,
                                                        y, y_sp, o);
    else
        k_quantize_any<T, 4, 1><<<g, kThreads, 0, st>>>(x, C, HW, groups, nch,
                                                        y, y_sp, o);
    return launched("qa_d_quantize_nhwc");
}

template <class T>
bool dequantize_planes(const T* x, int64_t x_sn, int64_t x_sp, int64_t N,
                       int64_t C, int64_t HW, float* y, double scale,
                       int64_t off, hipStream_t st) {
    constexpr int CH = 16 / sizeof(T);
    const int64_t gx = ceil_div(N * HW, 256), gy = ceil_div(C, CH);
    if (!tile_grid_ok(N * HW, gy)) {
        set_error("qa_d_dequantize_nchw",
                  "2^31 pixels or more, or more than 65535 chunks of channels");
        return false;
    }
    const bool vec = x_sp % CH == 0 && x_sn % CH == 0 && (uintptr_t)x % 16 == 0;
    const bool v4 = HW % 4 == 0 && (uintptr_t)y % 16 == 0;
    auto go = [&](auto v, auto f) {
        k_dequantize_tile<T, decltype(v)::value, decltype(f)::value>
            <<<dim3((unsigned)gx, (unsigned)gy), kThreads, 0, st>>>(
                x, x_sn, x_sp, (int)C, (uint32_t)HW, (uint32_t)(N * HW), y,
                scale, off);
    };
    if (vec && v4)
        go(std::true_type{}, std::true_type{});
    else if (vec)
        go(std::true_type{}, std::false_type{});
    else if (v4)
        go(std::false_type{}, std::true_type{});
    else
        go(std::false_type{}, std::false_type{});
    return launched("qa_d_dequantize_nchw");
}

}  // namespace

bool launch_quantize_planes(const float* x, int64_t N, int64_t C, int64_t HW,
                            void* y, int y_code, int64_t y_sp, double scale,
                            int64_t zp, int64_t qmin, int64_t qmax,
                            int64_t so, hipStream_t st) {
    QuantTo o;
    o.scale = scale;
    o.inv = 1.0 / scale;
    o.invf = (float)o.inv;
    o.invlo = (float)(o.inv - (double)o.invf);
    o.f32ok = qa_f32_form_ok(scale, zp, qmin, qmax);
    o.zp = zp;
    o.qmin = qmin;
    o.qmax = qmax;
    o.so = so;
    return y_code == 1
               ? quantize_planes<int8_t>(x, N, C, HW, (int8_t*)y, y_sp, o, st)
               : quantize_planes<int16_t>(x, N, C, HW, (int16_t*)y, y_sp, o,
                                          st);
}

}  // namespace qa

using namespace qa;

QA_API int qa_d_dequantize_nchw(const void* x, int in_code, int64_t x_sn,
                                int64_t x_sp, int64_t N, int64_t C,
                                int64_t HW, float* y, double scale,
                                int64_t zp, int64_t in_so, void* stream) {
    if (N * C * HW <= 0) return 0;
    if (!x || !y || (in_code != 1 && in_code != 2) || x_sp < C) {
        set_error("qa_d_dequantize_nchw",
                  "needs int8 or int16 storage, its pixel stride at least C");
        return -1;
    }
    hipStream_t st = (hipStream_t)stream;
    const int64_t off = in_so - zp;
    const bool done =
        in_code == 1 ? dequantize_planes<int8_t>((const int8_t*)x, x_sn, x_sp,
                                                 N, C, HW, y, scale, off, st)
                     : dequantize_planes<int16_t>((const int16_t*)x, x_sn,
                                                  x_sp, N, C, HW, y, scale,
                                                  off, st);
    return done ? 0 : -1;
}
