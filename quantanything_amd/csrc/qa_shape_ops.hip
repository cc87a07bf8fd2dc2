// Integer shaping operators whose output parameters are the input's, so they
// move stored values without arithmetic (quant_layers.py:593-650):
//   Pad with the zero point           (float_ops.py:499-513, pad_value = zp)
//   MaxPool with qmin as padding      (float_ops.py:518-560, pad_value = qmin)
//   GlobalMaxPool                     (float_ops.py:586-589)
// Stored values (q - so) of any storage code; the padding value arrives as a
// stored value too.
#include <algorithm>
#include <cstdlib>
#include <utility>

#include "../../include/qa_hip.h"
#include "qa_common.h"

namespace qa {
namespace {

constexpr int kThreads = 256;

// Any strides: one output element a thread, the axis of the smallest output
// stride fastest (the launcher orders the axes).
template <class T>
__global__ __launch_bounds__(kThreads) void k_pad_nd(qa_nd_pad d,
                                                     int64_t total) {
    const T fill = (T)d.fill;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * kThreads) {
        int64_t rem = i, xo = 0, yo = 0;
        bool inside = true;
        for (int k = (int)d.ndim - 1; k >= 0; --k) {
            const int64_t c = rem % d.shape[k];
            rem /= d.shape[k];
            yo += c * d.ys[k];
            const int64_t src = c - d.lo[k];
            inside = inside && src >= 0 && src < d.xshape[k];
            xo += src * d.xs[k];
        }
        ((T*)d.y)[yo] = inside ? ((const T*)d.x)[xo] : fill;
    }
}

// The innermost axis contiguous on both sides: 16 bytes of an output row a
// thread, read in one (possibly unaligned) access where they come from
// inside the input. Indices in 32 bits. A 16x64x112x112 map padded by 2 + 1
// channels and 3 rows and columns: 15.7 us (85 us an element a thread with
// the image's x axis fastest, 64 bytes apart).
template <class T>
__global__ __launch_bounds__(kThreads) void k_pad_rows(qa_nd_pad d,
                                                       uint32_t chunks,
                                                       uint32_t total) {
    constexpr int CH = 16 / sizeof(T);
    const T fill = (T)d.fill;
    const int last = (int)d.ndim - 1;
    const int n_in = (int)d.shape[last], lo = (int)d.lo[last];
    const int xe = lo + (int)d.xshape[last];
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < total;
         i += gridDim.x * kThreads) {
        uint32_t rem = i / chunks;
        const int c = (int)(i - rem * chunks) * CH;
        int64_t xo = 0, yo = c;
        bool inside = true;
        for (int k = last - 1; k >= 0; --k) {
            const uint32_t n = (uint32_t)d.shape[k], q = rem / n;
            const int64_t v = rem - q * n, src = v - d.lo[k];
            rem = q;
            yo += v * d.ys[k];
            inside = inside && src >= 0 && src < d.xshape[k];
            xo += src * d.xs[k];
        }
        const T* x = (const T*)d.x + xo - lo;  // element c of the row: x[c]
        T* y = (T*)d.y + yo;
        T v[CH];
        if (inside && c >= lo && c + CH <= xe) {
            __builtin_memcpy(v, x + c, 16);
        } else {
#pragma unroll
            for (int k = 0; k < CH; ++k)
                v[k] = inside && c + k >= lo && c + k < xe ? x[c + k] : fill;
        }
        if (c + CH <= n_in) {
            __builtin_memcpy(y, v, 16);
        } else {
#pragma unroll
            for (int k = 0; k < CH; ++k)
                if (c + k < n_in) y[k] = v[k];
        }
    }
}

// One output element per thread, channels fastest (coalesced on
// channels-last tensors). A window tap outside the image contributes the
// padding value, as the reference's padded array does.
template <class T>
__global__ __launch_bounds__(kThreads) void k_maxpool(qa_maxpool_desc d,
                                                      int64_t total) {
    const T* x = (const T*)d.x;
    T* y = (T*)d.y;
    const int pad = (int)d.pad;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * kThreads) {
        const int64_t c = i % d.C;
        int64_t r = i / d.C;
        const int64_t ox = r % d.OW;
        r /= d.OW;
        const int64_t oy = r % d.OH;
        const int64_t n = r / d.OH;
        const T* xb = x + n * d.x_sn + c * d.x_sc;
        int acc = INT32_MIN;
        for (int64_t ky = 0; ky < d.KH; ++ky) {
            const int64_t iy = oy * d.SH - d.PT + ky * d.DH;
            const bool row_in = iy >= 0 && iy < d.H;
            for (int64_t kx = 0; kx < d.KW; ++kx) {
                const int64_t ix = ox * d.SW - d.PL + kx * d.DW;
                const int v = (row_in && ix >= 0 && ix < d.W)
                                  ? (int)xb[iy * d.x_sh + ix * d.x_sw]
                                  : pad;
                acc = max(acc, v);
            }
        }
        y[n * d.y_sn + c * d.y_sc + oy * d.y_sh + ox * d.y_sw] = (T)acc;
    }
}

// Channels-last int8 / int16 windows: a thread reduces 16 bytes of channels
// of one output pixel. Elementwise maxima of packed int16: of bytes b3 b2 b1
// b0, the maximum of the words as int16 pairs carries that of b3 and b1 in
// its high bytes whatever the low ones hold, and that of the words shifted
// left by 8 those of b2 and b0.
typedef short s2 __attribute__((ext_vector_type(2)));

template <class T>
struct MaxAcc {
    s2 hi[4], lo[4];  // int16 storage uses hi alone
    __device__ __forceinline__ void set(int pad) {
        const uint32_t w = sizeof(T) == 1
                               ? (uint32_t)(uint8_t)pad * 0x01010101u
                               : (uint32_t)(uint16_t)pad * 0x00010001u;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            hi[k] = __builtin_bit_cast(s2, w);
            lo[k] = __builtin_bit_cast(s2, w << 8);
        }
    }
    __device__ __forceinline__ void add(const uint32_t* w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            hi[k] = __builtin_elementwise_max(hi[k],
                                              __builtin_bit_cast(s2, w[k]));
            if (sizeof(T) == 1)
                lo[k] = __builtin_elementwise_max(
                    lo[k], __builtin_bit_cast(s2, w[k] << 8));
        }
    }
    __device__ __forceinline__ uint4 value() const {
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            w[k] = __builtin_bit_cast(uint32_t, hi[k]);
            if (sizeof(T) == 1)
                w[k] = (w[k] & 0xff00ff00u) |
                       (__builtin_bit_cast(uint32_t, lo[k]) >> 8 &
                        0x00ff00ffu);
        }
        return make_uint4(w[0], w[1], w[2], w[3]);
    }
};

// The end of the tensor's last element. 16 bytes that end before it lie
// between its first and last element, whatever they hold past a pixel's
// channels (maxpool_cl_ok: no negative strides).
template <class T>
__device__ __forceinline__ const T* pool_end(const qa_maxpool_desc& d) {
    return (const T*)d.x + (d.N - 1) * d.x_sn + (d.H - 1) * d.x_sh +
           (d.W - 1) * d.x_sw + d.C;
}

// 16 bytes of channels at p, the first `real` of them the pixel's (the
// others anything); element loads where the tensor ends within them
template <class T>
__device__ __forceinline__ void load_chunk(const T* p, int real,
                                           const T* end, uint32_t* w) {
    constexpr int CH = 16 / sizeof(T);
    if (real >= CH || p + CH <= end) {
        const uint4 v = *(const uint4*)p;
        w[0] = v.x;
        w[1] = v.y;
        w[2] = v.z;
        w[3] = v.w;
        return;
    }
    w[0] = w[1] = w[2] = w[3] = 0;
#pragma unroll
    for (int k = 0; k < CH; ++k)
        if (k < real) {
            const uint32_t b = (uint32_t)p[k] &
                               (sizeof(T) == 1 ? 0xffu : 0xffffu);
            w[k * sizeof(T) / 4] |= b << (8 * (k * sizeof(T) % 4));
        }
}

template <class T>
__device__ __forceinline__ void store_chunk(T* p, int real, uint4 v) {
    constexpr int CH = 16 / sizeof(T);
    if (real >= CH) {
        *(uint4*)p = v;
        return;
    }
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < CH; ++k)
        if (k < real)
            p[k] = (T)(w[k * sizeof(T) / 4] >> (8 * (k * sizeof(T) % 4)));
}

// K: a K x K window, its taps unrolled so that all loads are in flight
// where a whole wave's windows lie inside the image; 0: any window.
// 16x32x112x112, 5x5 (12.8 MB moved, 25 taps from L1): 12.6 us; 105 us with
// a channel a thread. A last chunk of fewer channels is loaded whole
// (8x100x20x20, 5x5: 6.1 us, 14.7 us by elements).
template <class T, int K>
__global__ __launch_bounds__(kThreads) void k_maxpool_cl(qa_maxpool_desc d,
                                                         uint32_t nch,
                                                         uint32_t total) {
    constexpr int CH = 16 / sizeof(T);
    const T* const end = pool_end<T>(d);
    for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < total;
         i += gridDim.x * kThreads) {
        uint32_t r = i / nch;
        const int c = (int)(i - r * nch) * CH;
        uint32_t q = r / (uint32_t)d.OW;
        const int ox = (int)(r - q * (uint32_t)d.OW);
        r = q / (uint32_t)d.OH;
        const int oy = (int)(q - r * (uint32_t)d.OH);
        const int64_t n = r;
        const int KH = K ? K : (int)d.KH, KW = K ? K : (int)d.KW;
        const int real = min(CH, (int)d.C - c);
        const int iy0 = oy * (int)d.SH - (int)d.PT;
        const int ix0 = ox * (int)d.SW - (int)d.PL;
        const T* xb = (const T*)d.x + n * d.x_sn + c;
        MaxAcc<T> acc;
        const int iy1 = iy0 + (KH - 1) * (int)d.DH;
        const int ix1 = ix0 + (KW - 1) * (int)d.DW;
        const bool in = iy0 >= 0 && ix0 >= 0 && iy1 < (int)d.H &&
                        ix1 < (int)d.W &&
                        (real >= CH ||
                         xb + iy1 * d.x_sh + ix1 * d.x_sw + CH <= end);
        if (K > 0 && __all(in)) {
            const T* p = xb + iy0 * d.x_sh + ix0 * d.x_sw;
            uint4 v[K > 0 ? K * K : 1];
#pragma unroll
            for (int t = 0; t < K * K; ++t)
                v[t] = *(const uint4*)(p + (t / K) * (d.DH * d.x_sh) +
                                       (t % K) * (d.DW * d.x_sw));
            const uint32_t w0[4] = {v[0].x, v[0].y, v[0].z, v[0].w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                acc.hi[k] = __builtin_bit_cast(s2, w0[k]);
                acc.lo[k] = __builtin_bit_cast(s2, w0[k] << 8);
            }
#pragma unroll
            for (int t = 1; t < K * K; ++t) {
                const uint32_t w[4] = {v[t].x, v[t].y, v[t].z, v[t].w};
                acc.add(w);
            }
        } else {
            bool first = true;  // no tap read yet: acc is the padding value
            acc.set((int)d.pad);
            for (int ky = 0; ky < KH; ++ky) {
                const int iy = iy0 + ky * (int)d.DH;
                const bool row_in = (uint32_t)iy < (uint32_t)d.H;
                for (int kx = 0; kx < KW; ++kx) {
                    const int ix = ix0 + kx * (int)d.DW;
                    uint32_t w[4];
                    if (row_in && (uint32_t)ix < (uint32_t)d.W) {
                        load_chunk(xb + iy * d.x_sh + ix * d.x_sw, real, end,
                                   w);
                    } else {
                        const uint32_t u =
                            sizeof(T) == 1
                                ? (uint32_t)(uint8_t)d.pad * 0x01010101u
                                : (uint32_t)(uint16_t)d.pad * 0x00010001u;
                        w[0] = w[1] = w[2] = w[3] = u;
                    }
                    if (first) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            acc.hi[k] = __builtin_bit_cast(s2, w[k]);
                            acc.lo[k] = __builtin_bit_cast(s2, w[k] << 8);
                        }
                        first = false;
                    } else {
                        acc.add(w);
                    }
                }
            }
        }
        store_chunk((T*)d.y + n * d.y_sn + c + oy * d.y_sh + ox * d.y_sw,
                    real, acc.value());
    }
}

// Windows of many taps (a GlobalMaxPool): a work-group an output pixel and
// up to 16 chunks of channels, its threads taking the taps in turn and
// meeting in LDS. 16x64x28x28 -> 1x1: 6.0 us (84 us a thread a channel).
template <class T>
__global__ __launch_bounds__(kThreads) void k_maxpool_wide(qa_maxpool_desc d,
                                                           uint32_t nch,
                                                           int cb) {
    constexpr int CH = 16 / sizeof(T);
    __shared__ uint4 part[kThreads];
    const int tid = threadIdx.x, cl = tid & (cb - 1), t0 = tid / cb;
    const int step = kThreads / cb;
    const uint32_t chunk = blockIdx.y * cb + cl;
    uint32_t q = blockIdx.x / (uint32_t)d.OW;
    const int ox = (int)(blockIdx.x - q * (uint32_t)d.OW);
    const int64_t n = q / (uint32_t)d.OH;
    const int oy = (int)(q - (uint32_t)n * (uint32_t)d.OH);
    const bool live = chunk < nch;
    const int c = (int)(live ? chunk : 0) * CH;
    const int real = min(CH, (int)d.C - c);
    const int iy0 = oy * (int)d.SH - (int)d.PT;
    const int ix0 = ox * (int)d.SW - (int)d.PL;
    const T* xb = (const T*)d.x + n * d.x_sn + c;
    const T* const end = pool_end<T>(d);
    const int taps = (int)(d.KH * d.KW);
    // a thread without taps repeats the first one
    auto tap = [&](int t, uint32_t* w) {
        const int ky = t / (int)d.KW, kx = t - ky * (int)d.KW;
        const int iy = iy0 + ky * (int)d.DH, ix = ix0 + kx * (int)d.DW;
        const bool in = (uint32_t)iy < (uint32_t)d.H &&
                        (uint32_t)ix < (uint32_t)d.W;
        if (in) {
            load_chunk(xb + iy * d.x_sh + ix * d.x_sw, real, end, w);
        } else {
            const uint32_t u = sizeof(T) == 1
                                   ? (uint32_t)(uint8_t)d.pad * 0x01010101u
                                   : (uint32_t)(uint16_t)d.pad * 0x00010001u;
            w[0] = w[1] = w[2] = w[3] = u;
        }
    };
    MaxAcc<T> acc;
    {
        uint32_t w[4];
        tap(t0 < taps ? t0 : 0, w);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            acc.hi[k] = __builtin_bit_cast(s2, w[k]);
            acc.lo[k] = __builtin_bit_cast(s2, w[k] << 8);
        }
    }
#pragma unroll 4
    for (int t = t0 + step; t < taps; t += step) {
        uint32_t w[4];
        tap(t, w);
        acc.add(w);
    }
    part[tid] = acc.value();
    __syncthreads();
    for (int h = step / 2; h > 0; h /= 2) {
        if (t0 < h) {
            const uint4 a = part[tid + h * cb];
            const uint32_t w[4] = {a.x, a.y, a.z, a.w};
            acc.add(w);
            part[tid] = acc.value();
        }
        __syncthreads();
    }
    if (t0 == 0 && live)
        store_chunk((T*)d.y + n * d.y_sn + c + oy * d.y_sh + ox * d.y_sw,
                    real, acc.value());
}

// Whether the 16-byte channel kernels take a pool: channels contiguous, every
// other stride (none of them negative) and both bases on 16 bytes, extents
// and indices in 32 bits.
bool maxpool_cl_ok(const qa_maxpool_desc& d) {
    if (d.code != 1 && d.code != 2) return false;
    const int64_t ch = 16 / d.code, lim = (int64_t)1 << 30;
    const int64_t st[6] = {d.x_sn, d.x_sh, d.x_sw, d.y_sn, d.y_sh, d.y_sw};
    for (int64_t v : st)
        if (v < 0 || v % ch) return false;
    const int64_t ext[] = {d.H, d.W, d.KH, d.KW, d.C, d.KH * d.KW,
                           d.OH * d.SH, d.OW * d.SW, d.KH * d.DH,
                           d.KW * d.DW};
    for (int64_t v : ext)
        if (v >= lim) return false;
    return d.x_sc == 1 && d.y_sc == 1 && d.PT > -lim && d.PT < lim &&
           d.PL > -lim && d.PL < lim &&
           ((uintptr_t)d.x | (uintptr_t)d.y) % 16 == 0 &&
           d.N * d.OH * d.OW * ceil_div(d.C, ch) < ((int64_t)1 << 31);
}

// Launches a 16-byte form, or leaves the pool to the element kernel: false.
template <class T>
bool launch_maxpool_cl(const qa_maxpool_desc& d, hipStream_t st) {
    constexpr int64_t ch = 16 / sizeof(T);
    const int64_t nch = ceil_div(d.C, ch);
    const int64_t outs = d.N * d.OH * d.OW;
    // Many taps and few outputs: a work-group an output (taps without an
    // unrolled form in a thread, one after the other, against it, us: 64x512
    // of 7x7 -> 1x1 12.1 / 3.9, 4x4 windows of 32x256x32x32, 32768 chunks
    // of outputs, 5.6 / 5.0, 7x7 of 16x128x20x20, 51200, 11.4 / 13.4; with a
    // partial last chunk 4x4 of 4x15x21x21 4.1 / 4.9).
    const int64_t taps = d.KH * d.KW;
    const bool unrolled =
        d.KH == d.KW && (d.KH == 2 || d.KH == 3 || d.KH == 5);
    if ((taps >= 64 && outs * nch < 65536) ||
        (taps >= (d.C % ch ? 32 : 16) && !unrolled && outs * nch <= 32768)) {
        int cb = 1;
        while (cb < nch && cb < 16) cb *= 2;
        const dim3 g((unsigned)outs, (unsigned)ceil_div(nch, cb));
        k_maxpool_wide<T><<<g, kThreads, 0, st>>>(d, (uint32_t)nch, cb);
        return true;
    }
    // A partial last chunk stores by elements: not for small maps (element
    // kernel / this one, us: 4x15x41x41 5x5 5.5 / 8.2, 2x24x28x28 2x2 2.9 /
    // 3.4, 275 thousand outputs of 67 channels 2x2 3.2 / 3.4; 8x100x20x20 5x5
    // 7.2 / 6.1, 32x24x56x56 2x2 5.5 / 3.9).
    if (d.C % ch && outs * d.C < (taps >= 16 ? 1 << 18 : 3 << 17))
        return false;
    // Nor does a window without an unrolled form over a small map (3x64x37x37
    // 2x3 3.2 / 3.5, 1x32x20x20 3x5 3.9 / 4.8; 8x64x37x37 2x3 3.7 / 3.6,
    // int16 3x64x37x37 3.3 / 3.4).
    if (!unrolled && outs * d.C < (sizeof(T) == 1 ? 5 << 15 : 1 << 15))
        return false;
    const int64_t total = outs * nch;
    const unsigned nb =
        (unsigned)std::min<int64_t>(ceil_div(total, kThreads), 1 << 20);
    const uint32_t n32 = (uint32_t)nch, t32 = (uint32_t)total;
    const int64_t k = d.KH == d.KW ? d.KH : 0;
    if (k == 2)
        k_maxpool_cl<T, 2><<<nb, kThreads, 0, st>>>(d, n32, t32);
    else if (k == 3)
        k_maxpool_cl<T, 3><<<nb, kThreads, 0, st>>>(d, n32, t32);
    else if (k == 5)
        k_maxpool_cl<T, 5><<<nb, kThreads, 0, st>>>(d, n32, t32);
    else
        k_maxpool_cl<T, 0><<<nb, kThreads, 0, st>>>(d, n32, t32);
    return true;
}

bool code_ok(int64_t c) { return c == 1 || c == 2 || c == 4; }

unsigned blocks_for(int64_t total) {
    return (unsigned)std::min<int64_t>(ceil_div(total, kThreads), 1 << 16);
}

bool launched(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_hip_error(what, e);
        return false;
    }
    return true;
}

}  // namespace
}  // namespace qa

using namespace qa;

QA_API int qa_d_pad_nd(const qa_nd_pad* d, void* stream) {
    if (!d || d->ndim < 1 || d->ndim > 6 || !code_ok(d->code)) {
        set_error("qa_d_pad_nd", "bad descriptor");
        return -1;
    }
    int64_t total = 1;
    for (int k = 0; k < d->ndim; ++k) {
        if (d->shape[k] < 0 || d->xshape[k] < 0 || d->lo[k] < 0) {
            set_error("qa_d_pad_nd", "negative extent or padding");
            return -1;
        }
        total *= d->shape[k];
    }
    if (total == 0) return 0;
    if (!d->x || !d->y) {
        set_error("qa_d_pad_nd", "null tensor");
        return -1;
    }
    hipStream_t st = (hipStream_t)stream;
    // the axes by descending output stride (the innermost written
    // contiguously); a permutation of the axes changes no element
    qa_nd_pad o = *d;
    for (int k = 1; k < o.ndim; ++k)
        for (int j = k; j > 0 && std::abs(o.ys[j]) > std::abs(o.ys[j - 1]);
             --j) {
            std::swap(o.shape[j], o.shape[j - 1]);
            std::swap(o.lo[j], o.lo[j - 1]);
            std::swap(o.xshape[j], o.xshape[j - 1]);
            std::swap(o.xs[j], o.xs[j - 1]);
            std::swap(o.ys[j], o.ys[j - 1]);
        }
    const int last = (int)o.ndim - 1;
    const int64_t ch = 16 / o.code, chunks = ceil_div(o.shape[last], ch);
    const int64_t rows = total / o.shape[last];
    bool small = rows * chunks < ((int64_t)1 << 31);
    for (int k = 0; k <= last; ++k)
        small = small && o.shape[k] < (1 << 30) && o.lo[k] < (1 << 30) &&
                o.xshape[k] < (1 << 30);
    if (o.ys[last] == 1 && o.xs[last] == 1 && small && o.code <= 2 &&
        o.shape[last] >= ch && rows16_pay(o.code, o.ndim, total)) {
        const unsigned g = (unsigned)std::min<int64_t>(
            ceil_div(rows * chunks, kThreads), 1 << 20);
        if (o.code == 1)
            k_pad_rows<int8_t><<<g, kThreads, 0, st>>>(
                o, (uint32_t)chunks, (uint32_t)(rows * chunks));
        else
            k_pad_rows<int16_t><<<g, kThreads, 0, st>>>(
                o, (uint32_t)chunks, (uint32_t)(rows * chunks));
        return launched("qa_d_pad_nd") ? 0 : -1;
    }
    d = &o;
    const unsigned nb = blocks_for(total);
    switch (d->code) {
        case 1: k_pad_nd<int8_t><<<nb, kThreads, 0, st>>>(*d, total); break;
        case 2: k_pad_nd<int16_t><<<nb, kThreads, 0, st>>>(*d, total); break;
        default: k_pad_nd<int32_t><<<nb, kThreads, 0, st>>>(*d, total);
    }
    return launched("qa_d_pad_nd") ? 0 : -1;
}

QA_API int qa_d_maxpool(const qa_maxpool_desc* d, void* stream) {
    if (!d || !code_ok(d->code) || d->N < 0 || d->C < 0 || d->H < 0 ||
        d->W < 0 || d->OH < 0 || d->OW < 0 || d->KH < 1 || d->KW < 1 ||
        d->SH < 1 || d->SW < 1 || d->DH < 1 || d->DW < 1) {
        set_error("qa_d_maxpool", "bad descriptor");
        return -1;
    }
    const int64_t total = d->N * d->C * d->OH * d->OW;
    if (total == 0) return 0;
    if (!d->x || !d->y) {
        set_error("qa_d_maxpool", "null tensor");
        return -1;
    }
    hipStream_t st = (hipStream_t)stream;
    if (maxpool_cl_ok(*d) && (d->code == 1 ? launch_maxpool_cl<int8_t>(*d, st)
                                           : launch_maxpool_cl<int16_t>(*d, st)))
        return launched("qa_d_maxpool") ? 0 : -1;
    const unsigned nb = blocks_for(total);
    switch (d->code) {
        case 1: k_maxpool<int8_t><<<nb, kThreads, 0, st>>>(*d, total); break;
        case 2: k_maxpool<int16_t><<<nb, kThreads, 0, st>>>(*d, total); break;
        default: k_maxpool<int32_t><<<nb, kThreads, 0, st>>>(*d, total);
    }
    return launched("qa_d_maxpool") ? 0 : -1;
}
