// Int8 GEMMs with the table epilogue on 64 x 128, 256 x 128 and 256 x 256
// blocks (qa_gemm_big.hip has 128 x 128 and the operands' layouts). K runs
// through a ring of S LDS stages of 64 bytes, each BM activation rows and BN
// weight rows, filled by global_load_lds_dwordx4: no registers hold loads in
// flight, S - 1 steps are requested ahead. A wave owns 16 MT x 16 NT values
// (v_mfma_i32_16x16x64_i8) and reads the next step's fragments while a step's
// MFMAs run: with the reads of a step before its own MFMAs, a block alone on
// its CU took about 850 cycles a step, most of them those reads.
//
// What bounds it: no one unit. 16384x1024x1024 takes 28.3 us in 128 x 128
// blocks and 21.5-22.3 here (1540-1600 TOP/s), one block of 256 x 256 and 8
// waves on each CU. Counted there: a wave lives 37.7 k cycles and waits 11.8 k
// of them (direct loads, LDS, barriers); its SIMD's matrix core works 16.4 k;
// the LDS is busy 6.2 k without a bank conflict, and a wave waits 1.0 k to
// issue to it. Of the wave's 1762 VALU instructions 512 are MFMAs, most of the
// rest its epilogue of 128 accumulators a lane, and no other block is on the
// CU whose MFMAs could fill that time or the first stages' loads.
//
// The epilogue is the int8 table plan of qa_conv.h, identical in results to
// the convolution kernel's; residual, copy and pixel sums are template flags,
// full tiles skip the bounds tests.
//
// Weight row 4 c + j of a wave's 64 (j < 4) is staged as row 16 j + c: lane
// column c of the four MFMA blocks then holds four consecutive channels of a
// row, so the epilogue packs a word without a transpose across lanes and 16
// lanes store 64 contiguous bytes.
#include <type_traits>

#include "qa_conv_mfma.h"

namespace qa {
namespace {

// 16 bytes a lane from global memory to LDS bytes 16 lane of l (a plain
// function: in a template the host pass drops the kernel for the builtin)
__device__ __forceinline__ void direct_load16(const int8_t* g, int8_t* l) {
    __builtin_amdgcn_global_load_lds(g, l, 16, 0, 0);
}

// s_waitcnt vmcnt(N) alone (N < 64; expcnt and lgkmcnt not waited)
template <int N>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}
// vmcnt(L * n) for n in [0, S - 2]
template <int L, int S>
__device__ __forceinline__ void wait_steps(int n) {
    static_assert(S >= 2 && S <= 8 && L * (S - 2) < 64, "ring");
    switch (n) {
        case 0: wait_vm<0>(); break;
        case 1: wait_vm<L>(); break;
        case 2: wait_vm<2 * L>(); break;
        case 3: wait_vm<3 * L>(); break;
        case 4: wait_vm<4 * L>(); break;
        case 5: wait_vm<5 * L>(); break;
        default: wait_vm<6 * L>(); break;
    }
}

// RES / Y2 / RS: residual Add, rescaled second output, pixel sums of the
// activations (weights with an offset) in the epilogue. The stage's row r
// holds its 16-byte chunk c at position c ^ ((r >> 1) & 3): the 8 rows one
// fragment read serves at a time fall in distinct banks without padding (a
// 64-lane direct load fills 1 KB contiguously: 16 rows of 4 positions).
template <int BM, int BN, int WM, int WN, int S, bool RES, bool Y2, bool RS>
__global__ __launch_bounds__(
    64 * WM * WN, BM * BN / (WM * WN) <= 4096 ? 2 : 1) void k_gemm_stage(ConvArgs a) {
    constexpr int NW = WM * WN;
    constexpr int MT = BM / WM / 16, NT = BN / WN / 16;
    static_assert(NT % 4 == 0, "a lane holds words of 4 channels");
    constexpr int L = (BM + BN) / 16 / NW;  // direct loads a wave and step
    static_assert(L * 16 * NW == BM + BN, "whole loads");
    constexpr int STG = 64 * (BM + BN);
    extern __shared__ int4 gs_dyn[];
    __shared__ int s_tab[768];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int col = lane & 15, kg = lane >> 4;
    // consecutive work-groups go to different XCDs (round robin): the linear
    // index is remapped to make the tiles of each XCD consecutive; consecutive
    // tiles share their A rows (column blocks fastest), which then stay in
    // that XCD's L2
    const int nb = (a.Cout + BN - 1) / BN;
    const int ntile = gridDim.x;
    const int per = (ntile + 7) / 8;
    const int bid = blockIdx.x;
    const int xcd = bid & 7, idx = bid >> 3;
    const int rem = ntile - 8 * (per - 1);
    const int t = xcd < rem ? xcd * per + idx
                            : rem * per + (xcd - rem) * (per - 1) + idx;
    const int64_t m0 = (int64_t)(t / nb) * BM;
    const int n0 = (t % nb) * BN;
    const int K = a.KGp * 16;
    const int kx = a.Cg;  // bytes of an activation row
    const int nk = K / 64;
    const int8_t* xa = (const int8_t*)a.x;

    // the plan's tables before the operands: storing them waits for them
    // alone (loads complete in issue order)
    constexpr int TV = (768 + 64 * NW - 1) / (64 * NW);
    int tv[TV];
#pragma unroll
    for (int j = 0; j < TV; ++j)
        tv[j] = ((const int*)((const char*)a.plan +
                              PLAN_E))[min(tid + 64 * NW * j, 767)];

    // this lane's direct loads: the wave's load j fills stage rows
    // 16 (L wave + j) + lane / 4 (A's, then B's), the global chunk stored at
    // position lane % 4. Rows past M repeat the last one; weight rows past
    // Cout likewise (their columns are not stored).
    int8_t* const stg = (int8_t*)gs_dyn;
    const int gch = 16 * ((lane & 3) ^ ((lane >> 3) & 3));
    const int8_t* gp[L];
    int alim[L];  // K bytes its rows hold
#pragma unroll
    for (int j = 0; j < L; ++j) {
        const int r = 16 * (L * wave + j) + (lane >> 2);
        if (16 * (L * wave + j) < BM) {
            gp[j] = xa + min(m0 + r, a.M - 1) * a.x_sn;
            alim[j] = kx;
        } else {
            const int rb = r - BM;  // 64 q + 16 j' + c
            const int n = (rb & ~63) + 4 * (rb & 15) + ((rb >> 4) & 3);
            gp[j] = a.wp + (int64_t)min(n0 + n, a.Cout - 1) * a.wp_rstride;
            alim[j] = K;
        }
    }
    auto dload = [&](int ks, int slot) __attribute__((always_inline)) {
        int8_t* const sb = stg + slot * STG + 1024 * L * wave;
        const int ko = 64 * ks + gch;
#pragma unroll
        for (int j = 0; j < L; ++j)
            direct_load16(gp[j] + (ko < alim[j] ? ko : 0), sb + 1024 * j);
    };
    // rows 16 i + 4 kg + r, channels c0 + 64 u .. + 3 of the tile
    const int64_t p0 = m0 + 16 * MT * wm + 4 * kg;
    const int c0 = n0 + 16 * NT * wn + 4 * col;
    // the lane's channels' plan constants (used after the K loop, so that
    // nothing waits for them before the operands)
    const int4 hdr = *(const int4*)a.plan;
    int4 pc[NT];
    uint32_t cr[NT], cbo[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int c = min(c0 + 64 * (j >> 2) + (j & 3), a.Cout - 1);
        pc[j] = ((const int4*)((const char*)a.plan + PLAN_CH))[c];
        cr[j] = a.corr ? (uint32_t)a.corr[c] : 0u;
        cbo[j] = RS ? (uint32_t)a.boff[c] : 0u;
    }
#pragma unroll
    for (int sl = 0; sl < S - 1; ++sl)
        if (sl < nk) dload(sl, sl);

    v4i acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    int psum[MT];  // stored-byte sums of the lane's A rows
#pragma unroll
    for (int i = 0; i < MT; ++i) psum[i] = 0;
    // a lane's fragment of rows 16 i + col, chunk kg, at position
    // kg ^ ((col >> 1) & 3) of the row
    const int foff = col * 64 + 16 * (kg ^ ((col >> 1) & 3));
    struct Frag {
        v4i a[MT], b[NT];
    };
    auto fetch = [&](Frag& f, int slot) __attribute__((always_inline)) {
        const int8_t* sb = stg + slot * STG + foff;
#pragma unroll
        for (int j = 0; j < NT; ++j)
            f.b[j] = *(const v4i*)(sb + 64 * BM + (16 * NT * wn + 16 * j) * 64);
#pragma unroll
        for (int i = 0; i < MT; ++i)
            f.a[i] = *(const v4i*)(sb + (16 * MT * wm + 16 * i) * 64);
    };
    // the waits are explicit: on the direct loads (wait_vm), and on this
    // wave's fragment reads but those of the last step (lds_barrier)
    constexpr int NF = MT + NT;  // fragment reads of a step
    auto barrier = [&]() __attribute__((always_inline)) { lds_barrier<NF>(); };
    auto product = [&](const Frag& f, int ks) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                    f.a[i], f.b[j], acc[i][j], 0, 0, 0);
        if (RS && 64 * ks + 16 * kg < kx) {
#pragma unroll
            for (int i = 0; i < MT; ++i) psum[i] += bytes_sum(f.a[i], 16);
        }
    };
    int slot = 1, fill = S - 1;  // the next step's stage, the one to refill
    auto advance = [&]() __attribute__((always_inline)) {
        fill = fill == S - 1 ? 0 : fill + 1;
        slot = slot == S - 1 ? 0 : slot + 1;
    };
    // step ks from cur's registers, the next step's fragments read meanwhile:
    // this wave's loads of step ks + 1 done (those of the next S - 3 steps may
    // still be in flight), barrier (every wave's part landed, and every wave
    // has the fragments of step ks - 1, whose stage the refill overwrites:
    // only the NF reads of step ks may still be in flight).
    // No branch between the reads and the MFMAs: at one the compiler waits
    // for every read.
    auto steady = [&](const Frag& cur, Frag& nxt, int ks)
                      __attribute__((always_inline)) {
        wait_vm<L * (S - 3)>();
        barrier();
        dload(ks + S - 1, fill);
        fetch(nxt, slot);
        advance();
        product(cur, ks);
    };
    Frag f0, f1;
    wait_steps<L, S>(min(S - 2, nk - 1));
    barrier();
    fetch(f0, 0);
    int ks = 0;
    for (; ks + S < nk; ks += 2) {
        steady(f0, f1, ks);
        steady(f1, f0, ks + 1);
    }
    for (; ks + 1 < nk; ++ks) {
        wait_steps<L, S>(min(S - 3, nk - 2 - ks));
        barrier();
        if (ks + S - 1 < nk) dload(ks + S - 1, fill);
        fetch(f1, slot);
        advance();
        product(f0, ks);
        f0 = f1;
    }
    product(f0, ks);
#pragma unroll
    for (int j = 0; j < TV; ++j)
        if (64 * NW * (j + 1) <= 768 || tid + 64 * NW * j < 768)
            s_tab[tid + 64 * NW * j] = tv[j];
    // the zero-point correction folded into the plan constant (K <= 16384
    // keeps |w| + |corr| + |boff * rowsum| below 2^31, so the int32 sum never
    // wraps); every shift past the low word of the product: of the high word
    // alone
    int cm[NT], ct[NT];
    int64_t cc[NT];
    bool hi = true;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        cm[j] = pc[j].x;
        ct[j] = pc[j].y;
        hi &= ct[j] >= 32;
        cc[j] = plan_fold(
            (int64_t)(((uint64_t)(uint32_t)pc[j].w << 32) | (uint32_t)pc[j].z),
            cr[j], pc[j].x);
    }
    hi = __all(hi);
    __syncthreads();

    // Per value: the plan's multiply-add and shift, one med3 clip and one
    // table read whose LDS address folds in the clip's lower bound. With a
    // residual the rows of one MFMA block a pass of a rolled loop, the
    // accumulators moved down between passes and the next rows' words
    // requested one pass ahead: a launch of a network fetches the code anew
    // (11 KB for 30 KB unrolled: 11.6 against 12.9 us at 6304x384x384 there);
    // without one the moves and registers cost more than they save.
    constexpr int IB = RES ? 1 : MT;
    const int pA = hdr.x, pB = hdr.y, pSH = hdr.z;
    const int pD = ((const int*)a.plan)[4];
    const int* tabE = s_tab - pA;  // tabE[v] = E[v - pA] for v in [pA, pB]
    // CHK: bounds tests and any shift; else a tile whole inside the output
    // with hi. IDT: identity table (a plain requantize), the byte of
    // clip(q0) + D.
    auto epilogue = [&](auto checked, auto identity)
                        __attribute__((always_inline)) {
        constexpr bool CHK = decltype(checked)::value;
        constexpr bool IDT = decltype(identity)::value;
        uint32_t rn[IB][4][NT / 4];  // residual words of the next rows
        auto residual = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
            for (int ib = 0; ib < IB; ++ib)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int u = 0; u < NT / 4; ++u)
                        rn[ib][r][u] = word_load_args(
                            (const int8_t*)a.res +
                            (p0 + 16 * (i0 + ib) + r) * a.res_pst + c0 +
                            64 * u);
        };
        if (RES && !CHK) residual(0);
#pragma unroll 1
        for (int i0 = 0; i0 < MT; i0 += IB) {
            uint32_t rc[IB][4][NT / 4];
            if (RES && !CHK) {
#pragma unroll
                for (int ib = 0; ib < IB; ++ib)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int u = 0; u < NT / 4; ++u)
                            rc[ib][r][u] = rn[ib][r][u];
                if (i0 + IB < MT) residual(i0 + IB);
            }
#pragma unroll
            for (int ib = 0; ib < IB; ++ib) {
                int sm = 0;
                if (RS) {
                    sm = psum[ib];
                    sm += __shfl_xor(sm, 16);
                    sm += __shfl_xor(sm, 32);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t p = p0 + 16 * (i0 + ib) + r;
                    const bool pok = !CHK || p < a.M;
                    const uint32_t ps =
                        RS ? (uint32_t)__shfl(sm, 4 * kg + r) : 0u;
#pragma unroll
                    for (int u = 0; u < NT / 4; ++u) {
                        const int c = c0 + 64 * u;
                        const bool cfull = !CHK || c + 3 < a.Cout;
                        uint32_t rv = 0;
                        if (RES && !CHK) rv = rc[ib][r][u];
                        if (RES && CHK && pok) {
                            const int8_t* pr =
                                (const int8_t*)a.res + p * a.res_pst + c;
                            if (cfull) {
                                rv = word_load_args(pr);
                            } else {
#pragma unroll
                                for (int j = 0; j < 4; ++j)
                                    if (c + j < a.Cout)
                                        rv |= (uint32_t)(uint8_t)pr[j]
                                              << (8 * j);
                            }
                        }
                        int e[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int jj = 4 * u + j;
                            int w = acc[ib][jj][r];
                            if (RS) w += (int)(cbo[jj] * ps);
                            const int64_t q64 =
                                (int64_t)((uint64_t)((int64_t)w * cm[jj]) +
                                          (uint64_t)cc[jj]);
                            const int q0 =
                                CHK ? (int)(q64 >> ct[jj])
                                    : (int)(q64 >> 32) >> (ct[jj] & 31);
                            const int v = med3_i32(q0, pA, pB);
                            if (RES) {
                                const int tsum =
                                    s_tab[256 - pA + v] +
                                    s_tab[512 + ((rv >> (8 * j)) & 255)];
                                e[j] = s_tab[med3_i32(tsum, 0, pSH)];
                            } else if (IDT) {
                                e[j] = v + pD;
                            } else {
                                e[j] = tabE[v];
                            }
                        }
                        const uint32_t wy = pack_entries(e, 0);
                        const uint32_t w2 = Y2 ? pack_entries(e, 1) : 0u;
                        int8_t* py = (int8_t*)a.y + p * a.y_pst + c;
                        int8_t* p2 =
                            Y2 ? (int8_t*)a.y2 + p * a.y2_pst + c : nullptr;
                        if (!CHK || (pok && cfull)) {
                            word_store_args(py, wy);
                            if (Y2) word_store_args(p2, w2);
                        } else if (pok) {
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                if (c + j < a.Cout) {
                                    py[j] = (int8_t)(wy >> (8 * j));
                                    if (Y2) p2[j] = (int8_t)(w2 >> (8 * j));
                                }
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i + IB < MT; ++i) {
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = acc[i + IB][j];
                psum[i] = psum[i + IB];
            }
        }
    };
    if (!hi || m0 + BM > a.M || n0 + BN > a.Cout)
        epilogue(std::true_type{}, std::false_type{});
    else if (!RES && !Y2 && (hdr.w & PLAN_IDENT))
        epilogue(std::false_type{}, std::true_type{});
    else
        epilogue(std::false_type{}, std::false_type{});
}

template <int BM, int BN, int WM, int WN, int S, int F>
bool go(const ConvArgs& b, hipStream_t st) {
    const int64_t tiles = ceil_div(b.M, BM) * ceil_div(b.Cout, BN);
    if (tiles >= ((int64_t)1 << 31)) {
        set_error("launch_gemm_stage", "grid too large");
        return false;
    }
    constexpr size_t lds = (size_t)S * 64 * (BM + BN);
    k_gemm_stage<BM, BN, WM, WN, S, (F & 1) != 0, (F & 2) != 0, (F & 4) != 0>
        <<<dim3((unsigned)tiles), 64 * WM * WN, lds, st>>>(b);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_hip_error("launch_gemm_stage", e);
        return false;
    }
    return true;
}
template <int BM, int BN, int WM, int WN, int S>
bool flags(const ConvArgs& b, hipStream_t st) {
    switch ((b.res ? 1 : 0) | (b.y2 ? 2 : 0) | (b.rowsum ? 4 : 0)) {
        case 0: return go<BM, BN, WM, WN, S, 0>(b, st);
        case 1: return go<BM, BN, WM, WN, S, 1>(b, st);
        case 2: return go<BM, BN, WM, WN, S, 2>(b, st);
        case 3: return go<BM, BN, WM, WN, S, 3>(b, st);
        case 4: return go<BM, BN, WM, WN, S, 4>(b, st);
        case 5: return go<BM, BN, WM, WN, S, 5>(b, st);
        case 6: return go<BM, BN, WM, WN, S, 6>(b, st);
        default: return go<BM, BN, WM, WN, S, 7>(b, st);
    }
}

}  // namespace

// form: 3 / 4: the 128 x 128 blocks of launch_gemm_big with that many stages;
// 16: 64 x 128 here, 6 stages; 17: 256 x 256 and 18: 256 x 128 by 8 waves, 4
// stages; 0: the choice below (times of a launch in a graph of them, us;
// against the 128 x 128 blocks with three stages).
// * 256 x 256 blocks that fill at least 85% of their rounds over the CUs (a
//   CU holds one): a step's fill and reads are 3/4 and the traffic from L2
//   half of 128 x 128 blocks': 16384x1024x1024 21.5 against 28.3,
//   4096x1024x4096 22.1 / 29.6. Not with a residual or pixel sums, whose
//   registers do not fit beside the 128 accumulators.
// * 256 x 128 blocks that fill as much, from 1024 K-bytes: 8192x4096x1024
//   36.9 / 43.6. At 384 K-bytes they gain nothing (6304x384x1152 9.0 / 8.9).
// * 64 x 128 blocks up to half a CU a 128 x 128 block (a partial column
//   block counted by its columns: 12000x32x140 5.1 / 6.6): 256x4096x4096
//   16.7 / 24.4, 5000x3072x300 12.2 / 21.4, 2000x512x700 6.0 / 8.4.
// * else 128 x 128 (6304x384x1536 11.5 / 13.7 with 64 x 128; past half a
//   block a CU the deeper pipeline gains with every operand in L2 alone:
//   6304x1536x384 10.4 / 12.2, but 19.1 / 18.5 within a network).
bool launch_gemm_stage(const ConvArgs& b, hipStream_t st, int form) {
    if (form == 0) {
        const int64_t cus = cu_count();
        auto blocks = [&](int bm, int bn) {
            return ceil_div(b.M, bm) * ceil_div(b.Cout, bn);
        };
        auto fills = [&](int64_t n) {
            return 20 * n >= 17 * cus * ceil_div(n, cus);
        };
        if (!b.res && !b.rowsum && fills(blocks(256, 256)))
            form = 17;
        else if (b.KGp >= 64 && fills(blocks(256, 128)))
            form = 18;
        else
            form = 2 * ceil_div(b.M, 128) * b.Cout <= 128 * cus ? 16 : 3;
    }
    switch (form) {
        case 16: return flags<64, 128, 2, 2, 6>(b, st);
        case 17:
            if (!b.res && !b.rowsum)
                return b.y2 ? go<256, 256, 2, 4, 4, 2>(b, st)
                            : go<256, 256, 2, 4, 4, 0>(b, st);
            [[fallthrough]];
        case 18: return flags<256, 128, 4, 2, 4>(b, st);
        default: return launch_gemm_big(b, st, form);
    }
}

}  // namespace qa
