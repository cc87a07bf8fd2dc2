// int8 MFMA convolution / GEMM: tile choice and the variants with weights
// staged in LDS (kernel templates: qa_conv_mfma.h).
#include "qa_conv_mfma.h"

namespace qa {

bool mfma_launch_lds(const ConvArgs& b, int wm, bool split, int epi,
                     hipStream_t st) {
    return launch_variant<true>(b, wm, split, epi, st);
}

// The launch form of a descriptor's arguments: whether the output (and
// residual / copy) is dense channels-last (rowio; fastio with its words on
// 4 bytes; pixel strides *_pst),
// the table epilogue when a plan applies, and the magic divisors of the
// tap decode. Returns the epilogue variant (epi when no plan applies).
int fast_io_args(const ConvArgs& a, ConvArgs& b, int epi) {
    b = a;
    // dense channels-last int8 output (and residual / copy): 4-channel
    // words of a pixel at pixel * sp + channel, 4-byte aligned
    {
        const int64_t ohw = (int64_t)a.OH * a.OW;
        // pixel stride: sp, or the row stride sn of a GEMM (one pixel a row)
        auto pst = [&](int64_t sn, int64_t sp) { return ohw == 1 ? sn : sp; };
        auto dense = [&](const void* p, int64_t sn, int64_t sc, int64_t sp) {
            return p == nullptr || (sc == 1 && (ohw == 1 || sn == ohw * sp));
        };
        auto words = [&](const void* p, int64_t sn, int64_t sp) {
            return p == nullptr ||
                   (pst(sn, sp) % 4 == 0 && (uintptr_t)p % 4 == 0);
        };
        b.rowio = a.mode == EPI_QUANT &&
                  (a.G == 1 || a.Cog % 4 == 0 || a.layout == 2) &&
                  dense(a.y, a.y_sn, a.y_sc, a.y_sp) &&
                  dense(a.res, a.res_sn, a.res_sc, a.res_sp) &&
                  dense(a.y2, a.y2_sn, a.y2_sc, a.y2_sp);
        b.fastio = b.rowio && words(a.y, a.y_sn, a.y_sp) &&
                   words(a.res, a.res_sn, a.res_sp) &&
                   words(a.y2, a.y2_sn, a.y2_sp);
        b.y_pst = pst(a.y_sn, a.y_sp);
        b.res_pst = pst(a.res_sn, a.res_sp);
        b.y2_pst = pst(a.y2_sn, a.y2_sp);
    }
    if (a.mode == EPI_QUANT && a.plan && b.rowio) epi = Q8_TABLE;
    b.mg_cb = (((uint64_t)1 << 32) + a.CB - 1) / (uint64_t)a.CB;
    b.mg_kw = (((uint64_t)1 << 32) + a.KW - 1) / (uint64_t)a.KW;
    return epi;
}

// The 128 x 128 blocks of a GEMM; 0 below 96 columns or 64 rows, which would
// leave them half empty (8x4096x4096 13.7 us on 64 x 128 blocks, 8.0 on the
// convolution's tiles, K split; 64x4096x4096 13.0 / 14.5), and for a short
// product with a residual over few rows (1020x256x256 6.7 / 5.6, 1020x384x384
// 7.2 / 6.7, 197x64x1024 5.3 / 4.9; 1020x768x768 8.1 / 11.5).
static int64_t big_blocks(const ConvArgs& b) {
    if (b.Cout < 96 || b.M < 64 ||
        (b.res && b.M < 1024 && b.KGp <= 24))
        return 0;
    return ceil_div(b.M, 128) * ceil_div(b.Cout, 128);
}

// Tile choice (from measured sweeps over the channel-block width WM and
// K-splitting on MI355X): the widest channel block that still gives about
// 1.5 waves per SIMD (0.75 when K is long, >= 9 steps: those waves are long
// enough on their own), and the 4 waves of a work-group split K only when
// even 16-channel blocks leave most SIMDs idle.
bool launch_conv_mfma(const ConvArgs& a, hipStream_t st) {
    if (a.M <= 0 || a.Cog <= 0 || a.G <= 0) return true;
    if (a.layout == 2) {
        ConvArgs b;
        if (a.mode != EPI_QUANT || a.y_code != 1) {
            set_error("launch_conv_mfma", "int8 output expected");
            return false;
        }
        const int epi = fast_io_args(a, b, Q8_GENERAL);
        return launch_conv_dw(b, b.fastio ? epi : Q8_GENERAL, st);
    }
    if (a.M >= ((int64_t)1 << 31) || a.KGp < 4 || (a.KGp & 3) ||
        a.KGp >= (1 << 16) || a.CB < 1 || a.KW < 1 ||
        (int64_t)(a.KH - 1) * a.DH >= 32768 ||
        (int64_t)(a.KW - 1) * a.DW >= 32768) {
        set_error("launch_conv_mfma", "unsupported problem size");
        return false;
    }
    int epi = a.mode;
    if (a.mode == EPI_QUANT) {
        if (a.y_code != 1) {
            set_error("launch_conv_mfma", "int8 output expected");
            return false;
        }
        epi = Q8_GENERAL;  // chosen below, once the layout is known
    }
    ConvArgs b;
    epi = fast_io_args(a, b, epi);
    // bands of output rows with operands in LDS (tile hint bit 11, with
    // wm in the low bits)
    // (ignored, like every hint, where it does not apply)
    if ((a.tile_hint & TILE_VALID) && ((a.tile_hint >> 11) & 1)) {
        const int bw = a.tile_hint & 0xff;
        if ((bw == 1 || bw == 2 || bw == 4) && conv_band_applies(b, epi, bw))
            return launch_conv_band(b, bw, st);
    }
    // weights in registers, bands in LDS (tile hint bit 12, with wm in the
    // low bits); without a hint, the default for convolutions of more than
    // one 64-byte K-step (measured the fastest choice for most 3x3 layers)
    if ((a.tile_hint & TILE_VALID) && ((a.tile_hint >> 12) & 1)) {
        const int ww = a.tile_hint & 0xf;  // bits 4..7: the band height
        if (conv_wr_applies(b, epi, ww)) return launch_conv_wr(b, ww, st);
    }
    if (!(a.tile_hint & TILE_VALID) && a.KGp > 4 && (a.KH > 1 || a.KW > 1)) {
        for (int ww = a.Cog >= 64 ? 4 : a.Cog >= 32 ? 2 : 1; ww >= 1; ww >>= 1)
            if (conv_wr_applies(b, epi, ww)) return launch_conv_wr(b, ww, st);
    }
    // narrow GEMMs / pointwise convolutions, one 16 x 16 block a wave with
    // all of its operands in registers (tile hint bit 13)
    if ((a.tile_hint & TILE_VALID) && ((a.tile_hint >> 13) & 1) &&
        gemm_narrow_applies(b, epi))
        return launch_gemm_narrow(b, st, 1 + ((a.tile_hint >> 4) & 3));
    // Without a hint (times of a launch in a graph of them, us; blocks =
    // 16-row x 64-channel blocks):
    // * a GEMM or pointwise convolution the narrow kernel takes, up to 1024
    //   blocks (2048 for K of 256 to 576
    //   with the weights in fragment order, without it 1576x576x1152 8.8 us
    //   against 5.8 staged): 4096x576x64 3.8 against 7.1 on the
    //   tiles below, 197x384x1152 3.6 / 6.4, 1024x1024x1024 6.6 / 6.5 on the
    //   staged blocks, which win past it (4096x576x1024 9.9 / 8.2); two
    //   row tiles a wave past 512 blocks (4096x576x256 5.1 / 5.6); below
    //   128 channels, where those blocks would be half empty, up to 2048
    //   (16384x576x64 5.1 / 9.5; 200704x64x32 16.4 against 12.9 on the
    //   tiles below);
    // * the staged blocks of launch_gemm_stage from 16 blocks of 128 x 128
    //   (1024x4096x256, 16 of them: 13.0 us against 14.5 on the tiles below;
    //   256x4096x4096, 64: 16.7 / 39). A pointwise convolution over dense
    //   pixels is a GEMM of its pixels (128 -> 256 channels at 32x56x56
    //   21 / 33 us, 384 -> 1280 at 32x14x14 9.9 / 21.3).
    const bool hinted = (a.tile_hint & TILE_VALID) != 0;
    const bool pointwise = b.KH == 1 && b.KW == 1 && b.SH == 1 &&
                           b.SW == 1 && b.PH == 0 && b.PW == 0 &&
                           b.OH == b.H && b.OW == b.W;
    if (!hinted && pointwise && gemm_narrow_applies(b, epi)) {
        const int64_t blocks = ceil_div(a.M, 16) * ceil_div(a.Cout, 64);
        const int K = a.KGp * 16;
        if (blocks <= 1024 ||
            (blocks <= 2048 &&
             (a.Cout < 128 || (a.wfrag && K >= 256 && K <= 576))))
            return launch_gemm_narrow(b, st, blocks > 512 ? 2 : 1);
    }
    if (pointwise && b.M > b.N && b.rowio &&
        b.x_sn == (int64_t)b.H * b.W * b.x_sp) {
        ConvArgs r = b;
        r.N = (int32_t)b.M;
        r.H = r.W = r.OH = r.OW = 1;
        r.x_sn = b.x_sp;
        if (!hinted && gemm_big_applies(r, epi) && big_blocks(r) >= 16)
            return launch_gemm_stage(r, st, 0);
    }
    // large GEMMs (tile hint bit 10 chooses them, its low byte the blocks)
    if (gemm_big_applies(b, epi)) {
        if (hinted ? (a.tile_hint >> 10) & 1 : big_blocks(b) >= 16)
            return launch_gemm_stage(b, st, hinted ? a.tile_hint & 0xff : 0);
    }
    const int64_t ntiles = ceil_div(a.M, 16);
    const int64_t simds = 4 * (int64_t)cu_count();
    auto waves = [&](int wm, bool split) {
        return ntiles * ceil_div(a.Cog, 16 * wm) * a.G * (split ? 4 : 1);
    };
    const int KS = a.KGp >> 2;
    const int wm_max =
        a.Cog <= 16 ? 1 : (a.Cog <= 32 ? 2 : (a.Cog <= 64 ? 4 : 8));
    const int64_t want = KS >= 9 ? simds * 3 / 4 : simds * 3 / 2;
    int wm = wm_max;
    while (wm > 1 && waves(wm, false) < want) wm >>= 1;
    bool split = a.layout == 0 && KS >= 4 && waves(wm, false) < simds / 2;
    // up to a wave a SIMD, K split over 32-channel blocks keeps the waves
    // and halves a wave's steps (64x4096x4096 21.1 -> 14.8 us; from 8 steps:
    // 3000x512x64 6.4 -> 6.2, but 3000x256x64 5.3 -> 5.4)
    // (wave 0 alone finishes a split tile: not with the 128-bit epilogue)
    if (epi == Q8_TABLE && a.layout == 0 && KS >= 8 && !split && wm == 1 &&
        a.Cog > 16 && waves(1, false) <= simds) {
        wm = 2;
        split = true;
    }
    // weights staged in LDS when they fit next to the tables (64 KB per
    // work-group), otherwise read from L2
    auto lds_limit = [&](int w) {
        return 65536 - 3072 - 64 - (split ? 3 * (w * 4 + 1) * 256 : 0);
    };
    auto fits = [&](int w) {
        return alds_bytes(w, a.KGp) + (a.layout == 0 ? a.KGp * 16 : 0) <=
                   lds_limit(w) &&
               (int64_t)w * 16 * a.KGp <= ALDS_CHUNKS;
    };
    bool alds = fits(wm);
    // a caller's measured choice (qa_conv_desc.tile), where it applies
    if (a.tile_hint & TILE_VALID) {
        const int hw = a.tile_hint & 0xff;
        if (hw >= 1 && hw <= wm_max && (hw & (hw - 1)) == 0) {
            wm = hw;
            split = ((a.tile_hint >> 8) & 1) && a.layout == 0;
            alds = ((a.tile_hint >> 9) & 1) && fits(wm);
        }
    }
    return alds ? mfma_launch_lds(b, wm, split, epi, st)
                : mfma_launch_l2(b, wm, split, epi, st);
}

}  // namespace qa
