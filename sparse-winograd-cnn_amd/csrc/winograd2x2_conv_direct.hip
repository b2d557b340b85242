// Launches of the small-grid convolution (winograd2x2_conv_direct_kernel.h).  Part of what stands in for
// Winograd2x2ConvComputeLauncher (winograd2x2_cublas/winograd2x2_conv/winograd2x2_conv_cuda.cu.cc:65-93).
#include "winograd2x2_conv_direct_kernel.h"
#include "winograd2x2_conv_launch.h"

namespace swc {
namespace {

template <typename Cfg>
int launch_as(const float *TI, const float *Wt, float *Out, size_t M, int C, int K, int nW, const ConvEpilogue &ep, hipStream_t stream)
{
    struct Tag {};
    const int st = raise_lds_limit<Tag>(reinterpret_cast<const void *>(conv_direct_kernel<Cfg>), Cfg::LDS_BYTES);
    if (st != SWC_OK) return st;
    const size_t tiles_m = (M + Cfg::WM - 1) / Cfg::WM, tiles_n = (static_cast<size_t>(K) + Cfg::WN - 1) / Cfg::WN;
    if (tiles_m * tiles_n >= (1ull << 31)) return SWC_ERR_BAD_DIMS;
    conv_direct_kernel<Cfg><<<dim3(static_cast<unsigned>(tiles_m * tiles_n)), dim3(Cfg::NT), Cfg::LDS_BYTES, stream>>>(
        TI, Wt, Out, static_cast<unsigned>(M), C, K, nW, static_cast<unsigned>(tiles_m), static_cast<unsigned>(tiles_n),
        static_cast<size_t>(K) > M ? 1 : 0, ep);
    return check_launch();
}

template <bool BF16>
int launch_form(DirectForm form, const float *TI, const float *Wt, float *Out, size_t M, int C, int K, int nW, const ConvEpilogue &ep,
                hipStream_t s)
{
    switch (form) {
        // Blocks of 64 indices as they come are the only form that takes single columns.  bf16 operands: they also do with one block less where
        // C ends in the second half of one (behind the transform, 196x100->128 10.3 us against 10.9 in turned blocks of 32, 784x124->32
        // 10.9 / 11.7; but 196x96->128 10.7 / 9.7, 196x72->128 9.7 / 9.5).
        case DIRECT_16X16:
            return K % 4 == 0 && aligned16(Wt) && !(BF16 && C % 64 > 32)
                       ? launch_as<DirectCfg<1, 1, 8, BF16, 3, true>>(TI, Wt, Out, M, C, K, nW, ep, s)
                       : launch_as<DirectCfg<1, 1, 16, BF16>>(TI, Wt, Out, M, C, K, nW, ep, s);
        case DIRECT_16X32: return launch_as<DirectCfg<1, 2, 8, BF16, 3, true>>(TI, Wt, Out, M, C, K, nW, ep, s);
        case DIRECT_16X64: return launch_as<DirectCfg<1, 4, 8, BF16, 2, true>>(TI, Wt, Out, M, C, K, nW, ep, s);
        case DIRECT_32X64: return launch_as<DirectCfg<2, 4, BF16 ? 8 : 4, BF16, BF16 ? 1 : 2, !BF16>>(TI, Wt, Out, M, C, K, nW, ep, s);
        default: return SWC_ERR_UNSUPPORTED;
    }
}

}  // namespace

// 16-byte loads of TI and 32-bit byte offsets into a position's planes (a partial block reaches past the end by
// less than 128 rows of W before its lanes are masked).
static bool direct_eligible(const void *TI, size_t M, int C, int K)
{
    return C % 4 == 0 && aligned16(TI) && M * static_cast<size_t>(C) < (1ull << 29) && static_cast<size_t>(C + 128) * K < (1ull << 29);
}

// A workgroup fills a CU (sixteen waves of up to 128 registers), so a launch takes whole rounds over the CUs.  Measured
// per round, fp32: 3.1 us + 1.45 per 64 channels for 16x16 tiles, 3.5 + 2.5 for 16x32, 4.2 + 4.2 for 16x64, 5.5 + 7.6 for
// 32x64 (with bf16 operands 3 + 1.4, 3.2 + 1.95, 3.6 + 2.25, 5 + 5.2), so the smallest tile that needs one round wins.
// A round more, with the device full, takes 1.0 + 2.2, 1.6 + 3.2, 2.5 + 5.1 and 6.1 + 8.4 (bf16 0.9 + 2.1, 1.3 + 3.3, 1.8 + 3.7, 3.6 + 5.7;
// 500 fp32 and 700 bf16 shapes of 2 to 12 rounds, nine in ten within 10 %).  Counted like the first, 16x64 tiles were taken where 32x64 ones
// are faster (bf16, 5483x208->256 90.5 / 63.0 us, 4608x72->384 45.8 / 38.7), and 16x32 ones instead of split32 (2427x100->96 15.3 / 10.3).
// With a row of TI and a column of W per lane the first three were 3.2 + 2.4, 3.4 + 3.6 and 4 + 4.8 (49x512->512 22.9 -> 14.8 us,
// 196x512->512 34.1 -> 25.5, 784x64->64 5.7 -> 4.65), and blocks of 64 indices instead of 32 spill at three in flight (21.4).
// The ring kernels take 4.3 + 8.9 us per 64 channels at best (bf16 6 + 9) and hold that up to one 64x64 tile per CU:
// beyond one round of 32x64 tiles they are as fast or faster (784x64->64: 13.4 -> 5.7 us; 49x512->512: 75.6 -> 14.8;
// 784x256->256: 41.6 -> 21.4; 1024x512->512: 76.3 -> 68).  short16 deals out the same 32x64 tiles at four waves each and
// two or three to a CU; below 256 channels it is the faster one (1024 to 8192 rows, 64 channels: 13.3 to 14.8 us against
// 14.5 to 15.9; 128: 22.5 to 24.2 against 22.7 to 25.2; 192: 32.0 against 32.5; 256: 41.0 against 40.8), while ring32, which takes
// the other channel counts, is not (96 channels: 31 against 20).  Where only the
// synchronous kernel could run (44 us for 104x72->48, 6.6 here) every round is worth it, except that single columns
// (K % 4 != 0 or W unaligned) come in 16x16 tiles only.
DirectForm choose_direct(const void *TI, const void *Wt, size_t M, int C, int K, bool ring, bool short16, bool bf16, double *us)
{
    *us = 1e30;
    if (!direct_eligible(TI, M, C, K)) return DIRECT_NONE;
    const bool wide = K % 4 == 0 && aligned16(Wt);   // 8- and 16-byte loads along the columns
    if (const char *f = forced_conv_tiling()) {
        for (int i = DIRECT_16X16; i < DIRECT_FORMS; ++i)
            if (std::string_view(f) == kDirectNames[i] && (wide || i == DIRECT_16X16)) {
                *us = 0;
                return static_cast<DirectForm>(i);
            }
        return DIRECT_NONE;
    }
    static constexpr struct { size_t rows, cols; double base[2], per64[2], more[2], more64[2]; } kForms[DIRECT_FORMS] = {
        {}, {16, 16, {3.1, 3.0}, {1.45, 1.4}, {1.0, 0.9}, {2.2, 2.1}}, {16, 32, {3.5, 3.2}, {2.5, 1.95}, {1.6, 1.3}, {3.2, 3.3}},
        {16, 64, {4.2, 3.6}, {4.2, 2.25}, {2.5, 1.8}, {5.1, 3.7}}, {32, 64, {5.5, 5.0}, {7.6, 5.2}, {6.1, 3.6}, {8.4, 5.7}}};
    const size_t cus = device_cus();
    DirectForm best = DIRECT_NONE;
    for (int i = DIRECT_16X16; i <= (wide ? DIRECT_32X64 : DIRECT_16X16); ++i) {
        const size_t wgs = (M + kForms[i].rows - 1) / kForms[i].rows * ((K + kForms[i].cols - 1) / kForms[i].cols);
        const size_t rounds = (wgs + cus - 1) / cus;
        if (rounds > (ring ? 1 : wide ? ~size_t(0) : 4)) continue;
        if (i == DIRECT_32X64 && short16 && C < 256) continue;
        // the three that turn their operands round take as long for a last block of 32 channels that is not full
        const double per = i == DIRECT_32X64 ? static_cast<double>(C) / 64 : static_cast<double>((C + 31) / 32) / 2;
        const double this_us = kForms[i].base[bf16] + kForms[i].per64[bf16] * per + (rounds - 1) * (kForms[i].more[bf16] + kForms[i].more64[bf16] * per);
        if (this_us < *us) {
            *us = this_us;
            best = static_cast<DirectForm>(i);
        }
    }
    return best;
}

int launch_direct(DirectForm form, bool bf16, const float *TI, const float *Wt, float *Out, size_t M, int C, int K, int nW,
                  const float *scale, const float *shift, const float *residual, int residual_relu, hipStream_t stream)
{
    ConvEpilogue ep;
    ep.scale = scale;
    ep.shift = shift;
    ep.residual = residual;
    ep.residual_relu = residual_relu;
    return bf16 ? launch_form<true>(form, TI, Wt, Out, M, C, K, nW, ep, stream)
                : launch_form<false>(form, TI, Wt, Out, M, C, K, nW, ep, stream);
}

}  // namespace swc
