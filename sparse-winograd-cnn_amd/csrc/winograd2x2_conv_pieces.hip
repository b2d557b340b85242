// Launches of the convolution with weights in pieces (winograd2x2_conv_pieces_kernel.h) and of the kernel that makes those.  Part
// of what stands in for Winograd2x2ConvComputeLauncher (winograd2x2_cublas/winograd2x2_conv/winograd2x2_conv_cuda.cu.cc:65-93).
#include "winograd2x2_conv_pieces_kernel.h"
#include "winograd2x2_conv_launch.h"

namespace swc {
namespace {

// Columns of tiles that are gone through together.  Every panel of them reads all rows of TI again, and an XCD with the same panel's
// weights reads what they take: up to seven columns, in panels about as wide, and eight where the pieces of all fit two L2s (8 MiB).
// Behind the transform, in panels of four and the rest / so: 1600x192->320 37.7 us / 33.7, 910x128->448 26.8 / 23.5, 2016x64->512 28.3 / 24.7;
// but 637x512->512 59.3 / 62.1 in one panel.
size_t panel_width(size_t tiles_n, int C)
{
    const size_t most = tiles_n == 8 && tiles_n * 64 * C * 16 * 2 * kPieces <= (8u << 20) ? 8 : 7, panels = (tiles_n + most - 1) / most;
    return (tiles_n + panels - 1) / panels;
}

template <typename Main, typename Tail = Main>
int launch_as(const float *TI, const float *Wt, const void *Wp, float *Out, size_t M, int C, int K, int nW, size_t main_m, const ConvEpilogue &ep,
              hipStream_t stream)
{
    struct Tag {};
    const int st = raise_lds_limit<Tag>(reinterpret_cast<const void *>(conv_pieces_kernel<Main, Tail>), Main::LDS_BYTES);
    if (st != SWC_OK) return st;
    static_assert(Main::LDS_BYTES >= Tail::LDS_BYTES, "the launch asks for the main tiles' LDS");
    const size_t tiles_n = (static_cast<size_t>(K) + Main::WN - 1) / Main::WN, cus = device_cus();
    size_t tail_m = 0;
    if (std::is_same<Main, Tail>::value)
        main_m = (M + Main::WM - 1) / Main::WM;
    else
        tail_m = (M - main_m * Main::WM + Tail::WM - 1) / Tail::WM;   // main_m * WM <= M
    if ((main_m + tail_m) * tiles_n >= (1ull << 31)) return SWC_ERR_BAD_DIMS;
    const size_t main_wgs = main_m * tiles_n < cus ? main_m * tiles_n : cus;
    conv_pieces_kernel<Main, Tail><<<dim3(static_cast<unsigned>(main_wgs + tail_m * tiles_n)), dim3(Main::NT), Main::LDS_BYTES, stream>>>(
        TI, Wt, static_cast<const char *>(Wp), Out, static_cast<unsigned>(M), C, K, nW, static_cast<unsigned>(main_m),
        static_cast<unsigned>(main_wgs), static_cast<unsigned>(tail_m), static_cast<unsigned>(tiles_n),
        static_cast<unsigned>(panel_width(tiles_n, C)), ep);
    return check_launch();
}

constexpr size_t kInfinityCacheBytes = 256u << 20;
constexpr size_t kStreamedPlanes = 64u << 20;   // beyond so many bytes the transform stores past the caches

size_t steps_of(int C) { return (static_cast<size_t>(C) + 31) / 32; }
size_t groups_of(int K) { return (static_cast<size_t>(K) + 63) / 64; }

// Bytes of the pieces of W [16,C,K]; 0 where the offsets within a position's 64 columns would not fit 31 bits.
size_t pieces_bytes(int C, int K, bool bf16 = false)
{
    if (C <= 0 || K <= 0 || C > (1 << 17) || steps_of(C) * groups_of(K) >= (1ull << 27)) return 0;
    return 16 * groups_of(K) * steps_of(C) * (bf16 ? 4 * 1024 : 4 * kPieces * 1024 + sizeof(float));
}

// 16-byte loads of TI and the pieces, 32-bit byte offsets into a position's planes and 31-bit ones into the output; W itself is
// read where the fp32 instructions take over.
bool pieces_eligible(const void *TI, const void *Wt, const void *Wp, const void *Out, const void *residual, size_t M, int C, int K)
{
    return C % 4 == 0 && K % 4 == 0 && aligned16(TI) && aligned16(Wt) && aligned16(Wp) && aligned16(Out) && aligned16(residual) &&
           pieces_bytes(C, K) != 0 && M * static_cast<size_t>(C) < (1ull << 29) && static_cast<size_t>(C + 128) * K < (1ull << 29) &&
           M * 16 * static_cast<size_t>(K) < (1ull << 31);
}

// bf16 operands, us (through what else runs / pieces; in brackets behind the transform).  One round of 32-row tiles, 3.6 + 3.3 per 64
// channels, from 512 channels and 512 columns on (960x512->384 44.0 / 44.8 behind the transform), against split32
//   1024x512->512 37.9 / 30.0 (47.7 / 42.5)
// where the planes are few enough for the transform to leave them in the Infinity Cache (3200x384->72, 79 MB: 30.2 / 26.7, but 52.9 / 54.8).  Below,
// some are faster (1568x256->256 27.7 / 25.6 behind the transform) and some slower (1392x128->320 17.7 / 23.2, 975x256->512 28.3 / 29.9).
// More than a round of 64-row tiles, 6.8 per 64 channels less 2 each, against ring32, from 256 channels on and with columns for four tiles, which
// share the planes
//   4410x512->256 93.4 / 76.3 (152 / 126)      6272x512->512 203 / 181 (283 / 251)        6272x256->256 53.0 / 51.1 (95 / 85)
//   5000x256->512 (132 / 95)                   3920x384->320 (126 / 98)                   4320x320->384 (113 / 96)
//   12544x128->128 31.9 / 32.1: not taken
// and whole rounds alone only where the transform streams the planes (below, behind it, 3596x256->512 65.1 / 66.5, 3195x320->512 76.4 / 78.0).
// One round of 64-row tiles is no faster than split64 (3136x256->256 28.0 / 28.4, 2700x160->320 19.8 / 22.6).
PiecesChoice choose_bf16(size_t M, int C, double c, size_t cus, size_t tiles_n)
{
    PiecesChoice best;
    if (C < 256) return best;
    auto rounds_of = [&](size_t rows, size_t high) { return static_cast<double>(((rows + high - 1) / high * tiles_n + cus - 1) / cus); };
    if (rounds_of(M, 32) <= 1) {
        if (C >= 512 && tiles_n >= 8 && M * C * 64 <= (64u << 20)) best = {PIECES_32, 0, 3.6 + 3.3 * c};
        return best;
    }
    if (rounds_of(M, 64) <= 1 || tiles_n < 4) return best;
    const double us64 = 6.8 * c - 2.0;
    best = {PIECES_64, 0, rounds_of(M, 64) * us64};
    const size_t whole = M / 64 * tiles_n / cus, main_m = whole * cus / tiles_n;
    const double us = static_cast<double>(whole) * us64 + rounds_of(M - main_m * 64, 32) * 3.6 * c;
    if (main_m * 64 < M && us < best.us) best = {PIECES_64_32, main_m, us};
    if (best.form == PIECES_64 && M * C * 64 <= kStreamedPlanes) best = PiecesChoice();
    return best;
}
}  // namespace

// A workgroup fills a CU, so a launch takes rounds of tiles over the CUs.  Measured per round, 64-row tiles: 8 us + 8.25 per 64
// channels, 1 us more in all; 32-row tiles: 3.7 + 5.9, and 1.3 + 0.4 more in all.  Where 64-row tiles make more than a round, whole
// rounds of them and the rest in one round of 32-row ones, 5 + 6.9.  Against what runs on W itself:
//   14x14x256 -> 256, batch 64    split64       57.5 us   pieces64      43.5 us
//   7x7x512 -> 512, batch 64      split32       66.5      pieces32      55.4 (58.5)
//   14x14x256 -> 256, batch 128   split64+48    97.5      pieces64      81.7
//   28x28x128 -> 128, batch 64    wide48        55.0      not taken: pieces64 takes 49.0, and 63 behind the transform
//   14x14x512 -> 512, batch 128   split64+32   337        pieces64+32  295.7
//   784x256 -> 256                direct16x64   24.5      not taken: pieces32 takes 29.3
//   56x56x64 -> 64, batch 64      tall16        74.6      not taken: pieces64 takes 71.4
// Over 209 random shapes the choice made here was 5 % faster on the geometric mean where the best of all is 6 %.  Left out: fewer than
// 64 channels (10000x32->48 14.7 us against 15.6, 3456x48->512 34 against 42), and planes that exceed the Infinity Cache and are
// read by one column of tiles, which last as long as their bytes take (21756x320->64 129 us against 143.5, 14175x512->64 124 against 129).
PiecesChoice choose_pieces(const void *TI, const void *Wt, const void *Wp, const void *Out, const void *residual, size_t M, int C, int K, bool bf16)
{
    PiecesChoice best;
    if (!pieces_eligible(TI, Wt, Wp, Out, residual, M, C, K) || (bf16 && C % 64 != 0)) return best;
    if (const char *f = forced_conv_tiling()) {
        for (int i = PIECES_32; i < PIECES_FORMS; ++i)
            if (std::string_view(f) == kPiecesNames[i]) best = {static_cast<PiecesForm>(i), M / 128, 0.0};
        return best;
    }
    const size_t cus = device_cus(), tiles_n = groups_of(K);
    if (C < 64 || (tiles_n == 1 && M * C * 64 > kInfinityCacheBytes)) return best;
    const double c = static_cast<double>(C) / 64;
    if (bf16) return choose_bf16(M, C, c, cus, tiles_n);
    auto rounds_of = [&](size_t rows, size_t high) { return static_cast<double>(((rows + high - 1) / high * tiles_n + cus - 1) / cus); };
    auto us64 = [&](double rounds) { return 1.0 + rounds * (8.0 + 8.25 * c); };
    // Streamed planes come from memory, which one column of 32-row tiles after the other does not hide: 14 us (2100x512->96 52 us, behind the
    // transform 81; split32 60 and 76).
    const bool streamed = M * C * 64 > kStreamedPlanes;
    const double us32 = 1.3 + 0.4 * c + rounds_of(M, 32) * (3.7 + 5.9 * c) + (streamed ? 14.0 : 0.0);
    best = {PIECES_64, 0, us64(rounds_of(M, 64))};
    if (us32 < best.us) best = {PIECES_32, 0, us32};
    const size_t whole = M / 64 * tiles_n / cus, main_m = whole * cus / tiles_n;
    if (whole > 0 && main_m * 64 < M) {
        const double us = us64(static_cast<double>(whole)) + rounds_of(M - main_m * 64, 32) * (5.0 + 6.9 * c);
        if (us < best.us) best = {PIECES_64_32, main_m, us};
    }
    // The above holds for planes that the Infinity Cache has; behind the transform that wrote them larger ones come from memory, a half step
    // ahead only: 0.12 us for every MB beyond 50 (behind the transform 28x28x128 at batch 64 takes 63 us, wide48 62; 14x14x512 at batch 128 328, split64+32 346).
    const double mb = static_cast<double>(M) * C * 64 / 1e6;
    if (mb > 50) best.us += 0.12 * (mb - 50);
    return best;
}

int launch_pieces(const PiecesChoice &pick, bool bf16, const float *TI, const float *Wt, const void *Wp, float *Out, size_t M, int C, int K, int nW,
                  const float *scale, const float *shift, const float *residual, int residual_relu, hipStream_t s)
{
    ConvEpilogue ep;
    ep.scale = scale;
    ep.shift = shift;
    ep.residual = residual;
    ep.residual_relu = residual_relu;
    const bool ragged = C % 16 != 0, deep = steps_of(C) % 2 == 0 && !ragged;
    if (bf16) {
        using D32 = PiecesCfg<1, 4, false, 1>;   // C % 64 == 0: twice the half steps on their way
        using D64 = PiecesCfg<2, 4, false, 1>;
        switch (pick.form) {
            case PIECES_64: return launch_as<D64>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s);
            case PIECES_32: return launch_as<D32>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s);
            case PIECES_64_32: return launch_as<D64, D32>(TI, Wt, Wp, Out, M, C, K, nW, pick.main_m, ep, s);
            default: return SWC_ERR_UNSUPPORTED;
        }
    }
    switch (pick.form) {
        case PIECES_64:
            return ragged ? launch_as<PiecesCfg<2, 2, true>>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s)
                          : launch_as<PiecesCfg<2, 2, false>>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s);
        case PIECES_32:
            return ragged ? launch_as<PiecesCfg<1, 2, true>>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s)
                   : deep ? launch_as<PiecesCfg<1, 4, false>>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s)
                          : launch_as<PiecesCfg<1, 2, false>>(TI, Wt, Wp, Out, M, C, K, nW, 0, ep, s);
        case PIECES_64_32:
            return ragged ? launch_as<PiecesCfg<2, 2, true>, PiecesCfg<1, 2, true>>(TI, Wt, Wp, Out, M, C, K, nW, pick.main_m, ep, s)
                          : launch_as<PiecesCfg<2, 2, false>, PiecesCfg<1, 2, false>>(TI, Wt, Wp, Out, M, C, K, nW, pick.main_m, ep, s);
        default: return SWC_ERR_UNSUPPORTED;
    }
}

namespace {

template <int NP>
int make_pieces(const float *Weight, void *Pieces, int C, int K, swc_stream_t stream)
{
    if (Weight == nullptr || Pieces == nullptr) return SWC_ERR_NULL_POINTER;
    if (C <= 0 || K <= 0 || pieces_bytes(C, K) == 0) return SWC_ERR_BAD_DIMS;
    if (!aligned16(Pieces)) return SWC_ERR_UNSUPPORTED;
    const unsigned groups = static_cast<unsigned>(groups_of(K)), steps = static_cast<unsigned>(steps_of(C));
    weight_pieces_kernel<NP><<<dim3(16 * groups * steps), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        Weight, static_cast<char *>(Pieces), C, K, groups, steps);
    return check_launch();
}

}  // namespace
}  // namespace swc

extern "C" size_t swc_winograd2x2_weight_pieces_bytes(int C, int K) { return swc::pieces_bytes(C, K); }
extern "C" size_t swc_winograd2x2_weight_pieces_bf16_bytes(int C, int K) { return swc::pieces_bytes(C, K, true); }

extern "C" int swc_winograd2x2_weight_pieces(const float *Weight, void *Pieces, int C, int K, swc_stream_t stream)
{
    return swc::make_pieces<swc::kPieces>(Weight, Pieces, C, K, stream);
}

extern "C" int swc_winograd2x2_weight_pieces_bf16(const float *Weight, void *Pieces, int C, int K, swc_stream_t stream)
{
    return swc::make_pieces<1>(Weight, Pieces, C, K, stream);
}
