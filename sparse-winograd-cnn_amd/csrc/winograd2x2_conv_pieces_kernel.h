// The Winograd convolution on the bf16 matrix instructions, fp32 operands in three bf16 pieces, the weights taken apart
// beforehand (device code).  See winograd2x2_conv.hip for what it replaces in the reference.
#pragma once

#include "winograd2x2_conv_planes.h"

namespace swc {
namespace {

// As in winograd2x2_conv_split_kernel.h a value is h + m + l, each the bf16 value nearest to what the ones before leave, six of
// the nine products count, and eight waves multiply two of the sixteen positions each, one after the other, a tile of 32*TM rows
// x 64 columns.  What differs:
//
// The weights arrive in pieces (weight_pieces_kernel), in the order in which a wave reads them: their loads are whole kilobytes
// and they cost no vector instruction.  An MFMA keeps the vector unit from issuing for about 16 of its 32 clocks (12 of 16 for
// the 16x16 shape), so that a 32x32x16 one leaves room for four vector instructions: a half step of 16 indices is 24 of them beside 101
// (88 take TI apart, 12 look at its size), where taking both operands apart would be 180.
//
// The five small products of a tile are summed by themselves over the whole position and added to the sums of h.h once: 64
// registers more, no additions in the loop, and the result is nearer to float64 (256 channels, 30 % of the weights kept:
// 0.94e-7 -> 0.69e-7; 512: 1.13e-7 -> 0.75e-7; the fp32 instructions 1.3 to 2.6e-7).
//
// A workgroup takes tile after tile; the operands of the next one's first steps are on their way while the outputs of the one
// before are put together (28x28x128 at batch 64, planes in the Infinity Cache: 50.2 -> 48.6 us).
//
// Where the fp32 instructions take over is what it was there: operands above 2^30, sums below 2^-75 and not zero, or not finite.
//
// The loop is bound by the matrix pipes' clock (2.1 GHz under this load) and by what the L2 hands a CU: 20 KiB for the 48 MFMAs of
// a wave's step, of 56 bytes a clock at most.  With both operands in the L1 (timed on a copy) 14x14x256 at batch 64 takes 36.8 us
// instead of 43.6.  With 32 rows a step is 16 KiB for 24 MFMAs, which is bound by the L2 alone; twice the half steps on their way
// (HB 4, registers allow it there) make 7x7x512 at batch 64 57.4 -> 55.3 us.
//
// bf16 operands are the same with one piece (NP 1) and one product: no second look at the operands, whose rounding the caller asked
// for, and the sums of even and odd half steps by themselves, so that a sum is rounded as often as with 32 indices to an instruction.
// What bounds that form is not established: prepared weights take a quarter off the bytes that a CU reads, but one round of 64-row
// tiles takes as long with them as without (3136x256->256 28.0 us on W, 28.4).
constexpr int kPieces = 3;

template <int TM_, int HB_, bool RAGGED_, int NP_ = kPieces>
struct PiecesCfg {
    static constexpr int NP = NP_;
    static constexpr int TM = TM_, TN = 2;
    static constexpr int HB = HB_, RA = HB / 2;              // half steps of weights and of TI on their way
    static constexpr bool RAGGED = RAGGED_;                  // C is no multiple of 16
    static constexpr int WM = 32 * TM, WN = 64;
    static constexpr int E = WM * WN;
    static constexpr int NT = 512;
    static constexpr int STAGE = WM * 16;                    // floats a wave turns A round in: all rows x 16 indices
    static constexpr int LDS_BYTES = 8 * (E + STAGE) * 4;
    static constexpr int HALF_BYTES = TN * NP * 1024;             // prepared weights of 16 indices x 64 columns
    static_assert(LDS_BYTES <= 160 * 1024, "a CU has 160 KiB of LDS");
};

// Eight values into pieces, each the bf16 value nearest to what the ones before leave.
template <int NP>
__device__ __forceinline__ void pieces_of8(const floatx4 &u, const floatx4 &w, intx4 (&out)[NP])
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        floatx2 x = q < 2 ? floatx2{u[2 * q], u[2 * q + 1]} : floatx2{w[2 * q - 4], w[2 * q - 3]};
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const bf16x2 h = __builtin_convertvector(x, bf16x2);
            out[p][q] = __builtin_bit_cast(int, h);
            if (p + 1 == NP) break;
            x[0] -= static_cast<float>(h[0]);
            x[1] -= static_cast<float>(h[1]);
        }
    }
}

constexpr float kPieceTiny = 0x1p-75f, kPieceLarge = 0x1p30f;   // see winograd2x2_conv_split_kernel.h

// What a wave multiplies: the rows of a tile at one position with the weights of 64 columns.
struct PieceTile {
    unsigned m0, rows;   // first row, rows inside
    unsigned tn_id;      // column group
};

// A workgroup's tiles: `count` of them, `tile_of(i)` the i-th.
template <typename Cfg, typename TileOf>
__device__ __forceinline__ void pieces_tiles(const float *__restrict__ TI, const float *__restrict__ Wt, const char *__restrict__ Wp,
                                             float *__restrict__ Out, unsigned M, int C, int K, int nW, unsigned count, TileOf tile_of,
                                             float *P, const ConvEpilogue ep)
{
    constexpr int TM = Cfg::TM, TN = Cfg::TN, E = Cfg::E, NP = Cfg::NP;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, li = lane & 31, lg = lane >> 5;
    const unsigned groups = (static_cast<unsigned>(K) + 63) / 64, steps = (static_cast<unsigned>(C) + 31) / 32;
    const int halves = static_cast<int>(2 * steps);   // a multiple of HB

    const size_t a_plane = static_cast<size_t>(M) * C, b_plane = static_cast<size_t>(C) * K;
    const unsigned p_bytes = 2 * steps * Cfg::HALF_BYTES;
    unsigned a_off[2 * TM];   // within the tile; rows beyond its last one read as zero
#pragma unroll
    for (int j = 0; j < 2 * TM; ++j) a_off[j] = (16 * j + lane / 4) * static_cast<unsigned>(C) * 4u + lane % 4 * 16u;
    float *const stage = P + 8 * E + wave * Cfg::STAGE;
    const int stage_in = lane / 4 * 16 + ((lane % 4) ^ (lane / 8 % 4)) * 4;   // + 256 for each 16 rows more
    const int stage_out[2] = {li * 16 + ((2 * lg) ^ (li / 2 % 4)) * 4, li * 16 + ((2 * lg + 1) ^ (li / 2 % 4)) * 4};
    auto a_desc_of = [&](const PieceTile &t, int pos, bool live) __attribute__((always_inline)) {
        return make_rsrc(TI + pos * a_plane + static_cast<size_t>(t.m0) * C, live ? t.rows * static_cast<unsigned>(C) * 4u : 0u);
    };
    auto p_desc_of = [&](const PieceTile &t, int pos, bool live) __attribute__((always_inline)) {
        return make_rsrc(Wp + (static_cast<size_t>(pos) * groups + t.tn_id) * p_bytes, live ? p_bytes : 0u);
    };
    PieceTile t = tile_of(0);

    constexpr int HB = Cfg::HB, RA = Cfg::RA;
    floatx4 ra[RA][2 * TM];
    intx4 bs[HB][TN][NP];
    auto load_a = [&](auto slot_tag, const __amdgpu_buffer_rsrc_t desc, int k0) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_tag)::value;
        if constexpr (Cfg::RAGGED) {   // the last indices, C % 4 == 0; what lies beyond reads as zero
            const bool in = k0 + lane % 4 * 4 < C;
#pragma unroll
            for (int j = 0; j < 2 * TM; ++j)
                ra[slot][j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(desc, static_cast<int>(in ? a_off[j] : kOutOfRange), k0 * 4, 0));
        } else {
#pragma unroll
            for (int j = 0; j < 2 * TM; ++j)
                ra[slot][j] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(desc, static_cast<int>(a_off[j]), k0 * 4, 0));
        }
    };
    auto load_b = [&](auto buf_tag, const __amdgpu_buffer_rsrc_t desc, int half) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_tag)::value;
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int p = 0; p < NP; ++p)
                bs[buf][tn][p] = __builtin_bit_cast(intx4, __builtin_amdgcn_raw_buffer_load_b128(
                                                               desc, lane * 16, half * Cfg::HALF_BYTES + (tn * NP + p) * 1024, 0));
    };

    floatx16 acc[TM][TN], crs[TM][TN];
    auto zero_acc = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[tm][tn][r] = 0.f, crs[tm][tn][r] = 0.f;
    };
    auto park = [&]() __attribute__((always_inline)) {
        // accumulator register r of lane (lg, li): row 8*(r/4) + 4*lg + r%4 of the tile, columns 2*li + tn of the wave's
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const floatx2 v = {acc[tm][0][r], acc[tm][1][r]};
                *reinterpret_cast<floatx2 *>(&P[wave * E + (tm * 32 + 8 * (r / 4) + 4 * lg + r % 4) * 64 + 2 * li]) = v;
            }
    };
    [[maybe_unused]] auto again_in_fp32 = [&](const __amdgpu_buffer_rsrc_t a_desc, const __amdgpu_buffer_rsrc_t b_desc) __attribute__((always_inline)) {
        zero_acc();
        const int n = static_cast<int>(t.tn_id) * Cfg::WN + 2 * li;
        const unsigned b_off = (static_cast<unsigned>(lg * 4) * K + (n + 2 <= K ? n : K - 2)) * 4u;
        unsigned row_off[TM];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) row_off[tm] = ((tm * 32 + li) * static_cast<unsigned>(C) + lg * 4) * 4u;
        for (int k0 = 0; k0 < C; k0 += 8) {
            const bool in = k0 + lg * 4 < C;
            floatx2 b[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
                b[t] = __builtin_bit_cast(floatx2, __builtin_amdgcn_raw_buffer_load_b64(
                                                       b_desc, static_cast<int>(in ? b_off : kOutOfRange), (k0 + t) * K * 4, 0));
#pragma unroll
            for (int tm = 0; tm < TM; ++tm) {
                const floatx4 a = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                  a_desc, static_cast<int>(in ? row_off[tm] : kOutOfRange), k0 * 4, 0));
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], b[t][tn], acc[tm][tn], 0, 0, 0);
            }
        }
    };

    // the largest magnitudes of W, one for every 32 indices x 64 columns, behind the pieces
    [[maybe_unused]] const float *const w_most = reinterpret_cast<const float *>(Wp + static_cast<size_t>(16) * groups * p_bytes);

    floatx4 fr[TM][2];   // raw operands of the half step behind the one multiplied
    auto put_a = [&](auto slot_tag) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_tag)::value;
#pragma unroll
        for (int j = 0; j < 2 * TM; ++j) *reinterpret_cast<floatx4 *>(stage + stage_in + 256 * j) = ra[slot][j];
        asm volatile("" ::: "memory");   // other lanes' values are read back
        __builtin_amdgcn_wave_barrier();
    };
    auto get_a = [&](int tm) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 2; ++q) fr[tm][q] = *reinterpret_cast<const floatx4 *>(stage + stage_out[q] + 512 * tm);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    };
    intx4 as[2][NP];
    float most = 0.f;    // the largest magnitude among the operands of a lane
    auto take_a = [&](int tm, int to) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < (NP == 1 ? 0 : 2); ++q)
#pragma unroll
            for (int i = 0; i < 4; i += 2)
                most = __builtin_fmaxf(__builtin_fmaxf(most, __builtin_fabsf(fr[tm][q][i])), __builtin_fabsf(fr[tm][q][i + 1]));
        pieces_of8<NP>(fr[tm][0], fr[tm][1], as[to]);
    };
    auto multiply = [&](int tm, int from, auto buf_tag) __attribute__((always_inline)) {
        constexpr int buf = decltype(buf_tag)::value;
        auto mfma = [](const intx4 &x, const intx4 &y, const floatx16 &c) __attribute__((always_inline)) {
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), c, 0, 0, 0);
        };
        const intx4(&a)[NP] = as[from];
        if constexpr (NP == 1) {
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
                floatx16 &sum = buf % 2 == 0 ? acc[tm][tn] : crs[tm][tn];
                sum = mfma(a[0], bs[buf][tn][0], sum);
            }
            return;
        }
        constexpr int order[5][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};   // l.h, h.l, m.m, m.h, h.m
#pragma unroll
        for (int i = 0; i < 5; ++i)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) crs[tm][tn] = mfma(a[order[i][0] % NP], bs[buf][tn][order[i][1] % NP], crs[tm][tn]);
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = mfma(a[0], bs[buf][tn][0], acc[tm][tn]);
    };
    auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < (NP == 1 ? 0 : 6 * TN); ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // a matrix instruction,
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);   // five vector ones
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    __amdgpu_buffer_rsrc_t a_desc = a_desc_of(t, wave, true), p_desc = p_desc_of(t, wave, true);
    static_for<RA>([&](auto j_tag) __attribute__((always_inline)) { load_a(j_tag, a_desc, 16 * decltype(j_tag)::value); });
    static_for<HB>([&](auto j_tag) __attribute__((always_inline)) { load_b(j_tag, p_desc, decltype(j_tag)::value); });
    put_a(std::integral_constant<int, 0>{});
    get_a(0);
    if (TM > 1) get_a(1);
    load_a(std::integral_constant<int, 0>{}, a_desc, 16 * RA);
    take_a(0, 0);

    // The multiplication of half a step (16 indices) runs beside the taking apart of the next rows; operands are loaded into
    // registers that have just been used, behind a position's last step those of the wave's second position.
    auto position = [&](const __amdgpu_buffer_rsrc_t a_next, const __amdgpu_buffer_rsrc_t p_next, bool dead_end, int pos) __attribute__((always_inline)) {
        zero_acc();
        float most_here = 0.f;
        for (int h0 = 0; h0 < halves; h0 += HB) {
            int left = halves - h0;
            asm("" : "+s"(left));   // one copy of the loop's body
            const bool turn = left == HB, dead = turn && dead_end;
            const __amdgpu_buffer_rsrc_t an = turn ? a_next : a_desc, pn = turn ? p_next : p_desc;
            const int hn = turn ? 0 : h0 + HB;
            static_for<HB>([&](auto ks_tag) __attribute__((always_inline)) {
                constexpr int ks = decltype(ks_tag)::value, ahead = ks + 1 + RA;
                constexpr std::integral_constant<int, (ks + 1) % RA> slot{};
                put_a(slot);
                get_a(0);
                if constexpr (ahead < HB)
                    load_a(slot, a_desc, (h0 + ahead) * 16);
                else
                    load_a(slot, an, dead ? 0 : (hn + ahead - HB) * 16);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (TM > 1) {
                    take_a(1, 1);
                    multiply(0, 0, ks_tag);
                    interleave();
                    get_a(1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (ks == HB - 1) {
                    most_here = most;
                    if (turn) most = 0.f;
                }
                if constexpr (TM > 1) {
                    take_a(0, 0);
                    multiply(1, 1, ks_tag);
                } else {
                    multiply(0, ks % 2, ks_tag);
                    take_a(0, 1 - ks % 2);
                }
                interleave();
                load_b(ks_tag, pn, dead ? 0 : hn + ks);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        if constexpr (NP == 1) {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[tm][tn][r] = acc[tm][tn][r] + crs[tm][tn][r];
            return;
        }
        float none = 0.f, low = __builtin_inff();   // NaN where a sum is not finite; the smallest sum
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[tm][tn][r] = acc[tm][tn][r] + crs[tm][tn][r];
                    none = __builtin_fmaf(acc[tm][tn][r], 0.f, none);
                }
#pragma unroll
                for (int r = 0; r < 16; r += 2)
                    low = __builtin_fminf(low, __builtin_fminf(__builtin_fabsf(acc[tm][tn][r]), __builtin_fabsf(acc[tm][tn][r + 1])));
            }
        bool odd = none != 0.f || most_here > kPieceLarge;
        const float *const wm = w_most + (static_cast<size_t>(pos) * groups + t.tn_id) * steps;
        for (unsigned s = lane; s < steps; s += 64) odd |= wm[s] > kPieceLarge;
        if (__any(low < kPieceTiny)) {   // zero or tiny: the one is fine
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                    for (int r = 0; r < 16; ++r) odd |= acc[tm][tn][r] != 0.f && __builtin_fabsf(acc[tm][tn][r]) < kPieceTiny;
        }
        if (__any(odd)) again_in_fp32(a_desc, make_rsrc(Wt + pos * b_plane, static_cast<unsigned>(b_plane) * 4u));
    };

    // One copy of the loop for both passes and all tiles: a kernel's first run through its code waits for every line of it.
    for (unsigned i = 0;;) {
        const bool more = i + 1 < count;
        const PieceTile next = more ? tile_of(i + 1) : t;
#pragma unroll 1
        for (int pass = 0;; ++pass) {
            const bool last = pass == 1, live = !last || more;
            // behind the last position nothing is loaded: descriptors of no bytes
            const __amdgpu_buffer_rsrc_t a_next = a_desc_of(last ? next : t, last ? wave : wave + 8, live),
                                         p_next = p_desc_of(last ? next : t, last ? wave : wave + 8, live);
            position(a_next, p_next, !live, wave + 8 * pass);
            a_desc = a_next;
            p_desc = p_next;
            if (last) break;
            park();
        }
        OutputPlanes<Cfg> out;
        __syncthreads();
        out.template combine<0>(P);
        __syncthreads();
        park();
        __syncthreads();
        out.template combine<1>(P);
        if (more) __syncthreads();
        out.store(Out, M, K, nW, t.m0, t.rows, static_cast<int>(t.tn_id) * Cfg::WN, ep);
        if (!more) break;
        t = next;
        ++i;
    }
}

// Tile `id` of those that cover the rows from row0 on, end exclusive.  The 32 workgroups of an XCD have consecutive tiles: they
// share their L2's copy of the rows and the weights, `wide` columns at a time (see panel_width).
template <typename Cfg>
__device__ __forceinline__ PieceTile piece_tile(unsigned id, unsigned tiles_m, unsigned tiles_n, unsigned wide, unsigned row0, unsigned end)
{
    const unsigned panel = id / (tiles_m * wide), width = tiles_n - panel * wide < wide ? tiles_n - panel * wide : wide;
    const unsigned in = id - panel * tiles_m * wide, m0 = row0 + in / width * Cfg::WM;
    return PieceTile{m0, end - m0 < Cfg::WM ? end - m0 : Cfg::WM, panel * wide + in % width};
}

// The first main_wgs workgroups take the main_m * tiles_n tiles of Main, one after the other where there are more of them, those
// behind them the rows that are left in the lower tiles of Tail.
template <typename Main, typename Tail>
__global__ __launch_bounds__(Main::NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void conv_pieces_kernel(
    const float *__restrict__ TI, const float *__restrict__ Wt, const char *__restrict__ Wp, float *__restrict__ Out, unsigned M, int C,
    int K, int nW, unsigned main_m, unsigned main_wgs, unsigned tail_m, unsigned tiles_n, unsigned wide, ConvEpilogue ep)
{
    extern __shared__ __attribute__((aligned(16))) float P[];   // [8][E] and the staging tiles
    const unsigned n_main = main_m * tiles_n;
    const unsigned main_rows = main_m * Main::WM < M ? main_m * Main::WM : M;
    if (std::is_same<Main, Tail>::value || blockIdx.x < main_wgs) {
        auto tile_of = [&](unsigned i) __attribute__((always_inline)) {
            const unsigned before = i * main_wgs, here = n_main - before < main_wgs ? n_main - before : main_wgs;
            return piece_tile<Main>(before + xcd_swizzle(blockIdx.x, here), main_m, tiles_n, wide, 0, main_rows);
        };
        pieces_tiles<Main>(TI, Wt, Wp, Out, M, C, K, nW, (n_main - blockIdx.x + main_wgs - 1) / main_wgs, tile_of, P, ep);
    } else if constexpr (!std::is_same<Main, Tail>::value) {
        auto tile_of = [&](unsigned) __attribute__((always_inline)) {
            return piece_tile<Tail>(xcd_swizzle(blockIdx.x - main_wgs, tail_m * tiles_n), tail_m, tiles_n, wide, main_rows, M);
        };
        pieces_tiles<Tail>(TI, Wt, Wp, Out, M, C, K, nW, 1, tile_of, P, ep);
    }
}

// W [16,C,K] into pieces, in the order in which a wave reads them: [position][64 columns][16 indices][tn][piece][lane][8], and
// behind them the largest magnitude of every 32 indices x 64 columns.  A workgroup takes those of one position; what lies
// beyond C or K is zero.  With one piece there are no magnitudes.  Bound by memory: 10 bytes a value, 2.5 us and 1.2 us for every 2^20 values (512x512: 7.6 us).
template <int NP>
__global__ __launch_bounds__(256) void weight_pieces_kernel(const float *__restrict__ Wt, char *__restrict__ Wp, int C, int K, unsigned groups,
                                                            unsigned steps)
{
    __shared__ float most_of[4];
    const unsigned s = blockIdx.x % steps, pg = blockIdx.x / steps, g = pg % groups, pos = pg / groups;
    const int lane = threadIdx.x & 63, li = lane & 31, lg = lane >> 5, tn = threadIdx.x >> 6 & 1, ks = threadIdx.x >> 7;
    const int n = static_cast<int>(g * 64) + 2 * li + tn, k = static_cast<int>(s * 32) + 16 * ks + 8 * lg;
    floatx4 v[2];
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i / 4][i % 4] = n < K && k + i < C ? Wt[(static_cast<size_t>(pos) * C + k + i) * K + n] : 0.f;
        most = __builtin_fmaxf(most, __builtin_fabsf(v[i / 4][i % 4]));
    }
    intx4 out[NP];
    pieces_of8<NP>(v[0], v[1], out);
    char *const to = Wp + (((static_cast<size_t>(pg) * steps + s) * 2 + ks) * 2 + tn) * (NP * 1024) + lane * 16;
#pragma unroll
    for (int p = 0; p < NP; ++p) *reinterpret_cast<intx4 *>(to + p * 1024) = out[p];
    if (NP == 1) return;
#pragma unroll
    for (int d = 32; d > 0; d /= 2) most = __builtin_fmaxf(most, __shfl_xor(most, d));
    if (lane == 0) most_of[threadIdx.x >> 6] = most;
    __syncthreads();
    if (threadIdx.x == 0) {
        float *const w_most = reinterpret_cast<float *>(Wp + static_cast<size_t>(16) * groups * steps * (4 * NP * 1024));
        w_most[blockIdx.x] = __builtin_fmaxf(__builtin_fmaxf(most_of[0], most_of[1]), __builtin_fmaxf(most_of[2], most_of[3]));
    }
}

}  // namespace
}  // namespace swc
