// The Winograd convolution on small grids: sixteen waves per workgroup, one per position (device code).
// See winograd2x2_conv.hip for what it replaces in the reference.
#pragma once

#include "winograd2x2_conv_kernel.h"

namespace swc {
namespace {

// A workgroup owns a WM x WN tile of the [M,K] plane and all 16 positions of it, one wave per position.  A wave
// multiplies its WM rows of TI_i by its WN columns of W_i with the operands loaded straight from global memory into
// the MFMA registers: nothing is shared between the waves before the output transform, so there is no LDS and no
// barrier in the loop, and a tile's chain of dependent steps is C long instead of 16*C.  The 16 product tiles then
// meet in LDS once and every thread takes A^T P A of its elements, terms in ascending position
// (winograd2x2_conv_cuda.cu.cc:39-46).
//
// Why: with few tiles (a batch of one, or 7x7 planes) the one-tile-per-workgroup kernels run 16*C/BK dependent
// steps on a handful of CUs, each about 0.3 us of copy latency.
//
// v_mfma_f32_16x16x4_f32 (v_mfma_f32_16x16x32_bf16 with rounded operands).  Lane (li, lg) of a wave feeds indices
// 4*lg .. 4*lg+3 of every group of 16, as in the 16x16 ring tilings (the fp32 results are theirs bit for bit): one
// 16-byte load of its row of TI and four loads of its TN neighbouring columns of W per group, KB = 4*KL indices at a
// time.  Which columns a tile holds is free: tile tn takes columns TN*li + tn, so that one load of TN floats feeds TN
// tiles.  Where TI and W allow 16-byte loads (TURN) a load takes whole rows instead, 32 indices x 8 rows of TI (16 x 16 with blocks of
// 16 indices), 16 indices x 16 columns or 8 x 32 of W, and the wave turns them round in its own LDS: a load costs the L1 an
// access for every 64 bytes that neighbouring lanes share, and one for every lane where they share none, which held a 16x16 tile
// to 2.4 us per 64 indices.
template <int TM_, int TN_, int KL_, bool BF16_, int NBUF_ = 2, bool TURN_ = false>
struct DirectCfg {
    static constexpr int TM = TM_, TN = TN_, KL = KL_;
    static constexpr int NBUF = NBUF_;             // blocks of operands in flight
    static constexpr bool BF16 = BF16_, TURN = TURN_;
    static constexpr int KB = 4 * KL;              // reduction indices per block
    static constexpr int WM = 16 * TM, WN = 16 * TN;
    static constexpr int E = WM * WN;              // elements of a product tile
    static constexpr int NT = 1024;
    static constexpr bool TURN_W = TURN && TN <= 2;          // wider tiles load 16 bytes a lane as it is
    static constexpr int STAGE = !TURN ? 0 : TURN_W && WN > WM ? KB * WN : KB * WM;   // floats a wave turns its operands round in
    static constexpr int LDS_BYTES = 16 * (E + STAGE) * 4;   // the product tiles of the sixteen positions
    static_assert(KL % 8 == 0 || (KL == 4 && !BF16), "a bf16 MFMA takes eight indices per lane");
    static_assert(LDS_BYTES <= 160 * 1024, "a CU has 160 KiB of LDS");
};

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NT) void conv_direct_kernel(const float *__restrict__ TI, const float *__restrict__ Wt,
                                                              float *__restrict__ Out, unsigned M, int C, int K, int nW,
                                                              unsigned tiles_m, unsigned tiles_n, int n_major,
                                                              ConvEpilogue ep)
{
    constexpr int TM = Cfg::TM, TN = Cfg::TN, KL = Cfg::KL, KB = Cfg::KB, E = Cfg::E, WN = Cfg::WN;
    extern __shared__ __attribute__((aligned(16))) float P[];   // [16][E] and the staging blocks

    const unsigned lid = xcd_swizzle(blockIdx.x, gridDim.x);
    // Consecutive workgroups share an XCD's L2: let them share whichever operand is the larger one.
    const unsigned tm_id = n_major ? lid % tiles_m : lid / tiles_n;
    const unsigned tn_id = n_major ? lid / tiles_m : lid % tiles_n;
    const unsigned m0 = tm_id * Cfg::WM;
    const int n0 = static_cast<int>(tn_id) * WN;
    const int pos = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;

    // Rows and columns beyond the edge repeat the last one: what they produce is not stored.
    constexpr int LPR = KB >= 32 ? 8 : 4, NA = Cfg::TURN ? LPR / 4 : 1;   // TURN: lanes to a row, loads for 16 rows
    unsigned a_off[TM][NA], b_off;   // bytes
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int h = 0; h < NA; ++h) {
            const unsigned row = m0 + tm * 16 + (Cfg::TURN ? 8 * h + lane / LPR : li);
            a_off[tm][h] = ((row < M ? row : M - 1) * static_cast<unsigned>(C) + (Cfg::TURN ? lane % LPR : lg) * 4) * 4u;
        }
    if constexpr (Cfg::TURN_W) {   // lane: index lane / (4*TN) of the load's, columns 4 * (lane % (4*TN)) .. + 3
        const int n = n0 + lane % (4 * TN) * 4;
        b_off = (static_cast<unsigned>(lane / (4 * TN)) * K + (n + 4 <= K ? n : K - 4)) * 4u;   // K % 4 == 0
    } else {
        const int n = n0 + TN * li;
        b_off = (static_cast<unsigned>(lg * 4) * K + (n + TN <= K ? n : K - TN)) * 4u;   // K % TN == 0
    }
    // Descriptors of the position's planes: what a load adds to a lane's offset is the same for the whole wave and
    // sits in a scalar register, and what a lane must not read is an offset beyond the end: it reads as zero.
    const __amdgpu_buffer_rsrc_t a_desc = make_rsrc(TI + static_cast<size_t>(pos) * M * C, M * static_cast<unsigned>(C) * 4u);
    const __amdgpu_buffer_rsrc_t b_desc = make_rsrc(Wt + static_cast<size_t>(pos) * C * K, static_cast<unsigned>(C) * K * 4u);

    typedef float BVec __attribute__((ext_vector_type(TN)));
    constexpr int KR = 16 / TN, NR = KB / KR;   // TURN: indices to a load, loads to a block
    struct Frag {
        float4 a[TM][KL / 4];
        typename std::conditional<Cfg::TURN_W, floatx4[NR], BVec[KL]>::type b;
    };
    auto load = [&](Frag &f, int k0) __attribute__((always_inline)) {
        const bool whole = k0 + KB <= C;     // uniform; else the last block: indices beyond C are zero on both sides
        const int left = C - k0 - lg * 4;    // a group of 16 that starts at j holds indices of this lane while j < left (C % 4 == 0)
#pragma unroll
        for (int tm = 0; tm < TM; ++tm)
#pragma unroll
            for (int j = 0; j < KL / 4; ++j) {
                // TURN: load j holds rows 8*(j % NA) .. of indices 4*LPR*(j / NA) ..
                const int at = Cfg::TURN ? j / NA * 4 * LPR : 16 * j;
                const bool in = whole || (Cfg::TURN ? at + lane % LPR * 4 < C - k0 : at < left);
                f.a[tm][j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                            a_desc, static_cast<int>(in ? a_off[tm][j % NA] : kOutOfRange), (k0 + at) * 4, 0));
            }
        if constexpr (Cfg::TURN_W) {
#pragma unroll
            for (int i = 0; i < NR; ++i)
                f.b[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                                         b_desc, static_cast<int>(whole || KR * i + lane / (4 * TN) < C - k0 ? b_off : kOutOfRange),
                                                         (k0 + KR * i) * K * 4, 0));
        } else
#pragma unroll
        for (int t = 0; t < KL; ++t) {
            const int j = t / 4, voff = static_cast<int>(whole || 16 * j < left ? b_off : kOutOfRange), soff = (k0 + 16 * j + t % 4) * K * 4;
            if constexpr (TN == 4)
                f.b[t] = __builtin_bit_cast(BVec, __builtin_amdgcn_raw_buffer_load_b128(b_desc, voff, soff, 0));
            else if constexpr (TN == 2)
                f.b[t] = __builtin_bit_cast(BVec, __builtin_amdgcn_raw_buffer_load_b64(b_desc, voff, soff, 0));
            else
                f.b[t] = __builtin_bit_cast(BVec, __builtin_amdgcn_raw_buffer_load_b32(b_desc, voff, soff, 0));
        }
    };
    floatx4 acc[TM][TN];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[tm][tn][r] = 0.f;

    auto at4 = [](const float4 &v, int q) __attribute__((always_inline)) { return q == 0 ? v.x : q == 1 ? v.y : q == 2 ? v.z : v.w; };
    // Index 16*j + 4*g + t of a block lies in row 16*j + 4*t + g of the staging block: what the four lane groups read at a time is
    // then side by side.
    float *const stage = P + 16 * E + pos * Cfg::STAGE;
    auto multiply = [&](const Frag &raw) __attribute__((always_inline)) {
        struct {
            float4 a[TM][KL / 4];
            BVec b[KL];
        } f;
        if constexpr (Cfg::TURN) {   // 16-byte chunk c of row r of 16 rows x 4*LPR indices in slot c ^ (r % 8), c ^ (r / 2 % 4) with four
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int j = 0; j < KL / 4; ++j) {
                    const int r = 8 * (j % NA) + lane / LPR, c = lane % LPR;
                    *reinterpret_cast<float4 *>(stage + (tm * KB + j / NA * 4 * LPR) * 16 + r * 4 * LPR + (c ^ (LPR == 8 ? r % 8 : r / 2 % 4)) * 4) =
                        raw.a[tm][j];
                }
            asm volatile("" ::: "memory");   // other lanes' values are read back; a wave's LDS operations are executed in order
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int j = 0; j < KL / 4; ++j) {
                    const int c = j % NA * 4 + lg;
                    f.a[tm][j] = *reinterpret_cast<const float4 *>(stage + (tm * KB + j / NA * 4 * LPR) * 16 + li * 4 * LPR +
                                                                   (c ^ (LPR == 8 ? li % 8 : li / 2 % 4)) * 4);
                }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int j = 0; j < KL / 4; ++j) f.a[tm][j] = raw.a[tm][j];
        }
        if constexpr (Cfg::TURN_W) {
#pragma unroll
            for (int i = 0; i < NR; ++i) {
                const int k = KR * i + lane / (4 * TN), row = k / 16 * 16 + k % 4 * 4 + k / 4 % 4;
                *reinterpret_cast<floatx4 *>(stage + row * WN + lane % (4 * TN) * 4) = raw.b[i];
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int t = 0; t < KL; ++t)
                f.b[t] = *reinterpret_cast<const BVec *>(stage + (t / 4 * 16 + t % 4 * 4 + lg) * WN + TN * li);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        } else {
#pragma unroll
            for (int t = 0; t < KL; ++t) f.b[t] = raw.b[t];
        }
        if constexpr (Cfg::BF16) {
#pragma unroll
            for (int g = 0; g < KL / 8; ++g) {
                typedef float floatx8 __attribute__((ext_vector_type(8)));
                bf16x8 av[TM], bv[TN];
#pragma unroll
                for (int tm = 0; tm < TM; ++tm) {
                    const float4 u = f.a[tm][2 * g], v = f.a[tm][2 * g + 1];
                    av[tm] = __builtin_convertvector(floatx8{u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w}, bf16x8);
                }
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
                    bv[tn] = __builtin_convertvector(floatx8{f.b[8 * g][tn], f.b[8 * g + 1][tn], f.b[8 * g + 2][tn], f.b[8 * g + 3][tn],
                                                             f.b[8 * g + 4][tn], f.b[8 * g + 5][tn], f.b[8 * g + 6][tn], f.b[8 * g + 7][tn]},
                                                     bf16x8);
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn)
                        acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[tm], bv[tn], acc[tm][tn], 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int t = 0; t < KL; ++t)
#pragma unroll
                for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                    for (int tn = 0; tn < TN; ++tn)
                        acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(at4(f.a[tm][t / 4], t % 4), f.b[t][tn], acc[tm][tn], 0, 0, 0);
        }
    };

    if constexpr (Cfg::NBUF > 1) {
        constexpr int N = Cfg::NBUF;
        Frag f[N];
#pragma unroll
        for (int i = 0; i + 1 < N; ++i)
            if (i * KB < C) load(f[i], i * KB);
        for (int k0 = 0; k0 < C;)
#pragma unroll
            for (int i = 0; i < N; ++i) {
                if (k0 + (N - 1) * KB < C) load(f[(i + N - 1) % N], k0 + (N - 1) * KB);
                multiply(f[i]);
                k0 += KB;
                if (k0 >= C) break;
            }
    } else {
        for (int k0 = 0; k0 < C; k0 += KB) {
            Frag f;
            load(f, k0);
            multiply(f);
        }
    }

    // Accumulator register r of lane (lg, li): row 4*lg + r of the tile, its column li, i.e. TN*li + tn of the wave's.
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) P[pos * E + (tm * 16 + 4 * lg + r) * WN + TN * li + tn] = acc[tm][tn][r];
    __syncthreads();

    const size_t row_stride = 2 * static_cast<size_t>(nW) * K;
    const bool affine = ep.scale != nullptr, residual = ep.residual != nullptr;
    // Output j = 2*dy + dx of element e: nine of the sixteen products, ascending position.
    auto combine = [&](int e, auto j_tag) __attribute__((always_inline)) {
        constexpr int j = decltype(j_tag)::value;
        float y = 0.f;
        bool first = true;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int bit = 4 * i + j;
            if ((kPlus >> bit) & 1ull) {
                y = first ? P[i * E + e] : y + P[i * E + e];
                first = false;
            } else if ((kMinus >> bit) & 1ull) {
                y -= P[i * E + e];   // the first term of every output is a plus
            }
        }
        const unsigned gm = m0 + e / WN;
        const int col = n0 + e % WN;
        if (gm >= M || col >= K) return;
        const unsigned bt = gm / static_cast<unsigned>(nW);   // b*nH + th
        const unsigned tw = gm - bt * static_cast<unsigned>(nW);
        const size_t at = static_cast<size_t>(bt) * 2 * row_stride + 2 * static_cast<size_t>(tw) * K + col + (j / 2) * row_stride +
                          (j % 2) * static_cast<size_t>(K);
        if (affine) y = __builtin_fmaf(y, ep.scale[col], ep.shift[col]);
        if (residual) {
            float q = ep.residual[at];
            if (ep.residual_relu) q = q > 0.f ? q : 0.f;
            y += q;
        }
        store_streaming(Out + at, y);
    };
    {
        // an element per thread and pass, and which of its outputs the same for a whole wave
        constexpr int PER_J = E / 64 >= 16 ? 16 : E / 64;      // waves side by side in one output
        constexpr int JS = 16 / PER_J;                         // outputs taken at a time
        const int w = pos, jg = w / PER_J;
#pragma unroll
        for (int e0 = 0; e0 < E; e0 += PER_J * 64) {
            const int e = e0 + (w % PER_J) * 64 + lane;
            static_for<4>([&](auto j_tag) {
                if (JS == 1 || jg == decltype(j_tag)::value % JS) combine(e, j_tag);
            });
        }
    }
}

}  // namespace
}  // namespace swc
