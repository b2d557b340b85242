// What the convolution's forms with a wave per position share behind their products: sixteen planes of products, eight at a
// time in LDS, into the outputs (device code).
#pragma once

#include "winograd2x2_conv_kernel.h"

namespace swc {
namespace {

// A thread finishes four consecutive columns of QN rows of a Cfg::WM x 64 tile; sums of positions 0-7 first, then 8-15: terms
// in ascending position (winograd2x2_conv_cuda.cu.cc:39-46).
template <typename Cfg>
struct OutputPlanes {
    static constexpr int E = Cfg::E, NT = Cfg::NT, QN = (E / 4 + NT - 1) / NT;
    floatx4 y[QN][4];

    // P: planes 8*half .. 8*half+7, [8][E].
    template <int half>
    __device__ __forceinline__ void combine(const float *P)
    {
#pragma unroll
        for (int q = 0; q < QN; ++q) {
            const int e4 = q * NT + static_cast<int>(threadIdx.x);
            if (E / 4 % NT != 0 && e4 >= E / 4) break;
            static_for<8>([&](auto i_tag) __attribute__((always_inline)) {
                constexpr int i = 8 * half + decltype(i_tag)::value;
                const floatx4 p = *reinterpret_cast<const floatx4 *>(&P[(i % 8) * E + 4 * e4]);
                static_for<4>([&](auto j_tag) __attribute__((always_inline)) {
                    constexpr int j = decltype(j_tag)::value, bit = 4 * i + j;
                    constexpr unsigned long long below = (kPlus | kMinus) & (0x1111111111111111ull << j) & ((1ull << (4 * i)) - 1);
                    if constexpr ((kPlus >> bit) & 1ull)
                        y[q][j] = below == 0 ? p : y[q][j] + p;
                    else if constexpr ((kMinus >> bit) & 1ull)
                        y[q][j] = y[q][j] - p;   // the first term of every output is a plus
                });
            });
        }
    }

    // Offsets into the output stay below 2^31 bytes (checked by the launcher).
    __device__ __forceinline__ void store(float *__restrict__ Out, unsigned M, int K, int nW, unsigned m0, unsigned rows_valid, int n0,
                                          const ConvEpilogue &ep)
    {
        const size_t row_stride = 2 * static_cast<size_t>(nW) * K;
        const bool affine = ep.scale != nullptr, residual = ep.residual != nullptr;
        const __amdgpu_buffer_rsrc_t o_desc = make_rsrc(Out, M * 16u * static_cast<unsigned>(K));
#pragma unroll
        for (int q = 0; q < QN; ++q) {
            const int e4 = q * NT + static_cast<int>(threadIdx.x);
            const unsigned row = static_cast<unsigned>(e4) / 16u;
            const int col = n0 + e4 % 16 * 4;
            if (row >= rows_valid || col >= K) continue;
            const unsigned gm = m0 + row;
            const unsigned bt = gm / static_cast<unsigned>(nW);   // b*nH + th
            const unsigned tw = gm - bt * static_cast<unsigned>(nW);
            const size_t at = static_cast<size_t>(bt) * 2 * row_stride + 2 * static_cast<size_t>(tw) * K + col;
            size_t out_at[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) out_at[j] = at + (j / 2) * row_stride + (j % 2) * static_cast<size_t>(K);
            if (affine)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float sc = ep.scale[col + i], sh = ep.shift[col + i];
#pragma unroll
                    for (int j = 0; j < 4; ++j) y[q][j][i] = __builtin_fmaf(y[q][j][i], sc, sh);
                }
            if (residual) {
                const bool whole = !ep.residual_relu;
                floatx4 res[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) res[j] = *reinterpret_cast<const floatx4 *>(ep.residual + out_at[j]);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[q][j][i] += (whole | (res[j][i] > 0.f)) ? res[j][i] : 0.f;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                // sc1: written through as it is issued (see store_streaming)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(intx4, y[q][j]), o_desc, static_cast<int>(out_at[j] * 4), 0, 16);
            }
        }
    }
};

}  // namespace
}  // namespace swc
