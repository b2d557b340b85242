// The two passes of the model that are neither a Winograd layer nor a convolution: the 3x3 stride-2 max-pool behind a stage and the
// ReLU with the mean over all pixels in front of the classifier (ResNet-18-var/imagenet-resnet-transWino-prune.py, MaxPooling and
// GlobalAvgPooling of the graph).  Both read their input once and are bound by memory.  At 128 images, library -> here: the pool behind
// stage 2 (56x56x64, 128 MB) 49 -> 23 us, behind stage 3 (28x28x128, 64 MB) 43 -> 12, ReLU and mean over 14x14x512 (51 MB) in two passes
// 17 + 15 -> 10.5.
#include "swc_common.h"

namespace swc {
namespace {

// torch's rule: the largest, and a NaN where the window has one
__device__ __forceinline__ float larger(float m, float v) { return v > m || v != v ? v : m; }
// relu with NaN kept
__device__ __forceinline__ float relu(float v) { return v < 0.0f ? 0.0f : v; }

// A lane has four channels of one pooled pixel: nine 16-byte loads, whole lines per wave, and what neighbouring windows share comes
// from the caches (consecutive blocks stay on one XCD, whose L2 then has the rows).  Padding is in front of odd sides only.
__global__ __launch_bounds__(256) void max_pool_kernel(const float4 *__restrict__ X, float4 *__restrict__ Y, int H, int W, unsigned CV, unsigned oH,
                                                       unsigned oW, unsigned items)
{
    const unsigned id = xcd_swizzle(blockIdx.x, gridDim.x) * 256u + threadIdx.x;
    if (id >= items) return;
    unsigned p = id / CV;
    const unsigned cv = id % CV, ox = p % oW;
    p /= oW;
    const unsigned oy = p % oH, b = p / oH;
    const int y0 = static_cast<int>(2 * oy) - (H & 1), x0 = static_cast<int>(2 * ox) - (W & 1);
    const float4 *img = X + static_cast<size_t>(b) * H * W * CV + cv;
    // A window's padding stands for its pixel next to it, which changes no maximum and leaves nine loads without a branch.
    float4 v[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) {
        const int y = min(max(y0 + i / 3, 0), H - 1), x = min(max(x0 + i % 3, 0), W - 1);
        v[i] = img[(static_cast<size_t>(y) * W + x) * CV];
    }
    float4 m = v[0];
#pragma unroll
    for (int i = 1; i < 9; ++i) m = make_float4(larger(m.x, v[i].x), larger(m.y, v[i].y), larger(m.z, v[i].z), larger(m.w, v[i].w));
    Y[id] = m;
}

// A workgroup has 64 channels of one image, sixteen lanes of four channels by sixteen groups of pixels, whose sums meet in LDS.
__global__ __launch_bounds__(256) void relu_mean_kernel(const float4 *__restrict__ X, float4 *__restrict__ Y, unsigned pixels, unsigned CV, unsigned groups)
{
    __shared__ float4 sums[16][16];
    const unsigned b = blockIdx.x / groups, lane = threadIdx.x & 15u, part = threadIdx.x >> 4, cv = blockIdx.x % groups * 16u + lane;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (cv < CV) {
        const float4 *img = X + static_cast<size_t>(b) * pixels * CV + cv;
#pragma unroll 4
        for (unsigned p = part; p < pixels; p += 16) {
            const float4 v = img[static_cast<size_t>(p) * CV];
            s = make_float4(s.x + relu(v.x), s.y + relu(v.y), s.z + relu(v.z), s.w + relu(v.w));
        }
    }
    sums[part][lane] = s;
    for (unsigned half = 8; half > 0; half /= 2) {
        __syncthreads();
        if (part < half) {
            const float4 a = sums[part][lane], o = sums[part + half][lane];
            sums[part][lane] = make_float4(a.x + o.x, a.y + o.y, a.z + o.z, a.w + o.w);
        }
    }
    if (part == 0 && cv < CV) {
        const float n = static_cast<float>(pixels);
        const float4 a = sums[0][lane];
        Y[static_cast<size_t>(b) * CV + cv] = make_float4(a.x / n, a.y / n, a.z / n, a.w / n);
    }
}

// 16-byte loads of four channels, 32-bit numbers of items and pixels.
int check_operands(const float *Input, const float *Output, int C, int B, int H, int W)
{
    if (Input == nullptr || Output == nullptr) return SWC_ERR_NULL_POINTER;
    if (C <= 0 || B <= 0 || H <= 0 || W <= 0) return SWC_ERR_BAD_DIMS;
    if (C % 4 != 0 || !aligned16(Input) || !aligned16(Output) || H >= (1 << 30) || W >= (1 << 30)) return SWC_ERR_UNSUPPORTED;
    return SWC_OK;
}

}  // namespace
}  // namespace swc

extern "C" int swc_max_pool_same(const float *Input, float *Output, int C, int B, int H, int W, swc_stream_t stream)
{
    using namespace swc;
    const int st = check_operands(Input, Output, C, B, H, W);
    if (st != SWC_OK) return st;
    const size_t oH = (static_cast<size_t>(H) + 1) / 2, oW = (static_cast<size_t>(W) + 1) / 2, CV = static_cast<size_t>(C) / 4;
    if (oH * oW >= (1ull << 31) || oH * oW * CV >= (1ull << 31) || oH * oW * CV * B >= (1ull << 31)) return SWC_ERR_UNSUPPORTED;
    const unsigned items = static_cast<unsigned>(oH * oW * CV * B);
    max_pool_kernel<<<dim3((items + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        reinterpret_cast<const float4 *>(Input), reinterpret_cast<float4 *>(Output), H, W, static_cast<unsigned>(CV), static_cast<unsigned>(oH),
        static_cast<unsigned>(oW), items);
    return check_launch();
}

extern "C" int swc_relu_mean(const float *Input, float *Output, int C, int B, int H, int W, swc_stream_t stream)
{
    using namespace swc;
    const int st = check_operands(Input, Output, C, B, H, W);
    if (st != SWC_OK) return st;
    const size_t pixels = static_cast<size_t>(H) * W, groups = (static_cast<size_t>(C) + 63) / 64;
    // A partial sum is a chain of pixels / 16 additions, and B * C/64 workgroups is all there are.  Against the library's two passes, us and
    // error against float64 (2-norm): 1x14x14x512 14.1 / 4.1 and 5.5e-8 / 4.9e-8, 128x32x32x512 179 / 41 and 5.5e-8 / 3.9e-8, 1x32x32x64 17 / 5.8 and
    // 3.9e-8 / 3.7e-8; but 1x64x64x64 13.7 / 17.3 and 3.2e-8 / 5.5e-8, 1x256x256x64 23 / 423 and 4.7e-8 / 1.8e-7.
    if (pixels > 1024 || groups * B >= (1ull << 31)) return SWC_ERR_UNSUPPORTED;
    relu_mean_kernel<<<dim3(static_cast<unsigned>(groups * B)), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
        reinterpret_cast<const float4 *>(Input), reinterpret_cast<float4 *>(Output), static_cast<unsigned>(pixels), static_cast<unsigned>(C / 4),
        static_cast<unsigned>(groups));
    return check_launch();
}
