// Conv2d for the weight types that have no integer kernel (U8, U4, F8, F8R, F4, 4-bit codebook):
// the CPU backend dequantises such weights once and runs an f32 im2col convolution
// (src/backend/cpu/mod.rs:4204-4257, src/backend/cpu/microkernels/conv.rs:509-660).  Here the
// im2col matrix [B*Ho*Wo, C/g*KH*KW] is written as f32 rows, the fused-dequant MatMul kernels
// multiply it with the packed weight rows (bias and activation in their epilogue), and the
// [pixel, channel] result is turned into NCHW.  (More than 2048 pixels, one group: the matrix is not written, the
// tiles' operand comes straight from the image, conv_prep_kernel.h.)
#include "common.h"

namespace {

// col[r, e] = x[b, g*cg + ic, oh*s + i*d - pad, ow*s + j*d - pad] (0 outside), r = b*np + oh*wo + ow,
// e = (ic*KH + i)*KW + j (src/backend/cpu/im2col.rs:32-52).  Consecutive lanes take consecutive e.  I: the type that positions are counted
// in, 32 bits wherever they fit (the divisions of 64 bits were most of the time).
template <typename I>
__global__ void __launch_bounds__(256) im2col_f32_kernel(const float *x, float *col, I total, I np, I wo, I c, I cg, int g, I h, I w, int kh, int kw,
                                                         int stride, int pad, int dil, I kk)
{
    const unsigned khw = (unsigned)(kh * kw);
    for (I idx = (I)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (I)gridDim.x * 256) {
        const I r = idx / kk;
        const unsigned e = (unsigned)(idx - r * kk);
        const I nn = r / np, p = r - nn * np;
        const I oh = p / wo, ow = p - oh * wo;
        const unsigned ic = e / khw, rem = e - ic * khw;
        const unsigned i = rem / (unsigned)kw, j = rem - i * (unsigned)kw;
        const I ih = oh * (I)stride + (I)i * (I)dil - (I)pad, iw = ow * (I)stride + (I)j * (I)dil - (I)pad;   // (unsigned: above the image wraps round to past it)
        col[idx] = ih < h && iw < w ? x[((nn * c + (I)g * cg + ic) * h + ih) * w + iw] : 0.0f;
    }
}

// y[b, ch0 + f, p] = rows_out[(b*np + p)*ocg + f]: 32x32 tiles through LDS so that both sides coalesce
__global__ void __launch_bounds__(256) rows_to_nchw_kernel(const float *src, float *y, int64_t np, int64_t oc, int64_t ch0, int64_t ocg)
{
    __shared__ float tile[32][33];
    const int64_t nn = blockIdx.z;
    const int64_t p0 = (int64_t)blockIdx.x * 32, f0 = (int64_t)blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int64_t p = p0 + ty + 8 * k, f = f0 + tx;
        tile[ty + 8 * k][tx] = (p < np && f < ocg) ? src[(nn * np + p) * ocg + f] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int64_t f = f0 + ty + 8 * k, p = p0 + tx;
        if (f < ocg && p < np) y[(nn * oc + ch0 + f) * np + p] = tile[tx][ty + 8 * k];
    }
}

}  // namespace

hipError_t launch_im2col_f32(const float *x, float *col, int64_t b, int64_t c, int groups, int g, int64_t h, int64_t w,
                             int64_t ho, int64_t wo, int kh, int kw, int stride, int pad, int dil, hipStream_t s)
{
    const int64_t cg = c / groups, kk = cg * kh * kw, np = ho * wo, rows = b * np;
    int64_t blocks = (rows * kk + 255) / 256;
    if (blocks > 65535 * 16) blocks = 65535 * 16;
    if (blocks < 1) return hipSuccess;
    const dim3 grid((unsigned)blocks);
    // (the last step of the loop may pass `total` by the grid; positions above and left of the image wrap to 2^32 - pad ..)
    const int64_t lim = 1ll << 31;
    if (rows * kk < lim && b * c * h * w < lim && pad < (1 << 30) && (ho - 1) * stride + (int64_t)(kh - 1) * dil < lim && (wo - 1) * stride + (int64_t)(kw - 1) * dil < lim)
        hipLaunchKernelGGL(im2col_f32_kernel<uint32_t>, grid, dim3(256), 0, s, x, col, (uint32_t)(rows * kk), (uint32_t)np, (uint32_t)wo, (uint32_t)c, (uint32_t)cg,
                           g, (uint32_t)h, (uint32_t)w, kh, kw, stride, pad, dil, (uint32_t)kk);
    else
        hipLaunchKernelGGL(im2col_f32_kernel<uint64_t>, grid, dim3(256), 0, s, x, col, (uint64_t)(rows * kk), (uint64_t)np, (uint64_t)wo, (uint64_t)c, (uint64_t)cg,
                           g, (uint64_t)h, (uint64_t)w, kh, kw, stride, pad, dil, (uint64_t)kk);
    return hipGetLastError();
}

hipError_t launch_rows_to_nchw(const float *src, float *y, int64_t b, int64_t np, int64_t oc, int64_t ch0, int64_t ocg, hipStream_t s)
{
    if (b < 1 || np < 1 || ocg < 1) return hipSuccess;
    if (b > 65535 || (ocg + 31) / 32 > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((np + 31) / 32), (unsigned)((ocg + 31) / 32), (unsigned)b);
    hipLaunchKernelGGL(rows_to_nchw_kernel, grid, dim3(256), 0, s, src, y, np, oc, ch0, ocg);
    return hipGetLastError();
}
