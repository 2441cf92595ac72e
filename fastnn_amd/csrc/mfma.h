// Matrix-core kernel entry points.
#pragma once
#include <atomic>

#include "common.h"
#include "i8act.h"

// context services implemented beside the C ABI
int fnn_ctx_ensure_tmp(fnn_hip_ctx *ctx, int which, size_t bytes, void **ptr);
// whether fnn_ctx_ensure_tmp would give this call the bytes (a kernel that has others behind it leaves the call to them)
bool fnn_ctx_tmp_fits(fnn_hip_ctx *ctx, int which, size_t bytes);
int fnn_ctx_fail(fnn_hip_ctx *ctx, int code, const char *msg);
bool fnn_ctx_capturing(fnn_hip_ctx *ctx);
// true while device memory must not be allocated: graph capture, or a call through fnn_hip_qmatmul_static
bool fnn_ctx_no_alloc(fnn_hip_ctx *ctx);
bool fnn_ctx_static_mode(fnn_hip_ctx *ctx);
// memory for a copy of packed words in another order: null where this call may not allocate or the device has no room (the
// kernels read the registered words then)
void *fnn_ctx_copy_memory(fnn_hip_ctx *ctx, size_t bytes);
// value of a per-context option (FNN_OPT_*, set through fnn_hip_set_option)
int64_t fnn_ctx_option(const fnn_hip_ctx *ctx, int option);

// Raises a kernel's dynamic LDS limit once per device.  `done` is a bit mask of devices (one static per kernel
// instantiation); safe from several threads, and a second device gets its own call.
inline hipError_t fnn_raise_lds_limit(std::atomic<uint64_t> &done, const void *kernel, int bytes)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
    return e;
}

// M >= 5: activations prepared once as f16 operands, 4-wave output tiles with the
// activations staged through LDS and optional split of K (deterministic reduction).
// up to 32 rows (codebook type 64), where the fragment kernels below do not take the call: one launch, weights streamed into the MFMA operand
// registers, activations converted in the kernel, K split over workgroups and reduced by the last one to arrive (qgemm_stream.hip)
int fnn_stream_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p, int flags, bool *handled);
// whether it takes the call, and the microseconds that it is expected to take
bool fnn_stream_takes(fnn_hip_ctx *ctx, const fnn_hip_weight *w, const QMatmulArgs &p, int flags, float *us);
// arrival counters of that kernel's column tiles: FNN_STREAM_COUNTERS words of device memory, zero between launches
constexpr int FNN_STREAM_COUNTERS = 4096;
uint32_t *fnn_ctx_stream_counters(fnn_hip_ctx *ctx);
// int8 matrix-core GEMM over exact activation digit planes (qgemm_digits.hip: LDS tiles, or the register tiles of qgemm_wave_impl.h):
// M >= 17, I8 / I4 / U4 weights, where the kernels above and below do not take the call
int fnn_digits_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p, int flags, bool *handled);
// digit planes that path would multiply the call with by rule and options (3, 4); 0: the call is another kernel's
int fnn_digits_planes(fnn_hip_ctx *ctx, int dt, int64_t m, int64_t n, int64_t k, int flags);
float fnn_digits3_us(int dt, int64_t m, int64_t n, int64_t k);   // microseconds expected of three planes
// a middle number of activation rows (and any number with ragged weight rows), per-channel types: both operands in the order the
// matrix cores take them; asked first, takes what it is expected to finish before the kernels it would replace (qgemm_frag.hip)
int fnn_frag_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p, int flags, bool *handled);
// 5 to 16 rows, codebook weights with blocks of 32 (qgemm_codebook.hip)
int fnn_codebook_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p, int flags, bool *handled);
int fnn_frag_i8act(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const I8ActArgs &p, bool *handled);
// fragment-major copy of a weight's packed words, built on first use; null when it does not exist and this call may not build it
int fnn_fragment_words(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, int64_t kblocks, const uint32_t **words);
// that copy (kp 0) or the registered rows
int fnn_frag_words(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, int64_t kblocks, const uint32_t **words, int *kp);
// sum of the integer lanes per weight row (I8, I4), built on first use
int fnn_row_qsum(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const int32_t **qsum);
// microseconds expected of the f16 tiles (per-channel types)
float fnn_tiled_us(fnn_hip_ctx *ctx, int dt, int64_t m, int64_t n, int64_t k, int flags);
hipError_t launch_rows_to_nchw(const float *src, float *y, int64_t b, int64_t np, int64_t oc, int64_t ch0, int64_t ocg, hipStream_t s);
// (conv: the activations are a convolution's windows of its NCHW input, p.m output pixels of p.k values; p.a is not read)
struct ConvSource {
    const float *x;
    int c, h, w, kh, kw, stride, pad, dil, wo, np;   // np: output pixels of an image
    unsigned bytes;                                  // of x
    float *y;                                        // the result, [image][channel][np] (p.out is not used)
};
int fnn_tiled_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p,
                      int flags, bool *handled, const ConvSource *conv = nullptr);
// FNN_FLAG_ACT_QUANT with F8 weights: activations rounded to E4M3 (one power-of-two scale per row), fp8 matrix cores
int fnn_fp8_actquant_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p, bool *handled);

int64_t fnn_conv_operand_workgroups(const QConvArgs &p);
// the convolution from an int8 patch in LDS (qconv_patch.hip), asked first: rectangles of 32 * wpx pixels, nw waves over pixels (wpx), blocks of 32
// channels (wch) and K (wks), `per` rectangles a workgroup, gy workgroups over the channels
struct FnnPatchShape {
    int nw, wpx, wch, wks, gy, per, segs, cs, nss, sets, twl, th, pw, pp, tiles_x, tiles;
    size_t lds;
    int64_t workgroups(int64_t images) const { return images * ((tiles + per - 1) / per) * gy; }
};
bool fnn_patch_conv_takes(fnn_hip_ctx *ctx, hipStream_t stream, const fnn_hip_weight *w, const QConvArgs &p, FnnPatchShape *s);
int fnn_patch_conv(fnn_hip_ctx *ctx, hipStream_t stream, const fnn_hip_weight *w, const QConvArgs &p, const FnnPatchShape &s);

// single-f16 activation mode: mean lane value per weight row (null for types whose lanes have zero mean)
int fnn_row_means(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const float **umean);

// M <= 8: bandwidth-bound GEMV on the matrix cores (weights requested before anything else).
int fnn_mfma_qgemv(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p,
                   int flags, bool *handled);

// M <= 8 (16 by option), integer weights (I8, U8, I4, U4): int8 matrix cores, activations as four exact base-256 digit rows per slice of K (no
// decode arithmetic, activations converted once per workgroup).
int fnn_i8dot_qgemv(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p, bool *handled);
// that copy for the kernels that take rows of whole 64-byte blocks only, null where it does not apply
int fnn_fragment_blocks(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &q, const uint32_t **words_fr, int64_t *kb64);

// 9 <= M <= 16: the same organisation with the 16 activation rows as the MFMA operand rows, loaded straight
// into registers (no preparation or reduction launch).
int fnn_mfma_rows16(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &p,
                    int flags, bool *handled);
// the microseconds that it is expected to take
float fnn_rows16_us(int dtype, int64_t m, int64_t n, int64_t k);

// I8 activations x I8/I4 weights and the quantised Conv2d on int8 MFMA tiles with i32 accumulators.
float fnn_i8_tiled_us(int dt, int64_t m, int64_t n, int64_t k);   // microseconds expected of the LDS tiles
int fnn_i8_tiled_matmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const I8ActArgs &p, bool *handled);
// p.actq must already hold the (image, group) activation scales.
int fnn_i8_tiled_conv(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QConvArgs &p, bool *handled);

// Weight rows as 16-byte addressable pieces: the registered words, or (when kp % 4 != 0) a copy with the
// rows re-strided to a multiple of four words, zero-filled, made on first use and kept with the weight.
int fnn_aligned_rows(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const uint32_t **words, int64_t *kp);
