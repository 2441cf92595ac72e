// Host side of the fragment-major MatMul on I8 activations (kernels: qgemm_frag_int_impl.h).
//
// Launches: frag_codes_kernel (payload rows -> operand fragments; short products read the payload themselves),
// qgemm_frag_int_kernel, and with K split over workgroups frag_codes_reduce_kernel.
#include "mfma.h"
#include "qgemm_frag_int.h"
#include "range_io.h"

namespace {

// One wave per block of 16 rows and step of 64 k-values: lane r + 16 q moves the 16 codes of row r that it will hold as an
// operand; the store is one contiguous KB.  Rows start on any byte: the aligned words around a piece are shifted together.
template <bool IL>
__global__ void __launch_bounds__(256) frag_codes_kernel(const uint8_t *payload, int64_t m_rows, int64_t k, int nsteps, uint4 *af)
{
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const int step = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (step >= nsteps) return;
    const int64_t m = (int64_t)blockIdx.y * 16 + (lane & 15);
    const int64_t k0 = IL ? (int64_t)(step >> 1) * 128 + 32 * q + 16 * (step & 1) : (int64_t)step * 64 + 16 * q;
    uint32_t v[4] = {0, 0, 0, 0};
    if (m < m_rows && k0 < k) {
        const uint8_t *x = payload + 8 + m * k + k0;
        if (k0 + 16 <= k) {
            const uint32_t *w = reinterpret_cast<const uint32_t *>(reinterpret_cast<uintptr_t>(x) & ~(uintptr_t)3);
            const int off = (int)(reinterpret_cast<uintptr_t>(x) & 3);
            uint32_t t[5];
#pragma unroll
            for (int i = 0; i < 4; i++) t[i] = w[i];
            t[4] = off ? w[4] : 0u;   // (holds the last `off` codes of the piece)
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = __builtin_amdgcn_alignbyte(t[i + 1], t[i], off);
        } else {
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (k0 + i < k) v[i >> 2] |= (uint32_t)x[i] << (8 * (i & 3));
        }
    }
    if constexpr (IL) {   // the nibble decoders deliver k = 0,2,4,6,1,3,5,7 of each 8
        const uint32_t x0 = v[0], x1 = v[1], x2 = v[2], x3 = v[3];
        v[0] = __builtin_amdgcn_perm(x1, x0, 0x06040200u);
        v[1] = __builtin_amdgcn_perm(x1, x0, 0x07050301u);
        v[2] = __builtin_amdgcn_perm(x3, x2, 0x06040200u);
        v[3] = __builtin_amdgcn_perm(x3, x2, 0x07050301u);
    }
    af[((int64_t)blockIdx.y * nsteps + step) * 64 + lane] = make_uint4(v[0], v[1], v[2], v[3]);
}

// exact sums of the splits, then the I8-activation formula; one column per thread
__global__ void __launch_bounds__(256) frag_codes_reduce_kernel(FragIntArgs p)
{
    const int64_t total = p.m * p.n, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t m = i / p.n, n = i - m * p.n;
    const float sa = reinterpret_cast<const float *>(p.payload)[0], za = reinterpret_cast<const float *>(p.payload)[1];
    int acc = 0, qsum = 0;
    for (int z = 0; z < p.ks.splits; z++) {
        acc += p.part[(int64_t)z * total + i];
        qsum += p.qsum[(int64_t)z * p.m_pad + m];
    }
    const float input_sum = (float)qsum * sa + (float)p.k * za;
    const float dot = za != 0.0f ? (float)acc * sa + za * (float)p.wsum[n] : (float)acc * sa;
    float v = dot * p.scales[n] + p.zeros[n] * input_sum;
    if (p.bias) v = v + p.bias[n];
    p.out[i] = fnn_activation(v, p.act);
    if (p.acc_out) p.acc_out[i] = za != 0.0f ? 0 : acc;
}

// Which form: an estimate in microseconds (quantisation included), least squares over 3 500 drawn shapes in all their forms (7 % mean error; the terms as
// in qgemm_frag.hip).  Reading the payload in the kernel touches 16 separate 64-byte pieces per wave load (3.5 times the L1
// time of a contiguous KB) and saves the launch that lays the codes out.
struct IntShape { int mb, nb; };
constexpr IntShape kIntShapes[] = {{1, 1}, {1, 2}, {2, 2}, {2, 4}, {4, 4}};

struct IntLoad { float rounds, bytes, mfma, area, mn, mk, nk; };
IntLoad codes_load(IntShape t, bool direct, int splits, int64_t m, int64_t n, int64_t k, int groups, bool four)
{
    const float area = (float)(t.mb * t.nb);
    const float x = (float)((m + 16 * t.mb - 1) / (16 * t.mb)) * (float)((n + 16 * t.nb - 1) / (16 * t.nb)) * (float)splits / 256.f, cx = (float)(int)(x + 0.99999f);
    float r = area > 8.f ? cx : (x <= 4.f ? 0.5f * (cx + x) : x + 0.25f);
    if (r < 1.f) r = 1.f;
    const float seg = (float)(((groups + splits - 1) / splits + FRAG_NW - 1) / FRAG_NW), wb = four ? 64.f : 128.f;
    return {r, seg * 8.f * ((float)t.mb * 2048.f * (direct ? 3.5f : 1.f) + (float)t.nb * 16.f * wb) / 1e5f, seg * area * 64.f / 2400.f, area,
            (float)m * (float)n * 4.f / 1e6f, (float)m * (float)k * 9.f / 1e6f, (float)n * (float)groups * wb / 1e6f};
}
float codes_order(const IntLoad &l, bool direct, int splits)
{
    const float two = splits > 1 ? 1.f : 0.f;
    return direct ? 10.22f + l.rounds * (0.25f * l.bytes + 2.596f * l.mfma) + two * 2.91f + 0.277f * l.mn + 0.267f * l.mk + 0.0116f * l.nk
                  : 12.76f + l.rounds * (0.387f * l.bytes + 1.563f * l.mfma) + two * 3.12f + 0.438f * l.mn + 0.308f * l.mk + 0.013f * l.nk;
}
// Microseconds of the form that it picks (operand kernel + MatMul), to be compared with the LDS tiles': least squares over 590 drawn calls
// whose products are below 8e9 MACs, 7 % mean error.
float codes_us(const IntLoad &l, bool direct, int splits)
{
    const float two = splits > 1 ? 1.f : 0.f;
    return direct ? 2.59f + l.rounds * (0.388f * l.bytes + 3.112f * l.mfma + 0.0384f + 0.0094f * l.area) + two * 2.91f + 0.501f * l.mn + 0.134f * l.mk + 0.1066f * l.nk
                  : 5.11f + l.rounds * (0.567f * l.bytes + 1.415f * l.mfma + 0.0537f * l.area) + two * 3.12f + 0.401f * l.mn + 0.172f * l.mk + 0.1011f * l.nk;
}

}  // namespace

int fnn_frag_i8act(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const I8ActArgs &q, bool *handled)
{
    *handled = false;
    const int64_t opt = fnn_ctx_option(ctx, FNN_OPT_FRAGMENT);
    if (opt < 0 || fnn_ctx_option(ctx, FNN_OPT_TILE_SHAPE) != -1 || fnn_ctx_option(ctx, FNN_OPT_TILE_SPLIT) != 0 || fnn_ctx_static_mode(ctx)) return FNN_OK;
    if (w->dtype != FNN_DT_I8 && w->dtype != FNN_DT_I4) return FNN_OK;
    // exact i32 sums: |code| <= 128, |lane| <= 128 (16 q for nibbles); 32-bit payload offsets in the kernel that reads it
    if (q.words != w->words || q.n != w->rows || q.k != w->inner || q.m < 1 || q.m > (1 << 16) || q.n > (1 << 22) || q.k < 1 || q.k > (1 << 16)) return FNN_OK;
    if (reinterpret_cast<uintptr_t>(q.payload) & 3) return FNN_OK;
    const bool four = w->dtype == FNN_DT_I4;
    FragIntArgs p = {};
    p.kblocks = (int)((w->kp + 15) / 16);
    p.ks.kblocks = four ? p.kblocks : (p.kblocks + 1) / 2;   // groups of 128 k-values
    int mb = 0, nb = 0, splits = 1;
    bool direct = false;
    const bool direct_ok = q.k % 4 == 0 && q.m * q.k < (int64_t)1 << 31;
    if (opt > 0) {
        mb = (int)(opt & 15); nb = (int)((opt >> 4) & 15);
        splits = (int)((opt >> 8) & 15) > 0 ? (int)((opt >> 8) & 15) : 1;
        direct = ((opt >> 15) & 1) && direct_ok;
    } else {
        // (products beyond that run at the matrix cores' rate on the LDS tiles: 2048 x 4096 x 4096 78 us there, 112 here)
        if ((double)q.m * (double)q.n * (double)q.k > 8e9) return FNN_OK;
        float best = 1e30f, us = 0.f;
        for (IntShape t : kIntShapes) {
            if (t.mb > 1 && (t.mb / 2) * 16 >= q.m) continue;
            const int64_t wgs = ((q.m + 16 * t.mb - 1) / (16 * t.mb)) * ((q.n + 16 * t.nb - 1) / (16 * t.nb));
            for (int sp : {1, 2, 4}) {
                if (sp > 1 && (wgs * sp > 600 || sp * 8 > p.ks.kblocks)) break;
                for (int d = 0; d < 2; d++) {
                    if (d && (!direct_ok || q.m > 256)) continue;
                    const IntLoad l = codes_load(t, d != 0, sp, q.m, q.n, q.k, p.ks.kblocks, four);
                    const float o = codes_order(l, d != 0, sp);
                    if (o < best) { best = o; us = codes_us(l, d != 0, sp); mb = t.mb; nb = t.nb; splits = sp; direct = d != 0; }
                }
            }
        }
        if (us > 0.97f * fnn_i8_tiled_us(w->dtype, q.m, q.n, q.k)) return FNN_OK;
    }
    const int shape = mb * 16 + nb;
    if (shape != 0x11 && shape != 0x12 && shape != 0x22 && shape != 0x24 && shape != 0x44) return FNN_OK;
    if (splits > p.ks.kblocks) splits = p.ks.kblocks;
    p.ks.kb_per_split = (p.ks.kblocks + splits - 1) / splits;
    p.ks.splits = (p.ks.kblocks + p.ks.kb_per_split - 1) / p.ks.kb_per_split;
    p.ks.seg = (p.ks.kb_per_split + FRAG_NW - 1) / FRAG_NW;
    p.ks.seg_last = (p.ks.kblocks - (p.ks.splits - 1) * p.ks.kb_per_split + FRAG_NW - 1) / FRAG_NW;
    p.mtiles = (int)((q.m + mb * 16 - 1) / (mb * 16));
    p.ntiles = (int)((q.n + nb * 16 - 1) / (nb * 16));
    p.rblocks = (int)((q.n + 15) / 16);
    p.m_pad = (int64_t)p.mtiles * mb * 16;
    p.by_mtiles = fast_div((uint32_t)p.mtiles);
    p.by_splits = fast_div((uint32_t)p.ks.splits);
    int rc;
    if ((rc = fnn_fragment_words(ctx, s, w, p.kblocks, &p.wf))) return rc;
    if (!p.wf) return FNN_OK;
    if ((rc = fnn_row_qsum(ctx, s, w, &p.wsum))) return rc;
    const int nsteps = p.ks.kblocks * 2;
    void *ws0 = nullptr, *ws1 = nullptr;
    if (!direct && (rc = fnn_ctx_ensure_tmp(ctx, 0, (size_t)p.m_pad * nsteps * 64, &ws0))) return rc;
    const size_t part_bytes = ((size_t)p.ks.splits * q.m * q.n * 4 + 255) / 256 * 256;
    if (p.ks.splits > 1 && (rc = fnn_ctx_ensure_tmp(ctx, 1, part_bytes + (size_t)p.ks.splits * p.m_pad * 4, &ws1))) return rc;
    *fnn_ctx_prepared(ctx) = FnnPreparedOperand{};
    p.af = (const int8_t *)ws0;
    p.part = (int32_t *)ws1;
    p.qsum = ws1 ? (int32_t *)((char *)ws1 + part_bytes) : nullptr;
    p.payload = q.payload;
    p.scales = q.scales; p.zeros = q.zeros; p.bias = q.bias; p.out = q.out; p.acc_out = q.acc_out;
    p.m = q.m; p.n = q.n; p.k = q.k; p.act = q.act;
    p.vec4 = q.n % 4 == 0 && !((reinterpret_cast<uintptr_t>(p.out) | reinterpret_cast<uintptr_t>(p.acc_out) | reinterpret_cast<uintptr_t>(p.scales) |
                                reinterpret_cast<uintptr_t>(p.zeros) | reinterpret_cast<uintptr_t>(p.bias) | reinterpret_cast<uintptr_t>(p.wsum)) & 15);
    if (!direct) {
        const dim3 grid((unsigned)((nsteps + 3) / 4), (unsigned)((q.m + 15) / 16));
        if (four) hipLaunchKernelGGL(frag_codes_kernel<true>, grid, dim3(256), 0, s, q.payload, q.m, q.k, nsteps, (uint4 *)ws0);
        else hipLaunchKernelGGL(frag_codes_kernel<false>, grid, dim3(256), 0, s, q.payload, q.m, q.k, nsteps, (uint4 *)ws0);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    }
    hipError_t e = four ? fnn_frag_int_launch_i4(mb, nb, p, s) : fnn_frag_int_launch_i8(mb, nb, p, s);
    if (e == hipSuccess && p.part) {
        hipLaunchKernelGGL(frag_codes_reduce_kernel, dim3((unsigned)((q.m * q.n + 255) / 256)), dim3(256), 0, s, p);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    *handled = true;
    return FNN_OK;
}
