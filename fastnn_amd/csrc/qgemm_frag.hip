// Host side of the fragment-major MatMul (kernels: qgemm_frag_impl.h): the weight's fragment-major copy, the activation
// operand, the shape of the launch, the reduction of a K split.
//
// Launches: frag_prep_kernel (f32 rows -> f16 hi + lo fragments, row exponents and sums), qgemm_frag_kernel, and with K
// split over workgroups frag_reduce_kernel (partials added in split order: results do not depend on scheduling).
#include "mfma.h"
#include "qgemm_frag.h"
#include "qgemm_wave.h"
#include "range_io.h"

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));   // rows of any K: 16-byte loads from 4-byte aligned addresses

constexpr float LO_UP = 2048.0f;

// Registered rows -> fragment-major copy.  Bound: memory (a weight read and written once).  A wave moves COPY_BLOCKS
// blocks of 1 KB, all of its loads in flight: lane r + 16 q the piece q of row r, every store one contiguous KB.  Rows start on any
// word: 16-byte loads from 4-byte aligned addresses (the last row's may reach into the zeroed margin behind it), and what lies
// past the end of a row is cleared.
constexpr int COPY_BLOCKS = 4;
__global__ void __launch_bounds__(256) frag_words_kernel(const uint32_t *src, int64_t rows, int64_t kp, uint32_t kblocks, FastDiv by_kblocks, uint32_t blocks,
                                                         u32x4 *dst)
{
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const uint32_t first = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * COPY_BLOCKS;
    u32x4 v[COPY_BLOCKS];
    int left[COPY_BLOCKS];   // words of the piece that belong to the row
#pragma unroll
    for (int i = 0; i < COPY_BLOCKS; i++) {
        const uint32_t blk = first + i < blocks ? first + i : blocks - 1;   // (past the end: the last one again)
        const uint32_t rb = by_kblocks.div(blk), kb = blk - rb * kblocks;
        const int64_t row = (int64_t)rb * 16 + r, w0 = (int64_t)kb * 16 + q * 4;
        left[i] = row < rows ? (int)(kp - w0) : 0;
        v[i] = *reinterpret_cast<const frag_u32x4 *>(src + (row < rows ? row : rows - 1) * kp + w0);
    }
#pragma unroll
    for (int i = 0; i < COPY_BLOCKS; i++) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (e >= left[i]) v[i][e] = 0u;
        if (first + i < blocks) dst[(int64_t)(first + i) * 64 + lane] = v[i];
    }
}

struct FragPrepArgs {
    const float *a;              // [m,k], or
    FragArgs prev;               // the MatMul whose partial tiles are reduced here: its result (k columns) is what is converted
    int use_sum;                 // ... or that result plus prev.residual
    _Float16 *af;
    FragRow *rows;
    int64_t m, k, m_pad;
    FragSplit ks;
    int four_bit, interleaved;
};

// eight results of a MatMul from its partial tiles, columns n .. n + 7 of row m: split order, bias, activation
__device__ __forceinline__ void reduce8(const FragArgs &p, int64_t m, int64_t n, float(&v)[8])
{
    const int64_t total = p.m * p.n;
    const float4 *pp = reinterpret_cast<const float4 *>(p.part + m * p.n + n);
    float4 t0 = pp[0], t1 = pp[1];
    for (int z = 1; z < p.ks.splits; z++) {
        const float4 u0 = pp[(int64_t)z * (total / 4)], u1 = pp[(int64_t)z * (total / 4) + 1];
        t0.x += u0.x; t0.y += u0.y; t0.z += u0.z; t0.w += u0.w;
        t1.x += u1.x; t1.y += u1.y; t1.z += u1.z; t1.w += u1.w;
    }
    v[0] = t0.x; v[1] = t0.y; v[2] = t0.z; v[3] = t0.w; v[4] = t1.x; v[5] = t1.y; v[6] = t1.z; v[7] = t1.w;
    if (p.bias) {
        const float4 b0 = *reinterpret_cast<const float4 *>(p.bias + n), b1 = *reinterpret_cast<const float4 *>(p.bias + n + 4);
        v[0] = v[0] + b0.x; v[1] = v[1] + b0.y; v[2] = v[2] + b0.z; v[3] = v[3] + b0.w;
        v[4] = v[4] + b1.x; v[5] = v[5] + b1.y; v[6] = v[6] + b1.z; v[7] = v[7] + b1.w;
    }
    if (p.act != FNN_ACT_NONE) {
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = fnn_activation(v[j], p.act);
    }
}

// Activation fragments: one workgroup per block of 16 rows and piece of K.  A row's values of a piece share a power of
// two, so a workgroup needs nothing from the others; its waves take the piece's steps in turn, lane r + 16 q the eight values of row r that lane will hold as an operand:
// every store is one contiguous KB.  STEPS: steps per wave that stay in registers between the row maxima and the
// conversion; longer pieces read their values twice (never with CHAIN).
// CHAIN: the values are the result of the MatMul before, reduced from its partial tiles and stored here (with its sum
// with a residual), so that the reduction and the preparation of the next MatMul are one launch.
template <bool CHAIN, int STEPS, int NW>
__global__ void __launch_bounds__(NW * 64) frag_prep_kernel(FragPrepArgs p)
{
    // Row sums in double from eight values on: chained in f32 over a lane's steps, the waves and the pieces they were 1.1e-7 off
    // (2-norm, K = 1000 .. 6000; now 5e-8), and with a large zero point that is the error of the result.
    __shared__ float red[NW][16];
    __shared__ double part[NW][STEPS == 1 ? 64 : 16];   // one step per wave: per lane
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, r = lane & 15, q = lane >> 4;
    int b0, b1;
    p.ks.piece_at((int)blockIdx.x, &b0, &b1);
    if (b0 >= b1) {   // an empty piece: its row sums are read all the same
        if (tid < 16) p.rows[(int64_t)blockIdx.x * p.m_pad + (int64_t)blockIdx.y * 16 + tid] = FragRow{0, 0.0f};
        return;
    }
    const int64_t m = (int64_t)blockIdx.y * 16 + r, K = p.k;
    const int sh = p.four_bit ? 2 : 1;                       // log2 of the steps per k block
    const int s0 = b0 << sh, s1 = b1 << sh, nsteps = p.ks.kblocks << sh;
    auto first_k = [&](int s) { return ((((int64_t)(s >> sh) << 2) + q) << (sh + 3)) + ((s & ((1 << sh) - 1)) << 3); };
    auto load8 = [&](int s, float(&v)[8]) {
        const int64_t k0 = first_k(s);
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = 0.0f;
        if (s >= s1 || m >= p.m || k0 >= K) return;
        if constexpr (CHAIN) {   // (K % 8 == 0)
            reduce8(p.prev, m, k0, v);
            const int64_t at = m * K + k0;
            *reinterpret_cast<float4 *>(p.prev.out + at) = make_float4(v[0], v[1], v[2], v[3]);
            *reinterpret_cast<float4 *>(p.prev.out + at + 4) = make_float4(v[4], v[5], v[6], v[7]);
            if (p.prev.residual) {
                const float4 r0 = *reinterpret_cast<const float4 *>(p.prev.residual + at), r1 = *reinterpret_cast<const float4 *>(p.prev.residual + at + 4);
                const float4 s0_ = make_float4(v[0] + r0.x, v[1] + r0.y, v[2] + r0.z, v[3] + r0.w);
                const float4 s1_ = make_float4(v[4] + r1.x, v[5] + r1.y, v[6] + r1.z, v[7] + r1.w);
                *reinterpret_cast<float4 *>(p.prev.sum_out + at) = s0_;
                *reinterpret_cast<float4 *>(p.prev.sum_out + at + 4) = s1_;
                if (p.use_sum) { v[0] = s0_.x; v[1] = s0_.y; v[2] = s0_.z; v[3] = s0_.w; v[4] = s1_.x; v[5] = s1_.y; v[6] = s1_.z; v[7] = s1_.w; }
            }
        } else {
            const float *x = p.a + m * K + k0;
            if (k0 + 8 <= K) {
                const f4u t0 = *reinterpret_cast<const f4u *>(x), t1 = *reinterpret_cast<const f4u *>(x + 4);
                v[0] = t0[0]; v[1] = t0[1]; v[2] = t0[2]; v[3] = t0[3];
                v[4] = t1[0]; v[5] = t1[1]; v[6] = t1[2]; v[7] = t1[3];
            } else {
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (k0 + j < K) v[j] = x[j];
            }
        }
    };
    float keep[STEPS][8];
    float mx = 0.0f;
    double sum = 0.0;
    auto stats = [&](const float(&v)[8]) {
        mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))),
                             fmaxf(fmaxf(fabsf(v[4]), fabsf(v[5])), fmaxf(fabsf(v[6]), fabsf(v[7])))));
        sum += frag_sum8(v);
    };
    const bool in_regs = CHAIN || s1 - s0 <= NW * STEPS;
    if (in_regs) {
#pragma unroll
        for (int t = 0; t < STEPS; t++) load8(s0 + wv + NW * t, keep[t]);
#pragma unroll
        for (int t = 0; t < STEPS; t++) stats(keep[t]);
    } else {
        for (int s = s0 + wv; s < s1; s += NW) { load8(s, keep[0]); stats(keep[0]); }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if constexpr (STEPS == 1) {
        part[wv][lane] = sum;
    } else {
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        if (q == 0) part[wv][r] = sum;
    }
    if (q == 0) red[wv][r] = mx;
    __syncthreads();
#pragma unroll
    for (int w2 = 0; w2 < NW; w2++) mx = fmaxf(mx, red[w2][r]);
    int e = 0;
    if (mx > 0.0f && mx < __builtin_huge_valf()) {
        int ex;
        (void)frexpf(mx, &ex);
        e = 15 - ex;            // mx * 2^e in [2^14, 2^15)
    }
    auto convert = [&](int s, const float(&v)[8]) {
        f16x8 h, l;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int src = p.interleaved ? ((j & 1) * 4 + (j >> 1)) : j;   // the nibble decoders deliver k = 0,4,1,5,2,6,3,7
            const float xs = ldexpf(v[src], e);
            const _Float16 hh = (_Float16)xs;
            h[j] = hh;
            l[j] = (_Float16)((xs - (float)hh) * LO_UP);
        }
        _Float16 *d = p.af + (((int64_t)blockIdx.y * nsteps + s) * 2) * 512 + lane * 8;
        *reinterpret_cast<f16x8 *>(d) = h;
        *reinterpret_cast<f16x8 *>(d + 512) = l;
    };
    if (in_regs) {
#pragma unroll
        for (int t = 0; t < STEPS; t++)
            if (s0 + wv + NW * t < s1) convert(s0 + wv + NW * t, keep[t]);
    } else {
        for (int s = s0 + wv; s < s1; s += NW) { load8(s, keep[0]); convert(s, keep[0]); }
    }
    if (wv != 0) return;
    double t = 0.0;
#pragma unroll
    for (int w2 = 0; w2 < NW; w2++) t += part[w2][STEPS == 1 ? lane : r];
    if constexpr (STEPS == 1) {   // in the order of the kernel that converts for itself: the two give the same bits
        t += __shfl_xor(t, 16, 64);
        t += __shfl_xor(t, 32, 64);
    }
    if (q == 0) p.rows[(int64_t)blockIdx.x * p.m_pad + (int64_t)blockIdx.y * 16 + r] = FragRow{e, (float)t};
}

template <bool CHAIN>
hipError_t launch_frag_prep(const FragPrepArgs &a, hipStream_t s)
{
    const int steps = a.ks.piece << (a.four_bit ? 2 : 1);
    const dim3 grid((unsigned)(a.ks.splits * FRAG_NW * a.ks.pieces), (unsigned)((a.m + 15) / 16));
    if (steps <= 4) hipLaunchKernelGGL((frag_prep_kernel<CHAIN, 1, 4>), grid, dim3(256), 0, s, a);
    else if (steps <= 8) hipLaunchKernelGGL((frag_prep_kernel<CHAIN, 1, 8>), grid, dim3(512), 0, s, a);
    else if (steps <= 16) hipLaunchKernelGGL((frag_prep_kernel<CHAIN, 2, 8>), grid, dim3(512), 0, s, a);
    else hipLaunchKernelGGL((frag_prep_kernel<CHAIN, 4, 8>), grid, dim3(512), 0, s, a);
    return hipGetLastError();
}

// sum of the K-split partial tiles in split order + bias / activation; four columns per thread
__global__ void __launch_bounds__(256) frag_reduce_kernel(FragArgs p)
{
    const int64_t total = p.m * p.n;
    if (p.vec4) {
        const int64_t i4 = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (i4 * 4 >= total) return;
        const int64_t n = i4 * 4 % p.n;
        const float4 *pp = reinterpret_cast<const float4 *>(p.part) + i4;
        float4 d = pp[0];
        for (int z = 1; z < p.ks.splits; z++) {
            const float4 t = pp[(int64_t)z * (total / 4)];
            d.x += t.x; d.y += t.y; d.z += t.z; d.w += t.w;
        }
        float r[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (p.bias) r[j] = r[j] + p.bias[n + j];
            r[j] = fnn_activation(r[j], p.act);
        }
        reinterpret_cast<float4 *>(p.out)[i4] = make_float4(r[0], r[1], r[2], r[3]);
        if (p.residual) {
            const float4 q = reinterpret_cast<const float4 *>(p.residual)[i4];
            reinterpret_cast<float4 *>(p.sum_out)[i4] = make_float4(r[0] + q.x, r[1] + q.y, r[2] + q.z, r[3] + q.w);
        }
        return;
    }
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const int64_t n = i % p.n;
    float d = p.part[i];
    for (int z = 1; z < p.ks.splits; z++) d += p.part[(int64_t)z * total + i];
    if (p.bias) d = d + p.bias[n];
    d = fnn_activation(d, p.act);
    p.out[i] = d;
    if (p.residual) p.sum_out[i] = d + p.residual[i];
}

struct FragPlan {
    int mb, nb;
    int op_mb, op_nb;            // the tiles when the operand is in place (the same unless direct)
    FragSplit ks;
    int64_t m_pad;
    bool four_bit, direct;       // direct: activations converted by the MatMul kernel (then mb, nb, tiles are that kernel's)
    size_t op_bytes, ws_bytes;   // activation fragments; with the row tables behind them
};

// Microseconds a launch form takes: least squares over 97 000 measurements of 9 600 drawn calls (M 17 .. 2048, K 256 .. 16384,
// N 16 .. 16384, seven types; 7 % mean error, one launch 6 and 7 %; the form they choose is 0.5 to 2 % off the best one on average up
// to 160 rows).  The calls read their weights from the Infinity Cache (up to 300 MB of them in turn), those with weights of more
// than 4 MB also from memory (640 MB in turn): a fragment kernel loses 1.5 to 2.5 us on 17 MB from memory, the streaming kernel 0.5.
// What decides is the load of the busiest CU: the row tiles of a column tile and split go to one XCD (one L2 fetches their
// weights), so 18 column tiles are three for the 32 CUs of some XCD, not 2.25.  The load counts the operand bytes through the
// L1 and the matrix instructions, a round of resident workgroups the latency of its k blocks; per call the preparation, the K split's
// second launch and partials, output and weight bytes, and what an operand beyond an XCD's L2 (4 MB) costs to read again.
struct FragShape { int mb, nb, per_cu; };   // per_cu: workgroups that the registers and the LDS of a CU hold
constexpr FragShape kTwoLaunch[] = {{1, 1, 4}, {1, 2, 4}, {2, 2, 2}, {2, 4, 2}, {3, 4, 1}, {4, 4, 1}};
constexpr FragShape kDirect[] = {{1, 1, 0}, {1, 2, 0}, {1, 4, 0}};

int64_t cu_load(int64_t mtiles, int64_t columns) { return ((columns + 7) / 8 * mtiles + 31) / 32; }

float two_launch_us(FragShape t, int splits, int64_t m, int64_t n, int kblocks, bool four)
{
    static const float kFit[2][11] = {{4.83f, 0.1196f, 0.0985f, 0.0060f, 0.1715f, 0.1674f, 2.914f, 2.452f, 0.858f, 0.717f, 0.1457f},    // 8-bit
                                      {4.97f, 0.1057f, 0.1036f, 0.0101f, 0.2262f, 0.1137f, 3.695f, 2.346f, 0.587f, 0.721f, 0.1967f}};   // 4-bit
    static const float kAgain[2] = {0.59f, 1.53f};
    const float *c = kFit[four], kpb = four ? 128.f : 64.f, spb = four ? 4.f : 2.f, mn = (float)m * (float)n / 1e6f;
    const int64_t mt = (m + 16 * t.mb - 1) / (16 * t.mb), nt = (n + 16 * t.nb - 1) / (16 * t.nb);
    const int kps = (kblocks + splits - 1) / splits, sp = (kblocks + kps - 1) / kps;
    const int64_t load = cu_load(mt, nt * sp);
    const float l = (float)load, rounds = (float)((load + t.per_cu - 1) / t.per_cu), seg = (float)((kps + FRAG_NW - 1) / FRAG_NW);
    const float operand = 4.f * (float)m * (float)kblocks * kpb;
    const float again = operand > 4e6f ? (float)(mt * nt * sp) * seg * 8.f * (float)t.mb * 64.f * kpb / 1e8f * (1.f - 4e6f / operand) : 0.f;
    const float us = c[0] + l * (seg * (c[1] * (float)t.mb * spb + c[2] * (float)t.nb + c[3] * spb * (float)(t.mb * t.nb)) + c[5] * (float)(t.mb * t.nb)) +
                     c[4] * rounds * seg + c[6] * (float)m * (float)kblocks * kpb / 1e6f + (sp > 1 ? c[7] + c[8] * mn * (float)sp : 0.f) + c[9] * mn +
                     c[10] * (float)n * (float)kblocks * 64.f / 1e6f + kAgain[four] * again;
    // (a split is a third launch: below this a program that enqueues call by call waits for its own launches.  17 x 5184 x 391 I4:
    // four splits 9.1 us of the device, 11.5 a call, none 9.9 and 10.3)
    return sp > 1 && us < 11.5f ? 11.5f : us;
}

// The one launch: the busiest CU's steps, the chain of a wave, weight bytes, and the activations, which every column tile fetches
// and converts.  Negative: the form does not apply (eight steps, K of 1025 .. 2048, need the registers of the smaller tiles;
// from a load of eight on, which was not measured, the second launch is the better form).
float direct_us(FragShape t, int64_t m, int64_t n, int kblocks, bool four)
{
    static const float kFit[2][5] = {{2.75f, 0.0945f, 0.2591f, 0.0461f, 8.51f}, {1.91f, 0.0692f, 0.3642f, 0.0885f, 9.00f}};   // 8-bit, 4-bit
    const int seg = (kblocks + FRAG_NW - 1) / FRAG_NW, steps = seg * (four ? 4 : 2);
    const int64_t mt = (m + 16 * t.mb - 1) / (16 * t.mb), nt = (n + 16 * t.nb - 1) / (16 * t.nb), load = cu_load(mt, nt);
    if (steps > 8 || (steps > 4 && t.mb * t.nb > 2) || (m > 16 && load > 8)) return -1.f;
    const float *c = kFit[four], padded = steps <= 2 ? 2.f : (steps <= 4 ? 4.f : 8.f);
    return c[0] + c[1] * (float)load * padded * (float)t.nb + c[2] * padded + c[3] * (float)n * (float)kblocks * 64.f / 1e6f +
           c[4] * (float)(mt * t.mb * nt) * (float)kblocks * (four ? 128.f : 64.f) * 64.f / 1e8f;
}

// Which of its shapes: a fit that is twice as far off on average (10 %) but orders them better, 0.7 % off the best shape on average
// where that one is 1.2 % off.
float direct_order(FragShape t, int64_t m, int64_t n, int kblocks, bool four)
{
    static const float kFit[2][5] = {{0.1563f, 0.2627f, 0.f, 1.57f, 0.196f}, {0.f, 0.1852f, 0.0705f, 0.f, 0.443f}};   // 8-bit, 4-bit
    const int seg = (kblocks + FRAG_NW - 1) / FRAG_NW, steps = seg * (four ? 4 : 2);
    const float *c = kFit[four], padded = steps <= 2 ? 2.f : (steps <= 4 ? 4.f : 8.f);
    const float l = (float)cu_load((m + 16 * t.mb - 1) / (16 * t.mb), (n + 16 * t.nb - 1) / (16 * t.nb));
    return l * (c[0] * (float)(seg * t.nb) + padded * (c[1] + c[2] * (float)t.nb)) + c[3] * (float)m * (float)n / 1e6f + c[4] * padded;
}

// ... and what the kernel behind this one takes (from 9 rows on): the streaming kernel, that for 9 .. 16 rows, three digit planes or the f16 tiles.
// Negative: four digit planes.  They keep 30 bits of an activation and exact sums, hi + lo f16 rows 22 bits and f32 sums: the
// product of 4096 x 4096 I8 is 6.2e-8 off (2-norm, against 64 bits) there and 1.3e-7 here, so those calls stay there at any time.
// (q null: a call to come, of a type that has neither planes nor, from 33 rows on, the streaming kernel.)
float others_us(fnn_hip_ctx *ctx, const fnn_hip_weight *w, int64_t m, int flags, const QMatmulArgs *q)
{
    float us;
    if (q && m <= 32 && fnn_stream_takes(ctx, w, *q, flags, &us)) return us;
    if (m <= 16) return fnn_rows16_us(w->dtype, m, w->rows, w->inner);
    const int planes = fnn_digits_planes(ctx, w->dtype, m, w->rows, w->inner, flags);
    if (planes == 4) return -1.f;
    return planes == 3 ? fnn_digits3_us(w->dtype, m, w->rows, w->inner) : fnn_tiled_us(ctx, w->dtype, m, w->rows, w->inner, flags);
}

// K dealt out over `splits` and the bytes of the operand, for the plan's tiles
void frag_sizes(FragPlan *f, int64_t m, int splits)
{
    if (splits > f->ks.kblocks) splits = f->ks.kblocks;
    f->ks.kb_per_split = (f->ks.kblocks + splits - 1) / splits;
    f->ks.splits = (f->ks.kblocks + f->ks.kb_per_split - 1) / f->ks.kb_per_split;
    f->ks.seg = (f->ks.kb_per_split + FRAG_NW - 1) / FRAG_NW;
    f->ks.seg_last = (f->ks.kblocks - (f->ks.splits - 1) * f->ks.kb_per_split + FRAG_NW - 1) / FRAG_NW;
    f->m_pad = (m + f->op_mb * 16 - 1) / (f->op_mb * 16) * (f->op_mb * 16);
    // pieces of eight steps (256 k-values): a preparation workgroup per piece and row block
    const int seg = f->ks.seg > f->ks.seg_last ? f->ks.seg : f->ks.seg_last, eight = f->four_bit ? 2 : 4;
    f->ks.piece = f->op_mb * f->op_nb <= 8 && seg > eight ? eight : seg;
    f->ks.pieces = (seg + f->ks.piece - 1) / f->ks.piece;
    f->op_bytes = (size_t)f->m_pad * f->ks.kblocks * (f->four_bit ? 128 : 64) * 4;
    f->ws_bytes = f->op_bytes + (size_t)f->ks.splits * FRAG_NW * f->ks.pieces * f->m_pad * sizeof(FragRow);
}

// The launch for an [M, K] x [N, K]^T product with this weight; false: the call is not this kernel's.  The same for every
// call of the same sizes, so that the MatMul before can prepare the operand (q null: the call is not there yet).
bool frag_plan(fnn_hip_ctx *ctx, const fnn_hip_weight *w, int64_t m, int flags, const QMatmulArgs *q, FragPlan *out)
{
    const int64_t opt = fnn_ctx_option(ctx, FNN_OPT_FRAGMENT);
    if (opt < 0 || (flags & (FNN_FLAG_ACT_F16_SINGLE | FNN_FLAG_ACT_QUANT | FNN_FLAG_FORCE_GENERIC | FNN_FLAG_PREFER_FMA))) return false;
    const int dt = w->dtype;
    const int64_t n = w->rows, k = w->inner;
    if (dt < FNN_DT_I8 || dt > FNN_DT_F4 || m < 1 || m > (1 << 16) || n < 1 || n > (1 << 22) || k < 1 || k > (1 << 20)) return false;
    FragPlan f = {};
    f.four_bit = dt == FNN_DT_I4 || dt == FNN_DT_U4 || dt == FNN_DT_F4;
    f.ks.kblocks = (int)((w->kp + 15) / 16);
    const bool integer = dt == FNN_DT_I8 || dt == FNN_DT_I4 || dt == FNN_DT_U4;
    const int direct_steps = (f.ks.kblocks + FRAG_NW - 1) / FRAG_NW * (f.four_bit ? 4 : 2);
    const bool direct_ok = m * k < (int64_t)1 << 29;   // (32-bit buffer offsets)
    int splits = 1;
    if (opt > 0) {
        if (opt & FRAG_OPT_WAVE) return false;
        f.mb = (int)(opt & 15); f.nb = (int)((opt >> 4) & 15);
        splits = (int)((opt >> 8) & 15) > 0 ? (int)((opt >> 8) & 15) : 1;
        f.direct = (opt >> 15) & 1;
        bool known = false;
        if (f.direct) {
            for (FragShape t : kDirect) known |= t.mb == f.mb && t.nb == f.nb;
            known &= direct_ok && direct_steps <= 8 && (direct_steps <= 4 || f.mb * f.nb <= 2);
            splits = 1;
        } else {
            for (FragShape t : kTwoLaunch) known |= t.mb == f.mb && t.nb == f.nb && !(f.four_bit && t.mb * t.nb > 12);
        }
        if (!known) return false;
    } else {
        // Up to 8 rows of whole 16-byte pieces the one-launch kernels for few rows are ahead (up to four rows everywhere,
        // beyond where a segment is longer than four steps: 5 .. 8 rows F8 832 x 5749 5.4 us either way, 9 .. 16 rows
        // 960 x 5454 U8 7.4 against 5.7); ragged rows have no such kernel (2 x 4728 x 11904 F4: 233 us there, 14 here).
        // 9 .. 16 rows of longer segments by the times: the kernels behind convert the activations in every workgroup, in
        // whole rounds over the CUs; two launches convert them once.  2430 drawn calls of 9 .. 16 rows: 1.10 times as fast on
        // average, a third of them 1.4 times (3072 x 12288 I8, M = 16: 20.8 us there, 15.2 here), and 1.3e-7 off 64 bits where
        // those are 2.4e-7 (hi + lo rows of whole K slices) to 5.2e-7 (the streaming kernel's int8 rounds).
        const bool ragged = w->kp % 4 != 0 || k % 8 != 0;
        if (m > 2048 || !fnn_frag_options_untouched(ctx)) return false;
        if (m <= 8 && !ragged && (m <= 4 || direct_steps > 4 || integer)) return false;
        const bool by_time = m > 16 || (!ragged && direct_steps > 4);
        const float others = by_time ? others_us(ctx, w, m, flags, q) : 1e30f;
        if (others < 0.f) return false;
        float best = 1e30f, order = 1e30f;
        if (direct_ok && (m > 16 || !by_time))
            for (FragShape t : kDirect) {
                const float us = direct_us(t, m, n, f.ks.kblocks, f.four_bit), o = direct_order(t, m, n, f.ks.kblocks, f.four_bit);
                if (us >= 0.f && o < order) { order = o; best = us; f.mb = t.mb; f.nb = t.nb; f.direct = true; }
            }
        if (by_time || ragged)
            for (FragShape t : kTwoLaunch) {
                if ((t.mb - 1) * 16 >= m || (f.four_bit && t.mb * t.nb > 12)) continue;   // (a nibble block's four steps and that tile do not fit the registers)
                const int64_t wgs = ((m + 16 * t.mb - 1) / (16 * t.mb)) * ((n + 16 * t.nb - 1) / (16 * t.nb));
                for (int sp : {1, 2, 4, 8}) {
                    if (sp > 1 && (wgs * sp > 1024 || sp * 8 > f.ks.kblocks)) break;
                    float us = two_launch_us(t, sp, m, n, f.ks.kblocks, f.four_bit);
                    if (by_time && m <= 16 && us < 8.5f) us = 8.5f;   // (enqueued call by call, two launches take 7.5 to 8 us however small they are)
                    if (us >= (f.direct ? 0.96f * best : best)) continue;   // (about equal: the one launch)
                    best = us; f.mb = t.mb; f.nb = t.nb; f.direct = false; splits = sp;
                }
            }
        // (the margin: where the two are about equal the fits decide at random, and what was there stays.  With one half of the drawn
        // calls fitted, on the other half, weights of more than 4 MB, from memory / from cache: 17 .. 32 rows take 0.80 / 0.78 of the
        // others' time on average, 0.3 / 0.2 % of the calls lose more than 3 %; 33 .. 95 rows 0.75 / 0.72, 0.5 / 0.8 %; 161 .. 800 rows 0.95 / 0.95,
        // 1.6 / 1.5 %, the worst 1.17 times.  Fitted from the cache alone, 3.5 % of the calls of 17 .. 32 rows lost with weights
        // from memory (32 x 2048 x 8192 F8 12.6 us streamed, 14.1 here; 64 x 4096 x 11008 I4 25.5 on the LDS tiles, 29.4 here).  A wider
        // margin for operands beyond an XCD's L2 and from 500 rows on, where the fits are at their worst, halves what is lost there.)
        // (9 .. 16 rows: at 0.90 0.2 % of the drawn calls lose more than 3 %, 8 % at the worst; at 0.97 a sixth do.)
        const float margin = m <= 16 || m >= 500 || 4.f * (float)m * (float)f.ks.kblocks * (f.four_bit ? 128.f : 64.f) > 4e6f ? 0.90f : 0.97f;
        if (best > 1e29f || best > margin * others) return false;
        if (float us; fnn_wave_choice(w->dtype, m, n, k, &us) && best > margin * us) return false;
    }
    f.op_mb = f.mb; f.op_nb = f.nb;
    if (f.direct) {
        float best = 1e30f;
        for (FragShape t : kTwoLaunch) {
            const float us = (t.mb - 1) * 16 >= m || (f.four_bit && t.mb * t.nb > 12) ? 1e30f : two_launch_us(t, 1, m, n, f.ks.kblocks, f.four_bit);
            if (us < best) { best = us; f.op_mb = t.mb; f.op_nb = t.nb; }
        }
    }
    frag_sizes(&f, m, splits);
    *out = f;
    return true;
}

FragPrepArgs prep_args(const FragPlan &f, const fnn_hip_weight *w, int64_t m, void *ws)
{
    FragPrepArgs a = {};
    a.af = (_Float16 *)ws;
    a.rows = (FragRow *)((char *)ws + f.op_bytes);
    a.m = m; a.k = w->inner; a.m_pad = f.m_pad;
    a.ks = f.ks;
    a.four_bit = f.four_bit ? 1 : 0;
    a.interleaved = w->dtype == FNN_DT_I4 || w->dtype == FNN_DT_U4 ? 1 : 0;
    return a;
}

}  // namespace

// an option that names another kernel or its shape keeps the calls with that kernel
bool fnn_frag_options_untouched(fnn_hip_ctx *ctx)
{
    static const int opts[][2] = {{FNN_OPT_TILE_SHAPE, -1}, {FNN_OPT_TILE_SPLIT, 0}, {FNN_OPT_TILE_STAGES, 0}, {FNN_OPT_TILE_MIN_M, 5}, {FNN_OPT_GEMM_INT8, 1},
                                  {FNN_OPT_GEMM_INT8_MIN_M, 17}, {FNN_OPT_DIGIT_PLANES, 0}, {FNN_OPT_STREAM_MIN_M, 17}, {FNN_OPT_STREAM_MAX_M, 32},
                                  {FNN_OPT_STREAM_SHAPE, 0}, {FNN_OPT_ROWS16_ROW_TILES, 0}, {FNN_OPT_ROWS16_MIN_M, 9}, {FNN_OPT_GEMV_ROW_TILES, 0},
                                  {FNN_OPT_GEMV_INT8, 1}, {FNN_OPT_GEMV_INT8_MAX_M, 8}};
    for (const auto &o : opts)
        if (fnn_ctx_option(ctx, o[0]) != o[1]) return false;
    return true;
}

int fnn_fragment_words(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, int64_t kblocks, const uint32_t **out)
{
    *out = nullptr;
    fnn_hip_weight *wm = const_cast<fnn_hip_weight *>(w);
    if (fnn_ctx_option(ctx, FNN_OPT_GEMV_TILE_MAJOR) == 0) return FNN_OK;
    const int64_t blocks = (w->rows + 15) / 16 * kblocks;   // of 1 KB
    if (!wm->words_fr && blocks < (int64_t)1 << 31 && (wm->words_fr = (uint32_t *)fnn_ctx_copy_memory(ctx, (size_t)blocks * 1024 + 256))) {
        hipLaunchKernelGGL(frag_words_kernel, dim3((unsigned)((blocks + 4 * COPY_BLOCKS - 1) / (4 * COPY_BLOCKS))), dim3(256), 0, s, w->words, w->rows, w->kp,
                           (uint32_t)kblocks, fast_div((uint32_t)kblocks), (uint32_t)blocks, reinterpret_cast<u32x4 *>(wm->words_fr));
        if (hipGetLastError() != hipSuccess) {
            (void)hipFree(wm->words_fr);
            wm->words_fr = nullptr;
            return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, "building the fragment-major weight rows failed");
        }
    }
    *out = wm->words_fr;
    return FNN_OK;
}

int fnn_frag_words(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, int64_t kblocks, const uint32_t **words, int *kp)
{
    if (int rc = fnn_fragment_words(ctx, s, w, kblocks, words)) return rc;
    *kp = *words ? 0 : (int)w->kp;
    if (!*words) *words = w->words;   // (a load past the last registered row stays inside the zeroed margin behind it)
    return FNN_OK;
}

int fnn_frag_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &q, int flags, bool *handled)
{
    *handled = false;
    FragPlan f;
    if (q.words != w->words || q.n != w->rows || q.k != w->inner || !frag_plan(ctx, w, q.m, flags, &q, &f)) return FNN_OK;
    // What travels between the MatMuls of a plan (range_io.h): the operand may be in place, and the next one's may be asked
    // for.  From 33 rows on: below, the MatMuls that convert for themselves are ahead of a reduction launch each.  (Integer
    // weights as the next ones: their MatMul prepares its own operand.)
    FnnPrepIo *pio = fnn_ctx_prep_io(ctx);
    FnnPreparedOperand *have = fnn_ctx_prepared(ctx);
    const int interleaved = w->dtype == FNN_DT_I4 || w->dtype == FNN_DT_U4 ? 1 : 0;
    const bool handed = pio->offered && have->buffer && have->fragments == 1 + (f.four_bit ? 1 : 0) && have->a == q.a && have->m == q.m && have->k == q.k &&
                        have->rows_pad == f.m_pad && have->kpad == f.ks.kb_per_split && have->interleaved == interleaved;
    const bool direct = f.direct && !handed;
    // what does not fit is left to the kernels behind this one
    if ((!handed && !direct && !fnn_ctx_tmp_fits(ctx, 0, f.ws_bytes)) ||
        (f.ks.splits > 1 && !fnn_ctx_tmp_fits(ctx, 1, (size_t)f.ks.splits * q.m * q.n * 4))) return FNN_OK;
    FragArgs p = {};
    int rc;
    if ((rc = fnn_frag_words(ctx, s, w, f.ks.kblocks, &p.wf, &p.words_kp))) return rc;
    p.ks = f.ks; p.m_pad = f.m_pad; p.k = q.k;
    p.scales = q.scales; p.zeros = q.zeros; p.bias = q.bias; p.out = q.out;
    p.m = q.m; p.n = q.n; p.act = q.act;
    fnn_take_residual(ctx, q.out, q.m * q.n, &p.residual, &p.sum_out);
    p.vec4 = q.n % 4 == 0 && !((reinterpret_cast<uintptr_t>(p.out) | reinterpret_cast<uintptr_t>(p.residual) | reinterpret_cast<uintptr_t>(p.sum_out) |
                                reinterpret_cast<uintptr_t>(p.scales) | reinterpret_cast<uintptr_t>(p.zeros) | reinterpret_cast<uintptr_t>(p.bias)) & 15);
    const int mb = direct ? f.mb : f.op_mb, nb = direct ? f.nb : f.op_nb;
    p.mtiles = (int)((q.m + mb * 16 - 1) / (mb * 16));
    p.ntiles = (int)((q.n + nb * 16 - 1) / (nb * 16));
    p.by_mtiles = fast_div((uint32_t)p.mtiles);
    p.by_splits = fast_div((uint32_t)f.ks.splits);
    const int own_slot = handed ? have->slot : 0, next_slot = own_slot == 0 ? 4 : 0;
    void *ws0 = handed ? have->buffer : nullptr, *ws1 = nullptr, *next_ws = nullptr;
    FragPlan nf;
    const bool chain = pio->next_w && q.m >= 33 && p.vec4 && q.n % 8 == 0 && (pio->next_a == q.out || (p.residual && pio->next_a == p.sum_out)) &&
                       pio->next_w->inner == q.n && !fnn_ctx_static_mode(ctx) &&
                       (pio->next_w->dtype == FNN_DT_U8 || pio->next_w->dtype == FNN_DT_F8 || pio->next_w->dtype == FNN_DT_F8R || pio->next_w->dtype == FNN_DT_F4) &&
                       frag_plan(ctx, pio->next_w, q.m, pio->next_flags, nullptr, &nf) && nf.ks.piece << (nf.four_bit ? 2 : 1) <= 32 &&
                       fnn_ctx_ensure_tmp(ctx, next_slot, nf.ws_bytes, &next_ws) == FNN_OK && next_ws;
    if (!handed && !direct && (rc = fnn_ctx_ensure_tmp(ctx, 0, f.ws_bytes, &ws0))) return rc;
    if ((chain || f.ks.splits > 1) && (rc = fnn_ctx_ensure_tmp(ctx, 1, (size_t)f.ks.splits * q.m * q.n * 4, &ws1))) return rc;
    *have = FnnPreparedOperand{};   // (whatever was there is used by this call or stale)
    pio->consumed = handed ? 1 : 0;

    if (direct) p.a = q.a;
    else if (!ws0) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, "fragment MatMul: no operand buffer");
    FragPrepArgs a = prep_args(f, w, q.m, ws0);
    a.a = q.a;
    hipError_t e = handed || direct ? hipSuccess : launch_frag_prep<false>(a, s);
    if (e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    p.af = a.af; p.rows = a.rows;
    p.part = (float *)ws1;
    switch (w->dtype) {
    case FNN_DT_I8: e = fnn_frag_launch_i8(mb, nb, p, s); break;
    case FNN_DT_I4: e = fnn_frag_launch_i4(mb, nb, p, s); break;
    case FNN_DT_U8: e = fnn_frag_launch_u8(mb, nb, p, s); break;
    case FNN_DT_U4: e = fnn_frag_launch_u4(mb, nb, p, s); break;
    case FNN_DT_F8: e = fnn_frag_launch_f8(mb, nb, p, s); break;
    case FNN_DT_F8R: e = fnn_frag_launch_f8r(mb, nb, p, s); break;
    default: e = fnn_frag_launch_f4(mb, nb, p, s); break;
    }
    if (e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    if (chain) {
        FragPrepArgs na = prep_args(nf, pio->next_w, q.m, next_ws);
        na.prev = p;
        na.use_sum = pio->next_a == q.out ? 0 : 1;
        e = launch_frag_prep<true>(na, s);
        if (e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
        have->a = pio->next_a; have->buffer = next_ws; have->slot = next_slot;
        have->m = q.m; have->k = q.n; have->kpad = nf.ks.kb_per_split; have->rows_pad = nf.m_pad;
        have->fragments = 1 + (nf.four_bit ? 1 : 0); have->interleaved = na.interleaved;
        pio->produced = 1;
    } else if (p.part) {
        const int64_t items = p.vec4 ? q.m * q.n / 4 : q.m * q.n;
        hipLaunchKernelGGL(frag_reduce_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, p);
        if ((e = hipGetLastError()) != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    }
    *handled = true;
    return FNN_OK;
}
