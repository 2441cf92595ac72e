// Fragment-major MatMul kernel for a middle number of activation rows.
//
//   out[m,n] = act((sum_k A[m,k]*u(W[n,k]))*scale[n] + zero[n]*sum_k A[m,k] + bias[n])
//
// Both operands lie in memory in the order in which v_mfma_f32_16x16x32_f16 wants them in registers, so a wave's load is
// one contiguous KB that goes straight into operand registers: no LDS, no barrier and no address arithmetic in the K loop.
// Each of the eight waves of a workgroup takes an eighth of the workgroup's K range for the whole MB*16 x NB*16 output
// tile; the eight partial tiles meet in LDS once, at the end.
//
// Bound: the weight bytes and, at these sizes, the chain of a launch (first loads, K loop, meeting, epilogue); the matrix
// cores are busy 3 to 10 % of it.  Against the LDS tiles with their own preparation and
// reduction: U4 1003 x 3333 M = 77 14.0 -> 8.1 us (one launch), an MLP stack of eight F8 layers at 64 rows 253 -> 193 us.
#pragma once
#include "dech.h"
#include "qgemm_frag.h"

#include <type_traits>

namespace {

using namespace dech;

constexpr float FRAG_LO_UP = 2048.0f;
constexpr float FRAG_LO_DOWN = 1.0f / 2048.0f;   // the lo activation term is stored scaled by 2^11

// The eight partial tiles of a workgroup meet in LDS; scale, zero point, bias, activation, stores.
// sum[i]: sum of A[m,k] over this wave's segment, m = row 16 i + (lane & 15).
template <int MB, int NB, class SUM>
__device__ __forceinline__ void frag_finish(const FragArgs &p, unsigned mt, unsigned nt, unsigned z, const f32x4 (&total)[MB][NB],
                                            const SUM (&sum)[MB])
{
    extern __shared__ __attribute__((aligned(16))) f32x4 red[];   // [wave][tile][lane]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // D: column (lane & 15) = activation row, rows 4 (lane >> 4) + i = weight rows
    constexpr int TILES = MB * NB;
    __shared__ double xsum[FRAG_NW][MB * 16];
    if (lane < 16) {
#pragma unroll
        for (int i = 0; i < MB; i++) xsum[wv][i * 16 + lane] = sum[i];
    }
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
            red[(wv * TILES + i * NB + j) * 64 + lane] = total[i][j];
    // Output quads of this thread: quad c = 64 * tile + lane.  Their row and column constants are requested before the
    // barrier, their latency hides behind it.
    constexpr int QUADS = (TILES + FRAG_NW - 1) / FRAG_NW;
    const bool split = p.part != nullptr, has_bias = p.bias != nullptr && !split;
    int64_t om[QUADS], on[QUADS];
    float4 sc[QUADS], zp[QUADS], bi[QUADS];
    auto load4 = [&](const float *t, int64_t n) {
        if (p.vec4) return *reinterpret_cast<const float4 *>(t + n);
        const int64_t l = p.n - 1;
        return make_float4(t[n], t[n + 1 < l ? n + 1 : l], t[n + 2 < l ? n + 2 : l], t[n + 3 < l ? n + 3 : l]);
    };
#pragma unroll
    for (int r = 0; r < QUADS; r++) {
        const int c = tid + r * FRAG_NW * 64, t = c >> 6, ln = c & 63;
        om[r] = ((int64_t)mt * MB + t / NB) * 16 + (ln & 15);
        on[r] = ((int64_t)nt * NB + t % NB) * 16 + 4 * (ln >> 4);
        if (t >= TILES || om[r] >= p.m || on[r] >= p.n) { om[r] = -1; continue; }
        sc[r] = load4(p.scales, on[r]);
        zp[r] = load4(p.zeros, on[r]);
        bi[r] = has_bias ? load4(p.bias, on[r]) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < QUADS; r++) {
        if (om[r] < 0) continue;
        const int c = tid + r * FRAG_NW * 64;
        f32x4 v = red[c];
#pragma unroll
        for (int q = 1; q < FRAG_NW; q++) v += red[q * TILES * 64 + c];
        const int lrow = (c >> 6) / NB * 16 + (c & 15);
        double xd = xsum[0][lrow];
#pragma unroll
        for (int q = 1; q < FRAG_NW; q++) xd += xsum[q][lrow];
        const float xs = (float)xd;
        float d[4] = {v[0] * sc[r].x + zp[r].x * xs, v[1] * sc[r].y + zp[r].y * xs, v[2] * sc[r].z + zp[r].z * xs, v[3] * sc[r].w + zp[r].w * xs};
        float *o = p.out + om[r] * p.n + on[r];
        if (split) {
            o = p.part + ((int64_t)z * p.m + om[r]) * p.n + on[r];
        } else {
            if (has_bias) { d[0] = d[0] + bi[r].x; d[1] = d[1] + bi[r].y; d[2] = d[2] + bi[r].z; d[3] = d[3] + bi[r].w; }
            if (p.act != FNN_ACT_NONE) {
#pragma unroll
                for (int i = 0; i < 4; i++) d[i] = fnn_activation(d[i], p.act);
            }
        }
        if (p.vec4) {
            *reinterpret_cast<float4 *>(o) = make_float4(d[0], d[1], d[2], d[3]);
            if (p.residual && !split) {
                const int64_t at = om[r] * p.n + on[r];
                const float4 q = *reinterpret_cast<const float4 *>(p.residual + at);
                *reinterpret_cast<float4 *>(p.sum_out + at) = make_float4(d[0] + q.x, d[1] + q.y, d[2] + q.z, d[3] + q.w);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (on[r] + i >= p.n) continue;
                o[i] = d[i];
                if (p.residual && !split) {
                    const int64_t at = om[r] * p.n + on[r] + i;
                    p.sum_out[at] = d[i] + p.residual[at];
                }
            }
        }
    }
}

// of the 16 bytes `piece` of a row's last k block, the words that belong to the row
__device__ __forceinline__ void frag_own_words(u32x4 &w, int tail, int piece)
{
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (piece * 4 + e >= tail) w[e] = 0u;
}

// ROWS: the registered rows instead of the fragment-major copy (strides and ends that are known only at run time cost the
// others 1 %)
template <bool ROWS>
__device__ __forceinline__ const uint32_t *frag_row(const FragArgs &p, int rb, int lane)
{
    if constexpr (ROWS) return frag_row_at(p.wf, p.words_kp, (int)p.n, p.ks.kblocks, rb, lane & 15, lane >> 4);
    const int last_rb = ((int)p.n - 1) >> 4;
    return p.wf + ((int64_t)(rb < last_rb ? rb : last_rb) * p.ks.kblocks * 64 + lane) * 4;
}
template <bool ROWS>
__device__ __forceinline__ u32x4 frag_load(const FragArgs &p, const uint32_t *w0, int b)
{
    if constexpr (ROWS) return *reinterpret_cast<const frag_u32x4 *>(w0 + (int64_t)b * 16);
    return *reinterpret_cast<const u32x4 *>(w0 + (int64_t)b * 256);
}

template <int DT, int MB, int NB, bool ROWS>
__global__ void __launch_bounds__(FRAG_NW * 64) qgemm_frag_kernel(FragArgs p)
{
    using D = DecH<DT>;
    constexpr int SPB = D::WPS == 1 ? 4 : 2;   // steps of 32 k-values per k block (64 bytes of a weight row)
    constexpr int AR = 2;   // steps of the activations in flight
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // workgroup id -> tile.  Ids are dealt round-robin over the 8 XCDs: the row tiles of one column tile and split (the
    // readers of the same weights) have ids that agree modulo 8, so one L2 fetches those weights.
    const unsigned L = blockIdx.x;
    const unsigned grp = L >> 3, gq = p.by_mtiles.div(grp), mt = grp - gq * (unsigned)p.mtiles, u = gq * 8 + (L & 7);
    const unsigned nt = p.by_splits.div(u), z = u - nt * (unsigned)p.ks.splits;
    if (nt >= (unsigned)p.ntiles) return;

    int b0, b1;
    p.ks.segment((int)z, wv, &b0, &b1);

    f32x4 hi[MB][NB], lo[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) hi[i][j] = lo[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // The sum of a piece of K is scaled back by the row's power of two and joins the running sum before the next piece; the
    // largest tiles have no registers for a second set of sums, their segments are one piece.
    constexpr bool PIECES = MB * NB <= 8;
    f32x4 total[MB][NB];
    std::conditional_t<PIECES, double, float> xsum[MB];
    FragRow row[MB];   // of this lane's activation rows (lane & 15) in the current piece
    const FragRow *rows = p.rows + ((int64_t)z * FRAG_NW + wv) * p.ks.pieces * p.m_pad + (int64_t)mt * MB * 16 + (lane & 15);
    auto next_rows = [&] {
#pragma unroll
        for (int i = 0; i < MB; i++) row[i] = rows[i * 16];
        rows += p.m_pad;
    };
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < MB; i++) {
            xsum[i] += row[i].sum;
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float v = ldexpf(fmaf(lo[i][j][e], FRAG_LO_DOWN, hi[i][j][e]), -row[i].e);
                    if constexpr (PIECES) {
                        total[i][j][e] += v;
                        hi[i][j][e] = lo[i][j][e] = 0.0f;
                    } else {
                        total[i][j][e] = v;
                    }
                }
        }
    };
#pragma unroll
    for (int i = 0; i < MB; i++) {
        xsum[i] = 0;
        if constexpr (PIECES)
#pragma unroll
            for (int j = 0; j < NB; j++) total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (PIECES) next_rows();
    if (b0 < b1) {
        const int nsteps = p.ks.kblocks * SPB;
        const f16x8 *a0 = reinterpret_cast<const f16x8 *>(p.af) + (int64_t)mt * MB * nsteps * 128 + lane;
        const uint32_t *w0[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) w0[j] = frag_row<ROWS>(p, (int)nt * NB + j, lane);
        f16x8 a[AR][MB][2];
        u32x4 w[NB], wn[NB];
        auto load_a = [&](int s, f16x8(&d)[MB][2]) {
#pragma unroll
            for (int i = 0; i < MB; i++) {
                const f16x8 *q = a0 + ((int64_t)i * nsteps + s) * 128;
                d[i][0] = q[0];
                d[i][1] = q[64];
            }
        };
        auto load_w = [&](int b, u32x4(&d)[NB]) {
#pragma unroll
            for (int j = 0; j < NB; j++) d[j] = frag_load<ROWS>(p, w0[j], b);
        };
        // one k block; `last`: no requests past it
        auto block = [&](int b, auto last) {
            constexpr bool LAST = decltype(last)::value;
            if constexpr (!LAST) load_w(b + 1, wn);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < SPB; st++) {
                f16x8 wd[NB];
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    uint32_t ww[2];
                    ww[0] = w[j][st * D::WPS];
                    ww[1] = D::WPS == 2 ? w[j][st * D::WPS + 1] : 0u;
                    wd[j] = D::step(ww);
                }
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++) {
                        hi[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wd[j], a[st % AR][i][0], hi[i][j], 0, 0, 0);
                        lo[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wd[j], a[st % AR][i][1], lo[i][j], 0, 0, 0);
                    }
                __builtin_amdgcn_sched_barrier(0);
                if (!LAST || st + AR < SPB) load_a(b * SPB + st + AR, a[st % AR]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        load_w(b0, w);
#pragma unroll
        for (int r = 0; r < AR; r++) load_a(b0 * SPB + r, a[r]);
        // (the scheduler would sink every load to just before its use: the fences keep the requests where they are)
        __builtin_amdgcn_sched_barrier(0);
        int left = p.ks.piece;
        for (int b = b0; b < b1 - 1; b++) {
            block(b, std::false_type{});
#pragma unroll
            for (int j = 0; j < NB; j++) w[j] = wn[j];
            if (PIECES && --left == 0) {
                fold();
                next_rows();
                left = p.ks.piece;
            }
        }
        if (ROWS && b1 == p.ks.kblocks) {   // (wave-uniform) words of the next row: not a number, they would not vanish
#pragma unroll
            for (int j = 0; j < NB; j++) frag_own_words(w[j], p.words_kp - (b1 - 1) * 16, lane >> 4);
        }
        block(b1 - 1, std::true_type{});
    }
    if (!PIECES) next_rows();
    fold();
    frag_finish<MB, NB>(p, mt, nt, z, total, xsum);
}

// The same product with the f32 activations converted by the waves that multiply them: one launch instead of two, for
// products so small that a second launch costs more than converting a row block once per column tile.  A wave holds its
// whole segment (at most STEPS steps of 32 k-values) in registers, every load of it in flight at once.
template <int DT, int MB, int NB, int STEPS, bool ROWS>
__global__ void __launch_bounds__(FRAG_NW * 64) qgemm_frag_direct_kernel(FragArgs p)
{
    using D = DecH<DT>;
    constexpr int SPB = D::WPS == 1 ? 4 : 2;
    constexpr int BLOCKS = STEPS / SPB;
    constexpr bool IL = D::INTERLEAVED;
    static_assert(STEPS % SPB == 0 && STEPS >= SPB, "whole k blocks");
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned L = blockIdx.x;
    const unsigned grp = L >> 3, gq = p.by_mtiles.div(grp), mt = grp - gq * (unsigned)p.mtiles, nt = gq * 8 + (L & 7);
    if (nt >= (unsigned)p.ntiles) return;
    int b0, b1;
    p.ks.segment(0, wv, &b0, &b1);

    f32x4 hi[MB][NB], lo[MB][NB];
    FragRow row[MB];
#pragma unroll
    for (int i = 0; i < MB; i++) {
        row[i] = FragRow{0, 0.0f};
#pragma unroll
        for (int j = 0; j < NB; j++) hi[i][j] = lo[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (b0 < b1) {
        u32x4 w[BLOCKS][NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const uint32_t *w0 = frag_row<ROWS>(p, (int)nt * NB + j, lane);
#pragma unroll
            for (int b = 0; b < BLOCKS; b++) w[b][j] = frag_load<ROWS>(p, w0, b0 + b < b1 ? b0 + b : b1 - 1);
        }
        // a row past M asks for offset ~0, which the buffer's range check answers with zeros, like everything past the tensor
        const uint32_t K = (uint32_t)p.k;
        const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.a), 0, (int)((uint32_t)p.m * K * 4u), 0x00020000);
        float x[MB][STEPS][8];
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const uint32_t m = (mt * MB + i) * 16 + (lane & 15);
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                const uint32_t k0 = (uint32_t)(((b0 + s / SPB) * 4 + q) * SPB + s % SPB) * 8;
                const bool in = m < (uint32_t)p.m && k0 < K && b0 + s / SPB < b1;
                const uint32_t at = in ? (m * K + k0) * 4u : 0xffffffe0u;
                const u32x4 t0 = __builtin_amdgcn_raw_buffer_load_b128(xb, at, 0, 0), t1 = __builtin_amdgcn_raw_buffer_load_b128(xb, at, 16, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    x[i][s][j] = __uint_as_float(t0[j]);
                    x[i][s][4 + j] = __uint_as_float(t1[j]);
                }
            }
        }
        if (ROWS && b1 == p.ks.kblocks) {   // (wave-uniform; past the last block it is repeated)
#pragma unroll
            for (int b = 0; b < BLOCKS; b++)
                if (b0 + b >= b1 - 1)
#pragma unroll
                    for (int j = 0; j < NB; j++) frag_own_words(w[b][j], p.words_kp - (b1 - 1) * 16, q);
        }
        if (K % 8 != 0 && b1 == p.ks.kblocks) {   // (wave-uniform) the last values of a row run into the next row: they do not count
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int s = 0; s < STEPS; s++) {
                    const uint32_t k0 = (uint32_t)(((b0 + s / SPB) * 4 + q) * SPB + s % SPB) * 8;
#pragma unroll
                    for (int j = 0; j < 8; j++) x[i][s][j] = k0 + j < K ? x[i][s][j] : 0.0f;
                }
        }
#pragma unroll
        for (int i = 0; i < MB; i++) {
            float mx = 0.0f;
            double sum = 0.0;
#pragma unroll
            for (int s = 0; s < STEPS; s++) {
                const float(&v)[8] = x[i][s];
                mx = fmaxf(mx, fmaxf(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))),
                                     fmaxf(fmaxf(fabsf(v[4]), fabsf(v[5])), fmaxf(fabsf(v[6]), fabsf(v[7])))));
                sum += frag_sum8(v);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            sum += __shfl_xor(sum, 16, 64);
            sum += __shfl_xor(sum, 32, 64);
            int e = 0;
            if (mx > 0.0f && mx < __builtin_huge_valf()) {
                int ex;
                (void)frexpf(mx, &ex);
                e = 15 - ex;
            }
            row[i] = FragRow{e, (float)sum};
        }
#pragma unroll
        for (int s = 0; s < STEPS; s++) {
            f16x8 wd[NB];
#pragma unroll
            for (int j = 0; j < NB; j++) {
                uint32_t ww[2];
                ww[0] = w[s / SPB][j][(s % SPB) * D::WPS];
                ww[1] = D::WPS == 2 ? w[s / SPB][j][(s % SPB) * D::WPS + 1] : 0u;
                wd[j] = D::step(ww);
            }
#pragma unroll
            for (int i = 0; i < MB; i++) {
                f16x8 h, l;
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const float xs = ldexpf(x[i][s][IL ? (j & 1) * 4 + (j >> 1) : j], row[i].e);
                    const _Float16 hh = (_Float16)xs;
                    h[j] = hh;
                    l[j] = (_Float16)((xs - (float)hh) * FRAG_LO_UP);
                }
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    hi[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wd[j], h, hi[i][j], 0, 0, 0);
                    lo[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wd[j], l, lo[i][j], 0, 0, 0);
                }
            }
        }
    }
    f32x4 total[MB][NB];
    float xsum[MB];
#pragma unroll
    for (int i = 0; i < MB; i++) {
        xsum[i] = row[i].sum;
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) total[i][j][e] = 0.0f + ldexpf(fmaf(lo[i][j][e], FRAG_LO_DOWN, hi[i][j][e]), -row[i].e);
    }
    frag_finish<MB, NB>(p, mt, nt, 0, total, xsum);
}

template <int DT, int MB, int NB, bool ROWS>
hipError_t frag_launch_direct(const FragArgs &p, hipStream_t s)
{
    constexpr int SPB = DecH<DT>::WPS == 1 ? 4 : 2;
    const int steps = p.ks.seg_last * SPB;
    const dim3 grid(((unsigned)p.ntiles + 7) / 8 * 8 * (unsigned)p.mtiles), block(FRAG_NW * 64);
    constexpr int lds = FRAG_NW * MB * NB * 1024;
    if constexpr (SPB == 2)
        if (steps <= 2) { hipLaunchKernelGGL((qgemm_frag_direct_kernel<DT, MB, NB, 2, ROWS>), grid, block, lds, s, p); return hipGetLastError(); }
    if (steps <= 4) { hipLaunchKernelGGL((qgemm_frag_direct_kernel<DT, MB, NB, 4, ROWS>), grid, block, lds, s, p); return hipGetLastError(); }
    if constexpr (MB * NB <= 2)
        if (steps <= 8) { hipLaunchKernelGGL((qgemm_frag_direct_kernel<DT, MB, NB, 8, ROWS>), grid, block, lds, s, p); return hipGetLastError(); }
    return hipErrorInvalidValue;
}

template <int DT, int MB, int NB, bool ROWS>
hipError_t frag_launch_one(const FragArgs &p, hipStream_t s)
{
    constexpr int lds = FRAG_NW * MB * NB * 1024;
    auto kern = qgemm_frag_kernel<DT, MB, NB, ROWS>;
    if constexpr (lds > 64 * 1024) {
        static std::atomic<uint64_t> raised{0};
        const hipError_t e = fnn_raise_lds_limit(raised, reinterpret_cast<const void *>(kern), lds);
        if (e != hipSuccess) return e;
    }
    const unsigned groups = ((unsigned)(p.ntiles * p.ks.splits) + 7) / 8;
    hipLaunchKernelGGL(kern, dim3(groups * 8 * (unsigned)p.mtiles), dim3(FRAG_NW * 64), lds, s, p);
    return hipGetLastError();
}

template <int DT, bool ROWS>
hipError_t frag_launch_words(int mb, int nb, const FragArgs &p, hipStream_t s)
{
    if (p.a) {
        switch (mb * 16 + nb) {
        case 1 * 16 + 1: return frag_launch_direct<DT, 1, 1, ROWS>(p, s);
        case 1 * 16 + 2: return frag_launch_direct<DT, 1, 2, ROWS>(p, s);
        case 1 * 16 + 4: return frag_launch_direct<DT, 1, 4, ROWS>(p, s);
        default: return hipErrorInvalidValue;
        }
    }
    switch (mb * 16 + nb) {
    case 1 * 16 + 1: return frag_launch_one<DT, 1, 1, ROWS>(p, s);
    case 1 * 16 + 2: return frag_launch_one<DT, 1, 2, ROWS>(p, s);
    case 2 * 16 + 2: return frag_launch_one<DT, 2, 2, ROWS>(p, s);
    case 2 * 16 + 4: return frag_launch_one<DT, 2, 4, ROWS>(p, s);
    case 3 * 16 + 4: return frag_launch_one<DT, 3, 4, ROWS>(p, s);
    case 4 * 16 + 4:
        if constexpr (DecH<DT>::WPS == 2) return frag_launch_one<DT, 4, 4, ROWS>(p, s);   // (the four steps of a nibble block do not fit the registers beside it)
        return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
}

template <int DT>
hipError_t frag_launch(int mb, int nb, const FragArgs &p, hipStream_t s)
{
    return p.words_kp ? frag_launch_words<DT, true>(mb, nb, p, s) : frag_launch_words<DT, false>(mb, nb, p, s);
}

}  // namespace
