// Fragment-major MatMul of I8 activations on the int8 matrix cores (exact i32 sums).  The organisation is that of qgemm_frag_impl.h: contiguous wave loads
// straight into the registers of v_mfma_i32_16x16x64_i8, the eight waves of a workgroup split its K range, one meeting in LDS.
// Bound: as there, bytes and the chain of a launch.  Against operand kernel + LDS tiles + formula as launches of their own,
// quantisation included: 64 x 2048 x 2048 19.4 -> 11.7 us, 256 x 4096 x 4096 28.9 -> 21.0.
#pragma once
#include <climits>
#include <type_traits>

#include "dech.h"
#include "qgemm_frag_int.h"

namespace {

using namespace dech;
typedef int i32x4v __attribute__((ext_vector_type(4)));

// DIRECT: the codes are read from the payload (16 rows x 64 bytes per
// wave load instead of one contiguous KB, but no preparation launch).
template <int DT, int MB, int NB, bool DIRECT>
__global__ void __launch_bounds__(FRAG_NW * 64) qgemm_frag_int_kernel(FragIntArgs p)
{
    using D = DecI<DT>;
    constexpr bool W8 = D::WPS == 4;                  // 8-bit weights: a group is two k blocks, else one
    constexpr int WL = W8 ? 2 : 1;
    constexpr int SHIFT = DT == FNN_DT_I4 ? 4 : 0;    // 4-bit signed lanes enter as 16 q
    extern __shared__ __attribute__((aligned(16))) i32x4v ired[];   // [wave][tile][lane]
    __shared__ int qs_red[FRAG_NW][MB * 16];   // row sums of the codes per wave
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned L = blockIdx.x;   // (ids to tiles as in qgemm_frag_kernel)
    const unsigned grp = L >> 3, gq = p.by_mtiles.div(grp), mt = grp - gq * (unsigned)p.mtiles, u = gq * 8 + (L & 7);
    const unsigned nt = p.by_splits.div(u), z = u - nt * (unsigned)p.ks.splits;
    if (nt >= (unsigned)p.ntiles) return;
    int g0, g1;
    p.ks.segment((int)z, wv, &g0, &g1);

    i32x4v acc[MB][NB];
    int qs[MB];
#pragma unroll
    for (int i = 0; i < MB; i++) {
        qs[i] = 0;
#pragma unroll
        for (int j = 0; j < NB; j++) acc[i][j] = i32x4v{0, 0, 0, 0};
    }
    if (g0 < g1) {
        const int nsteps = ((p.kblocks + WL - 1) / WL) * 2;
        const i32x4v *a0 = reinterpret_cast<const i32x4v *>(p.af) + (int64_t)mt * MB * nsteps * 64 + lane;
        const uint32_t K = (uint32_t)p.k;
        const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(DIRECT ? p.payload : (const uint8_t *)nullptr), 0,
                                                                            DIRECT ? (int)(8u + (uint32_t)p.m * K) : 0, 0x00020000);
        const u32x4 *w0[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) {
            int rb = (int)nt * NB + j;
            if (rb > p.rblocks - 1) rb = p.rblocks - 1;
            w0[j] = reinterpret_cast<const u32x4 *>(p.wf) + (int64_t)rb * p.kblocks * 64 + lane;
        }
        i32x4v a[2][MB];
        u32x4 w[NB][WL], wn[NB][WL];
        // first k-value of this lane's 16 in step st of group g
        auto first_k = [&](int g, int st) { return (uint32_t)(W8 ? 128 * g + 64 * st + 16 * q : 128 * g + 32 * q + 16 * st); };
        auto load_a = [&](int g, int st, i32x4v(&d)[MB]) {
#pragma unroll
            for (int i = 0; i < MB; i++) {
                if constexpr (DIRECT) {
                    const uint32_t m = (mt * MB + i) * 16 + (lane & 15), k0 = first_k(g, st);
                    const uint32_t at = m < (uint32_t)p.m && k0 < K ? 8u + m * K + k0 : 0xffffffe0u;   // (out of range: zeros)
                    d[i] = __builtin_bit_cast(i32x4v, __builtin_amdgcn_raw_buffer_load_b128(xb, at, 0, 0));
                } else {
                    d[i] = a0[((int64_t)i * nsteps + 2 * g + st) * 64];
                }
            }
        };
        auto load_w = [&](int g, u32x4(&d)[NB][WL]) {
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int b = 0; b < WL; b++) {
                    int kb = g * WL + b;
                    if (W8 && kb > p.kblocks - 1) kb = p.kblocks - 1;   // (an odd last block: the activations are zero there)
                    d[j][b] = w0[j][(int64_t)kb * 64];
                }
        };
        auto group = [&](int g, auto last) {
            constexpr bool LAST = decltype(last)::value;
            if constexpr (!LAST) load_w(g + 1, wn);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < 2; st++) {
                i32x4v wd[NB];
#pragma unroll
                for (int j = 0; j < NB; j++) {
                    uint32_t ww[4];
#pragma unroll
                    for (int e = 0; e < D::WPS; e++) ww[e] = W8 ? w[j][WL - 1 ? st : 0][e] : w[j][0][2 * st + (e & 1)];
                    wd[j] = __builtin_bit_cast(i32x4v, D::step(ww));
                }
                // DIRECT: what lies past K in the row's 16 bytes belongs to the next row; its weights are zero, but the
                // row sum must not count it.
                const uint32_t k0 = first_k(g, st);
                const bool tail = DIRECT && (uint32_t)(g + 1) * 128u > K;   // (wave-uniform)
#pragma unroll
                for (int i = 0; i < MB; i++) {
                    i32x4v v = a[st][i];
                    if (tail) {
                        const int n16 = (int)K - (int)k0;   // bytes of the 16 that count
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int nb = n16 - 4 * e;
                            v[e] &= nb >= 4 ? -1 : (nb <= 0 ? 0 : (int)((1u << (8 * nb)) - 1u));
                        }
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) qs[i] = __builtin_amdgcn_sdot4(v[e], 0x01010101, qs[i], false);
                    if constexpr (DIRECT && D::INTERLEAVED) {
                        const uint32_t x0 = (uint32_t)v[0], x1 = (uint32_t)v[1], x2 = (uint32_t)v[2], x3 = (uint32_t)v[3];
                        v[0] = (int)__builtin_amdgcn_perm(x1, x0, 0x06040200u);
                        v[1] = (int)__builtin_amdgcn_perm(x1, x0, 0x07050301u);
                        v[2] = (int)__builtin_amdgcn_perm(x3, x2, 0x06040200u);
                        v[3] = (int)__builtin_amdgcn_perm(x3, x2, 0x07050301u);
                    }
                    if constexpr (DIRECT) a[st][i] = v;
                }
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int j = 0; j < NB; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wd[j], a[st][i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (!LAST) load_a(g + 1, st, a[st]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        load_w(g0, w);
        load_a(g0, 0, a[0]);
        load_a(g0, 1, a[1]);
        __builtin_amdgcn_sched_barrier(0);
        for (int g = g0; g < g1 - 1; g++) {
            group(g, std::false_type{});
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int b = 0; b < WL; b++) w[j][b] = wn[j][b];
        }
        group(g1 - 1, std::true_type{});
    }
    constexpr int TILES = MB * NB;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++) ired[(wv * TILES + i * NB + j) * 64 + lane] = acc[i][j];
#pragma unroll
    for (int i = 0; i < MB; i++) {
        int t = qs[i];
        t += __shfl_xor(t, 16, 64);
        t += __shfl_xor(t, 32, 64);
        if (lane < 16) qs_red[wv][i * 16 + lane] = t;
    }
    // the constants of this thread's output quads, requested before the barrier
    constexpr int QUADS = (TILES + FRAG_NW - 1) / FRAG_NW;
    const bool split = p.part != nullptr, has_bias = p.bias != nullptr && !split;
    int64_t om[QUADS], on[QUADS];
    float4 sc[QUADS], zp[QUADS], bi[QUADS];
    int4 wsum[QUADS];
    auto load4 = [&](const float *t, int64_t n) {
        if (p.vec4) return *reinterpret_cast<const float4 *>(t + n);
        const int64_t l = p.n - 1;
        return make_float4(t[n], t[n + 1 < l ? n + 1 : l], t[n + 2 < l ? n + 2 : l], t[n + 3 < l ? n + 3 : l]);
    };
    float sa = 0.0f, za = 0.0f;
    if (!split) {
        sa = reinterpret_cast<const float *>(p.payload)[0];
        za = reinterpret_cast<const float *>(p.payload)[1];
    }
#pragma unroll
    for (int r = 0; r < QUADS; r++) {
        const int c = tid + r * FRAG_NW * 64, t = c >> 6, ln = c & 63;
        om[r] = ((int64_t)mt * MB + t / NB) * 16 + (ln & 15);
        on[r] = ((int64_t)nt * NB + t % NB) * 16 + 4 * (ln >> 4);
        if (t >= TILES || om[r] >= p.m || on[r] >= p.n) { om[r] = -1; continue; }
        if (split) continue;
        const float4 ws = load4(reinterpret_cast<const float *>(p.wsum), on[r]);
        wsum[r] = make_int4(__float_as_int(ws.x), __float_as_int(ws.y), __float_as_int(ws.z), __float_as_int(ws.w));
        sc[r] = load4(p.scales, on[r]);
        zp[r] = load4(p.zeros, on[r]);
        bi[r] = has_bias ? load4(p.bias, on[r]) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
    if (split && nt == 0 && tid < MB * 16) {   // the row sums of this split
        int qsum = 0;
#pragma unroll
        for (int q2 = 0; q2 < FRAG_NW; q2++) qsum += qs_red[q2][tid];
        p.qsum[(int64_t)z * p.m_pad + (int64_t)mt * MB * 16 + tid] = qsum;
    }
#pragma unroll
    for (int r = 0; r < QUADS; r++) {
        if (om[r] < 0) continue;
        const int c = tid + r * FRAG_NW * 64;
        const int64_t at = om[r] * p.n + on[r];
        float d[4];
        int iv[4];
        i32x4v v = ired[c];
#pragma unroll
        for (int q2 = 1; q2 < FRAG_NW; q2++) v += ired[q2 * TILES * 64 + c];
#pragma unroll
        for (int i = 0; i < 4; i++) iv[i] = v[i] >> SHIFT;
        if (!split) {
            const int lrow = (c >> 6) / NB * 16 + (c & 15);
            int qsum = 0;
#pragma unroll
            for (int q2 = 0; q2 < FRAG_NW; q2++) qsum += qs_red[q2][lrow];
            // dot * sw + zw * input_sum, dot = acc * sa (+ za * sum q_w), input_sum = sa * sum q_a + K * za
            const float input_sum = (float)qsum * sa + (float)p.k * za;
            const int ws[4] = {wsum[r].x, wsum[r].y, wsum[r].z, wsum[r].w};
            const float sw[4] = {sc[r].x, sc[r].y, sc[r].z, sc[r].w}, zw[4] = {zp[r].x, zp[r].y, zp[r].z, zp[r].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float dot = za != 0.0f ? (float)iv[i] * sa + za * (float)ws[i] : (float)iv[i] * sa;
                d[i] = dot * sw[i] + zw[i] * input_sum;
            }
        }
        if (split) {
            int32_t *o = p.part + (int64_t)z * p.m * p.n + at;
            if (p.vec4) *reinterpret_cast<int4 *>(o) = make_int4(iv[0], iv[1], iv[2], iv[3]);
            else
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (on[r] + i < p.n) o[i] = iv[i];
            continue;
        }
        if (has_bias) { d[0] = d[0] + bi[r].x; d[1] = d[1] + bi[r].y; d[2] = d[2] + bi[r].z; d[3] = d[3] + bi[r].w; }
        if (p.act != FNN_ACT_NONE) {
#pragma unroll
            for (int i = 0; i < 4; i++) d[i] = fnn_activation(d[i], p.act);
        }
        if (za != 0.0f) iv[0] = iv[1] = iv[2] = iv[3] = 0;
        if (p.vec4) {
            *reinterpret_cast<float4 *>(p.out + at) = make_float4(d[0], d[1], d[2], d[3]);
            if (p.acc_out) *reinterpret_cast<int4 *>(p.acc_out + at) = make_int4(iv[0], iv[1], iv[2], iv[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (on[r] + i >= p.n) continue;
                p.out[at + i] = d[i];
                if (p.acc_out) p.acc_out[at + i] = iv[i];
            }
        }
    }
}

template <int DT, int MB, int NB, bool DIRECT>
hipError_t frag_int_launch_one(const FragIntArgs &p, hipStream_t s)
{
    constexpr int lds = FRAG_NW * MB * NB * 1024;
    auto kern = qgemm_frag_int_kernel<DT, MB, NB, DIRECT>;
    if constexpr (lds > 64 * 1024) {
        static std::atomic<uint64_t> raised{0};
        const hipError_t e = fnn_raise_lds_limit(raised, reinterpret_cast<const void *>(kern), lds);
        if (e != hipSuccess) return e;
    }
    const unsigned groups = ((unsigned)(p.ntiles * p.ks.splits) + 7) / 8;
    hipLaunchKernelGGL(kern, dim3(groups * 8 * (unsigned)p.mtiles), dim3(FRAG_NW * 64), lds, s, p);
    return hipGetLastError();
}

template <int DT, bool DIRECT>
hipError_t frag_int_launch_shape(int mb, int nb, const FragIntArgs &p, hipStream_t s)
{
    switch (mb * 16 + nb) {
    case 1 * 16 + 1: return frag_int_launch_one<DT, 1, 1, DIRECT>(p, s);
    case 1 * 16 + 2: return frag_int_launch_one<DT, 1, 2, DIRECT>(p, s);
    case 2 * 16 + 2: return frag_int_launch_one<DT, 2, 2, DIRECT>(p, s);
    case 2 * 16 + 4: return frag_int_launch_one<DT, 2, 4, DIRECT>(p, s);
    case 4 * 16 + 4: return frag_int_launch_one<DT, 4, 4, DIRECT>(p, s);
    default: return hipErrorInvalidValue;
    }
}

template <int DT>
hipError_t frag_int_launch(int mb, int nb, const FragIntArgs &p, hipStream_t s)
{
    return p.af ? frag_int_launch_shape<DT, false>(mb, nb, p, s) : frag_int_launch_shape<DT, true>(mb, nb, p, s);
}

}  // namespace
