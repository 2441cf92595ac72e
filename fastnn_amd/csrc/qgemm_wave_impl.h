// Int8 MatMul for many activation rows: one wave per SIMD with a large register tile, operands straight from memory.
//
// Bound: the matrix cores (v_mfma_i32_32x32x32_i8, 32 clocks each; MFMAs alone sustain 3.1 to 3.4 POP/s here) and, close behind, the 64 B/clk that a CU's L1 delivers: a wave tile of 96 x 128 (three digit planes of 32 activation
// rows) asks for 224 bytes per k-value with 8-bit and 160 with 4-bit weights against 12 clocks of its SIMD's matrix core, so
// the four waves of a CU need 14 and 10 clocks of L1 time in the same 12.  No LDS, no barrier: the operands lie in memory in
// fragment order, a wave's load is contiguous, and RING steps of 32 k-values are in flight per wave.  What is left at large M
// is the epilogue, which nothing overlaps at one wave per SIMD (7 to 12 us per round of tiles), and a matrix core that is
// busy half the time: I8 4096 x 4096 M = 2048 1.88 POP/s, matrix cores busy 47 % of the launch's clocks, waves waiting 24 % of
// theirs; M = 256 (one tile per CU, a chain of latencies) 21 % and 31 %.
// Measured against the LDS tiles of qgemm_digits.hip: I8 4096 x 4096 M = 256 29.6 -> 27.4 us, M = 1024 72.5 -> 65.5,
// M = 2048 130.6 -> 122; I8 4096 x 11008 M = 700 131 -> 111; I4 4096 x 4096 M = 256 27.2 -> 23.6.  Row blocks an odd number
// of pieces apart, to spread them over the L2's channels, gained nothing (122 -> 127 us).
#pragma once
#include <climits>
#include <type_traits>

#include "dech.h"
#include "qgemm_wave.h"

namespace {

using namespace dech;
typedef int wi32x4 __attribute__((ext_vector_type(4)));
typedef int wi32x16 __attribute__((ext_vector_type(16)));
typedef float wf32x4 __attribute__((ext_vector_type(4)));

// Operand rows in groups of 24 = 8 activation rows x 3 planes (plane j in rows [8j, 8j + 8) of the group).  WK: waves of the
// four that share an output tile and split K (they meet in LDS at the end); the others lie side by side (WK = 1: 2 x 2,
// WK = 2: 1 x 2).
// rg0, cg0: first group of 32 activation rows and of 128 columns of the workgroup
template <int DT, int WK>
__device__ __forceinline__ void wave_tile(const WaveArgs &p, unsigned rg0, unsigned cg0, int units_per_wave)
{
    using D = DecI<DT>;
    constexpr int TM = WAVE_ROWS * 3 / 32, TN = WAVE_COLS / 32;   // blocks of 32 x 32
    constexpr bool W8 = D::WPS == 4;
    constexpr int RING = WAVE_RING(W8);                // steps in flight, and the unit in which K is dealt out
    constexpr int SHIFT = DT == FNN_DT_I4 ? 4 : 0;     // 4-bit signed lanes enter as 16 q
    constexpr int WL = W8 ? RING : RING / 2;           // weight loads per ring: a 16-byte piece is one step or two
    extern __shared__ __attribute__((aligned(16))) wf32x4 wred[];   // [wave][group of rows][column block][lane]
    __shared__ __attribute__((aligned(16))) int2 row_const[4][WAVE_ROWS];
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, h = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = WK == 1 ? 0 : (WK == 2 ? wv >> 1 : wv);
    const int wm = WK == 1 ? wv >> 1 : 0, wn = WK == 4 ? 0 : wv & 1;
    constexpr int WN = WK == 4 ? 1 : 2;
    const int rb0 = (int)(rg0 + wm) * TM;                  // first block of 32 operand rows
    const int64_t m0 = (int64_t)(rg0 + wm) * WAVE_ROWS;    // first activation row
    const int64_t n0 = (int64_t)(cg0 + wn) * WAVE_COLS;
    const int u0 = wk * units_per_wave, u1 = u0 + units_per_wave < p.units ? u0 + units_per_wave : p.units;

    wi32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0;

    // Row and column constants of the outputs: requested before the last unit, so that the epilogue, which nothing overlaps
    // on this SIMD, does not begin with a trip to memory.
    float sc[TN], zp[TN], bi[TN];
    int rexp = 0;
    float xsum = 0.0f;
    auto load_constants = [&] {
        rexp = p.rexp[m0 + lr];   // (rows past M lie inside the tables)
        xsum = p.xsum[m0 + lr];
#pragma unroll
        for (int j = 0; j < TN; j++) {
            int64_t n = n0 + j * 32 + lr;
            if (n > p.n - 1) n = p.n - 1;
            sc[j] = p.scales[n];
            zp[j] = p.zeros[n];
            bi[j] = p.bias ? p.bias[n] : 0.0f;
        }
    };

    if (u0 < u1) {
        const wi32x4 *a0 = reinterpret_cast<const wi32x4 *>(p.af) + (int64_t)rb0 * p.nsteps * 64 + lane;
        const int block_words = p.words_kp ? 16 : 256, pair_words = p.words_kp ? 8 : 128;
        const uint32_t *w0[TN];   // two row blocks and a pair of pieces per load
#pragma unroll
        for (int j = 0; j < TN; j++) w0[j] = frag_row_at(p.wf, p.words_kp, (int)p.n, p.kblocks, (int)(n0 >> 4) + 2 * j + (lr >> 4), lr & 15, h);
        wi32x4 a[RING][TM];
        u32x4 w[WL][TN];
        auto load_a = [&](int s, int i) { return a0[((int64_t)i * p.nsteps + s) * 64]; };
        // piece x of a row: k block x / 2, q = 2 (x & 1) + h
        auto load_w = [&](int x, int j) {
            int kb = x >> 1;
            if (kb > p.kblocks - 1) kb = p.kblocks - 1;   // (past the last block the activations are zero)
            return (u32x4)*reinterpret_cast<const frag_u32x4 *>(w0[j] + (int64_t)kb * block_words + (x & 1) * pair_words);
        };
        auto decode = [&](int st, int j) {
            uint32_t ww[4];
#pragma unroll
            for (int e = 0; e < D::WPS; e++) ww[e] = W8 ? w[W8 ? st : 0][j][e] : w[W8 ? 0 : st / 2][j][2 * (st & 1) + (e & 1)];
            return __builtin_bit_cast(wi32x4, D::step(ww));
        };
        // One ring of steps.  A step's matrix instructions carry, one by one between them, the requests that refill what the
        // step before has used up and the decoding of the next step's weights: issued in a bunch they leave the matrix core
        // idle while the four waves' requests queue for the L1 (2048 x 4096 x 4096 I8: 113 us).
        wi32x4 wd[2][TN];
        auto unit = [&](int u, auto last) {
            constexpr bool LAST = decltype(last)::value;
#pragma unroll
            for (int st = 0; st < RING; st++) {
                constexpr int NM = TM * TN;
                const bool want_a = !LAST || st == 0;
                const bool want_w = want_a && (W8 || st % 2 == 0);
                const int sp = (st + RING - 1) % RING, step = (st == 0 ? u : u + 1) * RING + sp;   // slot to refill, its step
                const int wp = W8 ? sp : sp / 2, piece = W8 ? step : step / 2;
#pragma unroll
                for (int x = 0; x < NM; x++) {
                    const int i = x / TN, j = x % TN;
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[st][i], wd[st & 1][j], acc[i][j], 0, 0, 0);
                    // requests 0 .. TM + TN - 1 at equal distances, then the next step's decoding
#pragma unroll
                    for (int r = 0; r < TM + TN; r++)
                        if (r * NM / (TM + TN) == x) {
                            if (r < TM) { if (want_a) a[sp][r] = load_a(step, r); }
                            else if (want_w) w[wp][r - TM] = load_w(piece, r - TM);
                        }
                    if (x >= NM - TN && (!LAST || st < RING - 1)) wd[(st + 1) & 1][x - (NM - TN)] = decode((st + 1) % RING, x - (NM - TN));
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
#pragma unroll
        for (int st = 0; st < RING - 1; st++) {
#pragma unroll
            for (int i = 0; i < TM; i++) a[st][i] = load_a(u0 * RING + st, i);
            if (W8 || st % 2 == 0)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    if (W8 || st / 2 < WL - 1) w[W8 ? st : st / 2][j] = load_w(W8 ? u0 * RING + st : u0 * WL + st / 2, j);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < TN; j++) wd[0][j] = decode(0, j);
        for (int u = u0; u < u1 - 1; u++) unit(u, std::false_type{});
        load_constants();
        unit(u1 - 1, std::true_type{});
    } else {
        load_constants();
    }

    // D: acc[i][j][e] is operand row 32 i + (e / 4) * 8 + h * 4 + e % 4, column 32 j + lr.
    // A value of this lane, (row 8 g + 4 h + t, column block j): the three planes of one activation row combined
    auto value = [&](int g, int t, int j) {
        float v = 0.0f;
#pragma unroll
        for (int d = 2; d >= 0; d--) {
            const int slab = 3 * g + d;
            v = fmaf(v, 256.0f, (float)acc[slab >> 2][j][(slab & 3) * 4 + t]);
        }
        return v;
    };
    if (h == 0) row_const[wv][lr] = make_int2(rexp, __float_as_int(xsum));
    // The waves that split K hand each other their sums through LDS, four rows of a column as one piece, and share the groups of rows.
    // Then scale, bias, activation and stores, each in a pass of its own with its uniform test in front: nothing overlaps this part at one
    // wave per SIMD, and a wave fetches its code to run it once (0.25 us a KB).  Against single values
    // through LDS and the formula in a loop over rows, the kernel alone: I8 4096 x 4096 M = 256 19.6 -> 18.6 us, M = 2048 108 -> 102, 2048 x 8192
    // M = 1024 66 -> 59, I4 4096 x 4096 M = 1536 83 -> 78.
    constexpr int OWN = 4 / WK;   // groups of rows that this wave finishes
    float o[OWN][4][TN];
    if constexpr (WK == 1) {
#pragma unroll
        for (int x = 0; x < OWN; x++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int j = 0; j < TN; j++) o[x][t][j] = value(x, t, j);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
#pragma unroll
        for (int g = 0; g < 4; g++)
#pragma unroll
            for (int j = 0; j < TN; j++) wred[((wv * 4 + g) * TN + j) * 64 + lane] = wf32x4{value(g, 0, j), value(g, 1, j), value(g, 2, j), value(g, 3, j)};
        __syncthreads();
        const wf32x4 *q = wred + ((wn * 4 + wk * OWN) * TN) * 64 + lane;   // (the partners lie WN waves apart)
#pragma unroll
        for (int x = 0; x < OWN; x++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                wf32x4 v = q[(x * TN + j) * 64];
#pragma unroll
                for (int y = 1; y < WK; y++) v += q[((y * WN * 4 + x) * TN + j) * 64];
#pragma unroll
                for (int t = 0; t < 4; t++) o[x][t][j] = v[t];
            }
    }
#pragma unroll
    for (int x = 0; x < OWN; x++) {
        const wi32x4 *rc = reinterpret_cast<const wi32x4 *>(&row_const[wv][(wk * OWN + x) * 8 + h * 4]);
        const wi32x4 r01 = rc[0], r23 = rc[1];
        const int re[4] = {r01[0], r01[2], r23[0], r23[2]}, rs[4] = {r01[1], r01[3], r23[1], r23[3]};
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int j = 0; j < TN; j++) {
                const float d = re[t] == INT_MIN ? __builtin_nanf("") : ldexpf(o[x][t][j], -re[t] - SHIFT);   // (a non-finite row)
                o[x][t][j] = fmaf(zp[j], __int_as_float(rs[t]), d * sc[j]);
            }
    }
    auto every = [&](auto f) {
#pragma unroll
        for (int x = 0; x < OWN; x++)
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int j = 0; j < TN; j++) f(x, t, j);
    };
    if (p.bias) every([&](int x, int t, int j) { o[x][t][j] = o[x][t][j] + bi[j]; });
    auto activate = [&](auto a) { every([&](int x, int t, int j) { o[x][t][j] = fnn_activation(o[x][t][j], decltype(a)::value); }); };
    if (p.act == FNN_ACT_SILU) activate(std::integral_constant<int, FNN_ACT_SILU>{});
    else if (p.act == FNN_ACT_GELU) activate(std::integral_constant<int, FNN_ACT_GELU>{});
    else if (p.act == FNN_ACT_RELU) activate(std::integral_constant<int, FNN_ACT_RELU>{});
    const int64_t base = (m0 + wk * OWN * 8) * p.n + n0;                   // (uniform)
    const uint32_t lane_at = (uint32_t)(4 * h) * (uint32_t)p.n + (uint32_t)lr;
    const bool whole = m0 + WAVE_ROWS <= p.m && n0 + WAVE_COLS <= p.n;
    const int rows = (int)(p.m - m0 < WAVE_ROWS ? p.m - m0 : WAVE_ROWS) - wk * OWN * 8 - 4 * h, cols = (int)(p.n - n0 < WAVE_COLS ? p.n - n0 : WAVE_COLS) - lr;
    auto store = [&](float *dst) {
        if (whole) every([&](int x, int t, int j) { (dst + base + (int64_t)(x * 8 + t) * p.n)[lane_at + j * 32] = o[x][t][j]; });
        else
            every([&](int x, int t, int j) {
                if (x * 8 + t < rows && j * 32 < cols) (dst + base + (int64_t)(x * 8 + t) * p.n)[lane_at + j * 32] = o[x][t][j];
            });
    };
    store(p.out);
    if (p.residual) {
        every([&](int x, int t, int j) {
            if (x * 8 + t < rows && j * 32 < cols) o[x][t][j] = o[x][t][j] + (p.residual + base + (int64_t)(x * 8 + t) * p.n)[lane_at + j * 32];
        });
        store(p.sum_out);
    }
}

// The tiles' last round: 96 of 256 CUs busy for as long as the others were costs most of a round, so the tiles behind the whole rounds (TAIL > 0) are cut
// into the smaller ones of TAIL waves on a tile and K, which come in the same launch and fill what the whole ones leave.  I4 4096 x 11008 M = 2048
// (1376 tiles of 64 x 256: five rounds and 96) 240 -> 231 us a call, 258 -> 230 on another device; U4 2188 x 8320 M = 571 (256 + 41) 45.3 -> 43.2;
// over 420 drawn calls 2.3 % where the rule may take it.
template <int DT, int WK, int TAIL>
__global__ void __launch_bounds__(256, 1) qgemm_wave_kernel(WaveArgs p)
{
    constexpr int WM = WK == 1 ? 2 : 1, WN = WK == 4 ? 1 : 2;
    // Workgroup id -> tile.  Ids are dealt round-robin over the 8 XCDs; each XCD takes a contiguous share of the tiles, walked
    // in stripes of four row tiles, so that the workgroups resident on it read few different operand rows.
    auto tile_at = [&](unsigned T, unsigned *mt, unsigned *nt) {
        const unsigned stripe = p.by_stripe.div(T), first_m = stripe * 4, in_stripe = T - stripe * 4 * (unsigned)p.ntiles;
        const unsigned height = (unsigned)p.mtiles - first_m < 4 ? (unsigned)p.mtiles - first_m : 4;
        *nt = height == 4 ? in_stripe >> 2 : in_stripe / height;
        *mt = first_m + (in_stripe - *nt * height);
    };
    unsigned mt, nt;
    const unsigned main_xcd = (p.main_tiles + 7) / 8, y = blockIdx.x >> 3;
    if (y < main_xcd) {
        const unsigned T = (blockIdx.x & 7) * main_xcd + y;
        if (T >= p.main_tiles) return;
        tile_at(T, &mt, &nt);
        wave_tile<DT, WK>(p, mt * WM, nt * WN, p.units_per_wave);
    } else if constexpr (TAIL > WK) {
        constexpr unsigned SM = WM, SN = TAIL == 4 ? 2 : 1;   // parts of a tile
        const unsigned parts = (p.tiles - p.main_tiles) * SM * SN, part_xcd = (parts + 7) / 8, at = (blockIdx.x & 7) * part_xcd + (y - main_xcd);
        if (y - main_xcd >= part_xcd || at >= parts) return;
        tile_at(p.main_tiles + at / (SM * SN), &mt, &nt);
        const unsigned rg = mt * WM + (SM == 2 ? at & 1 : 0), cg = nt * WN + (SN == 2 ? (at / SM) & 1 : 0);
        if ((int64_t)rg * WAVE_ROWS >= p.m || (int64_t)cg * WAVE_COLS >= p.n) return;
        wave_tile<DT, TAIL>(p, rg, cg, p.tail_units_per_wave);
    }
}

template <int DT, int WK, int TAIL = 0>
hipError_t wave_launch_one(const WaveArgs &p, hipStream_t s)
{
    constexpr int lds = WK == 1 && TAIL == 0 ? 0 : 4 * 16 * WAVE_COLS / 32 * 256;
    auto kern = qgemm_wave_kernel<DT, WK, TAIL>;
    static std::atomic<uint64_t> raised{0};
    const hipError_t e = fnn_raise_lds_limit(raised, reinterpret_cast<const void *>(kern), lds);
    if (e != hipSuccess) return e;
    const unsigned parts = TAIL > WK ? (p.tiles - p.main_tiles) * (TAIL / WK) : 0;
    hipLaunchKernelGGL(kern, dim3((p.main_tiles + 7) / 8 * 8 + (parts + 7) / 8 * 8), dim3(256), lds, s, p);
    return hipGetLastError();
}

template <int DT>
hipError_t wave_launch(int wk, int tail, const WaveArgs &p, hipStream_t s)
{
    if (wk == 1) return tail == 2 ? wave_launch_one<DT, 1, 2>(p, s) : (tail == 4 ? wave_launch_one<DT, 1, 4>(p, s) : wave_launch_one<DT, 1>(p, s));
    if (wk == 2) return tail == 4 ? wave_launch_one<DT, 2, 4>(p, s) : wave_launch_one<DT, 2>(p, s);
    return wave_launch_one<DT, 4>(p, s);
}

}  // namespace
