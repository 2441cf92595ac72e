// Host side of the one-launch streaming MatMul for up to 32 activation rows (kernels: qgemm_stream_impl.h, one
// translation unit per weight type): which calls it takes, the shape of the launch, the split-K workspace.
#include "mfma.h"
#include "qgemm_stream.h"
#include "range_io.h"

namespace {

// RT, KR, splits and rounds from FNN_OPT_STREAM_SHAPE or by rule (MB follows from M).  The phases of a round (requests,
// conversion, matrix cores) follow one another inside a workgroup, so a workgroup does one round where it can: one row
// tile per wave, K / KR splits, and KR = 512 while that still gives the 256 CUs a workgroup each.
bool plan_stream(bool cb, int max_tiles, int max_mb, int64_t m, int64_t n, int64_t k, int64_t forced, StreamPlan *out)
{
    const int mb = (int)((m + 15) / 16);
    if (mb < 1 || mb > max_mb) return false;
    int rt = 1, kr = 512;
    const int64_t nt1 = (n + FNN_STREAM_NW * 16 - 1) / (FNN_STREAM_NW * 16);
    if (nt1 * ((k + 511) / 512) < 224) kr = 256;
    int64_t splits = 0;
    const bool low_up = forced & 128;
    if (forced > 0) {
        rt = (int)((forced >> 4) & 7);
        kr = (int)(forced & 15) * 256;
        splits = forced >> 8;
        if (rt < 1 || rt > 2 || (kr != 256 && kr != 512)) return false;
        if (low_up && (!cb || rt != 1 || kr != StreamPlan::wide_kr(mb))) return false;
    }
    if (mb * rt > max_tiles) return false;   // accumulator tiles that fit the registers
    const int64_t kr_total = (k + kr - 1) / kr;   // rounds over all of K
    if (splits == 0) splits = kr_total > 64 ? 64 : kr_total;
    if (splits > kr_total || splits > 64) return false;
    const int64_t rounds = (kr_total + splits - 1) / splits;
    if ((splits - 1) * rounds >= kr_total) return false;   // an empty split
    const int64_t ntiles = (n + FNN_STREAM_NW * rt * 16 - 1) / (FNN_STREAM_NW * rt * 16);
    // By rule the kernel takes a call only where it measured faster than preparation + tiles + reduction as three
    // launches: no more workgroups than the chip holds at once (a second wave of
    // workgroups repeats every phase).  4096 x 4096 at M = 32: 14.4 against 17.9 us; 2048 -> 8192 FP8: 13.3 against 17.4;
    // 4096 x 11008 (688 workgroups): 25.0 against 23.5; M = 64 on 4096 x 4096: 21.3 against 20.0.
    if (forced == 0 && ntiles * splits > 320) {
        // Wide outputs: two row tiles per wave (256 weight rows per workgroup) and as few rounds per workgroup as keep the
        // launch within one round of workgroups (one workgroup of this form per CU: at most 256).  4096 x 11008 (43 column tiles): 4 splits x 2 rounds of 512, 172 workgroups,
        // M = 17 19.2 us against 23.0 on the tiled path, M = 32 21.3 against 23.9 (8 splits x 1 round, 344 workgroups: 25.5).
        int64_t r2 = 0;
        if (mb * 2 <= max_tiles) {
            const int64_t ntiles2 = (n + FNN_STREAM_NW * 2 * 16 - 1) / (FNN_STREAM_NW * 2 * 16), total512 = (k + 511) / 512;
            for (int64_t r = 1; r <= 4 && !r2; r++) {
                const int64_t s = (total512 + r - 1) / r;
                if (s > 64 || (s - 1) * r >= total512) continue;   // (no empty split)
                if (ntiles2 * s > 256) continue;   // (one workgroup of this form per CU: 270 workgroups on 5120 x 13824 ran 33.7 us against 28.0 on the tiled path)
                if (ntiles2 * s < 128) break;                      // (too few workgroups: the tiled path is ahead)
                *out = StreamPlan{mb, 2, 512, (int)s, (int)r, (int)ntiles2};
                r2 = r;
            }
        }
        // Codebook weights: one row tile per wave, two workgroups per CU (their LDS: rounds of 512 up to 32 rows, of 256 beyond) and the
        // fewest rounds that leaves.  The tiles decode every nibble again for each 32 rows; two row tiles per wave cannot hide the look-ups.
        // 4096 x 11008 M = 64 62.3 us on the tiles, 43.1 so, 2048 x 11008 39.7 and 26.6, 2048 x 16384 37.4 and 29.2; M = 32, two row tiles per wave
        // against this, 28.0 and 27.3, 19.4 and 17.6, 21.0 and 19.3.
        if (cb) {
            const int64_t wide_kr = StreamPlan::wide_kr(mb), total = (k + wide_kr - 1) / wide_kr;
            for (int64_t r = 1; r <= 16; r++) {
                const int64_t s = (total + r - 1) / r;
                if (s > 64 || (s - 1) * r >= total || ntiles * s > 512) continue;   // (no empty split)
                if (ntiles * s < 256) break;   // (too few workgroups)
                // A long K over few columns, from 33 rows on: workgroups of one round leave the last one of a column tile more parts to add up than they save.  90
                // drawn calls of 17 to 60 splits take 1.18 times the tiles' time so, 1.57 at most (54 x 15104 x 976 34.6 us there, 54.5 so; 60 x 7296 x 1664 29.4
                // and 34.6; 56 x 4992 x 2496 25.7 and 29.3), five less (38 x 5120 x 2432 29.9 and 26.1).  17 and more of two rounds are 4 to 10 % ahead.
                if (mb > 2 && r == 1 && s > 16) continue;
                // Two row tiles per wave in half as many rounds, each of twice the values, are ahead where those are two and more: 43 x 8448 x 10368 6 rounds against 3,
                // 53.5 us and 50.8, 39 x 7680 x 15105 8 against 4, 65.0 and 61.0; 4 against 2 1 % behind with weights from cache, 4 to 7 % ahead from memory
                // (43 x 4352 x 12869 44.4 and 41.6).  They are 3 to 10 % behind with 5 against 3 or 7 against 4, 13 % with 2 against 1.
                if (mb > 2 && r >= 4 && r2 && r >= 2 * r2) break;
                // Without two row tiles as a plan these calls are the tiles' otherwise, which hold the activations' low halves scaled by 2^11.  So does this form then: unscaled
                // they are denormals from 2^-18 of a round's largest value on, and beside values of 2^24 on weights of zero a normal row comes out 1.7e-5 of its norm
                // off, not 1.6e-7 (64 x 3072 x 12288).  Four fused multiply-adds a product of 32 x 16 x 16: 64 x 4096 x 11008 40.8 -> 44.5 us, 64 x 2048 x 11008 25.6 -> 27.4.
                *out = StreamPlan{mb, 1, (int)wide_kr, (int)s, (int)r, (int)ntiles, r2 == 0};
                return true;
            }
        }
        return r2 != 0;
    }
    *out = StreamPlan{mb, rt, kr, (int)splits, (int)rounds, (int)ntiles, low_up};
    return true;
}

bool stream_plan_for(fnn_hip_ctx *ctx, const fnn_hip_weight *w, const QMatmulArgs &q, int flags, StreamPlan *pl)
{
    int64_t lo = fnn_ctx_option(ctx, FNN_OPT_STREAM_MIN_M), hi = fnn_ctx_option(ctx, FNN_OPT_STREAM_MAX_M);
    const int dt = w->dtype;
    const bool cb = dt == FNN_DT_I4CB;
    // Per-channel types: up to two blocks of 16 activation rows (three and four measured slower than the tiled path).
    // Codebook weights: the tiled path decodes them on the vector ALU inside its loop and is far from the memory bound,
    // so the range is wider, 5 <= M <= 64 with the options at their defaults.
    if (cb) { lo = lo < 5 ? lo : 5; hi = hi >= 32 ? 64 : hi; }
    // A long K over few output columns (the down projection of an MLP): the one-launch kernels for M <= 16 give every
    // workgroup whole rows -- few workgroups, each converting M x K activations -- while this kernel splits K over the
    // chip and its time hardly depends on M.  From M = 9 where K >= 4 N, or K >= 2 N from K = 8192 on (11008 -> 4096 I4:
    // 16.7-17.2 against 22.1-23.6 us; 4096 -> 1024 I8: 8.7 against 9.5; but 4096 -> 2048: 10.6 against 9.7, left out);
    // from M = 5 only where N <= 2048 and K >= 4 N with K >= 8192 (f16 types: 8192 -> 2048 FP8 12.0-12.2 against
    // 13.0-13.3 us) or K >= 16384 (types of the int8 GEMV, which is the better kernel below that: 16384 -> 1024 I4 13.7
    // against 20.2-20.8 us, 8192 -> 1024 I4 13.2 against 11.4).  U8, which has that GEMV too, keeps the f16 types' line: 5 to 8 rows of 8192 to 16384 values over 256
    // to 2048 columns 9.6 to 19.0 us here and 10.8 to 20.3 there, 8192 and 10240 -> 1024 and 10240 -> 2048 (12.5, 14.3, 14.9 and 11.0, 12.6, 13.0) apart.  Not
    // when the option was raised above its default.
    const bool int_type = dt == FNN_DT_I8 || dt == FNN_DT_I4 || dt == FNN_DT_U4;
    if (!cb && lo <= 17) {
        // ... and from M = 9 where K leaves the eight waves of the kernel for 9 <= M <= 16 a ragged last round (its waves
        // take slices of 512 k-values in turn: 9, 10 or 12 slices are two rounds with half of the waves idle in the
        // second).  5120 x 13824 I4: 18.0-19.0 against 32.7-34.0 us; 5120 x 5120: 13.4-13.7 against 17.0; 6144 x 6144: 14.4-14.9
        // against 17.1-17.5; 3072 (six slices, one round) stays: 9.8 against 10.8-11.2.
        const int64_t nsl = (q.k + 511) / 512, rnds = (nsl + 7) / 8;
        if (rnds >= 2 && nsl * 4 <= rnds * 8 * 3) lo = lo < 9 ? lo : 9;
        if (q.k >= 4 * q.n || (q.k >= 2 * q.n && q.k >= 8192)) lo = lo < 9 ? lo : 9;
        if (q.n <= 2048 && q.k >= 4 * q.n && q.k >= (int_type ? 16384 : 8192)) lo = lo < 5 ? lo : 5;
    }
    if (q.m < lo || q.m > hi || q.m > (cb ? 64 : 32) || q.n < 1) return false;
    if (flags & FNN_FLAG_ACT_F16_SINGLE) return false;
    if (cb && fnn_ctx_option(ctx, FNN_OPT_CODEBOOK_EXPANDED) != 0) return false;   // (the option names a form of the tiled path)
    if (cb && (q.as_written || q.qblock != 32 || q.k % 128 != 0 || q.bpr != q.k / 32 || (reinterpret_cast<uintptr_t>(q.scales) & 15) ||
               q.bpr * 4 * 256 >= (int64_t)1 << 31)) return false;
    if (dt < FNN_DT_I8 || (dt > FNN_DT_F4 && !cb)) return false;
    if (int_type && fnn_ctx_option(ctx, FNN_OPT_GEMM_INT8) == 0) return false;
    if (q.kp % 4 != 0 || q.k % 8 != 0 || q.k < 8) return false;
    // the f16 types multiply whatever bytes a lane load holds: every load must lie wholly inside or wholly past K
    if (!int_type && q.k % (dt == FNN_DT_F4 ? 128 : 64) != 0) return false;
    if ((reinterpret_cast<uintptr_t>(q.a) & 15) || (reinterpret_cast<uintptr_t>(q.words) & 15)) return false;
    // 32-bit buffer offsets: a column tile of 256 rows, the activation block
    if (q.kp * 4 * 256 >= (int64_t)1 << 31 || q.m * q.k * 4 >= (int64_t)0xFFFFFF00 || q.k >= (int64_t)1 << 28) return false;
    const int64_t forced = fnn_ctx_option(ctx, FNN_OPT_STREAM_SHAPE);
    return plan_stream(cb, int_type ? 4 : (cb ? 6 : 8), cb ? 4 : 2, q.m, q.n, q.k, forced, pl) && pl->ntiles <= FNN_STREAM_COUNTERS;
}

}  // namespace

// The time: least squares over 2620 drawn calls of 17 to 32 rows, weights from memory and from cache (5 % mean error): the conversion
// of a workgroup's activations, weight bytes, the tail, in which the last workgroup of a column tile reads what the others left,
// a second workgroup on some CU, workgroups at all, the partials' bytes.
bool fnn_stream_takes(fnn_hip_ctx *ctx, const fnn_hip_weight *w, const QMatmulArgs &q, int flags, float *us)
{
    StreamPlan pl;
    if (!stream_plan_for(ctx, w, q, flags, &pl)) return false;
    static const float kFit[2][8] = {{4.37f, 1.292f, 0.0731f, 0.155f, 0.0581f, 2.299f, 1.709f, 1.226f},    // 8-bit
                                     {4.70f, 1.110f, 0.0025f, 0.140f, 0.0710f, 1.342f, 2.325f, 1.587f}};   // 4-bit
    const bool four = w->dtype == FNN_DT_I4 || w->dtype == FNN_DT_U4 || w->dtype == FNN_DT_F4;
    const float *c = kFit[four], sp = (float)pl.splits, wgs = (float)(pl.splits * pl.ntiles), range = (float)(pl.rounds * pl.kr * pl.rt) / 512.f;
    *us = c[0] + c[1] * range * (float)pl.mb + c[2] * (float)q.n * (float)q.k * (four ? 0.5f : 1.f) / 1e6f + sp * (c[3] + c[4] * (float)(pl.mb * pl.rt)) +
          c[5] * (float)((pl.splits * pl.ntiles + 255) / 256 - 1) * range + c[6] * wgs / 256.f + c[7] * (float)q.m * (float)q.n * sp / 1e6f;
    return true;
}

int fnn_stream_qmatmul(fnn_hip_ctx *ctx, hipStream_t s, const fnn_hip_weight *w, const QMatmulArgs &q, int flags, bool *handled)
{
    *handled = false;
    StreamPlan pl;
    if (!stream_plan_for(ctx, w, q, flags, &pl)) return FNN_OK;
    const int dt = w->dtype;
    const bool cb = dt == FNN_DT_I4CB;
    StreamArgs p;
    p.words = q.words; p.scales = q.scales; p.zeros = q.zeros; p.a = q.a; p.bias = q.bias; p.out = q.out;
    p.codebook = cb ? q.codebook : nullptr; p.bpr = cb ? q.bpr : 0;
    p.residual = nullptr; p.sum_out = nullptr;
    p.part = nullptr; p.count = fnn_ctx_stream_counters(ctx);
    p.m = q.m; p.n = q.n; p.k = q.k; p.kp = q.kp;
    p.act = q.act; p.splits = pl.splits; p.rounds = pl.rounds; p.ntiles = pl.ntiles;
    if (int rc = fnn_fragment_blocks(ctx, s, w, q, &p.words_fr, &p.kb64)) return rc;
    if (pl.splits > 1) {
        const size_t wgf = (size_t)pl.mb * pl.rt * 4 * FNN_STREAM_NW * 64 + 16 * pl.mb;
        void *ws = nullptr;
        int rc = fnn_ctx_ensure_tmp(ctx, 1, (size_t)pl.splits * pl.ntiles * wgf * 4, &ws);
        if (rc) return rc;
        p.part = (float *)ws;
    }
    fnn_take_residual(ctx, q.out, q.m * q.n, &p.residual, &p.sum_out);
    hipError_t e;
    switch (dt) {
    case FNN_DT_I8: e = fnn_stream_launch_i8(pl, p, s); break;
    case FNN_DT_I4: e = fnn_stream_launch_i4(pl, p, s); break;
    case FNN_DT_U4: e = fnn_stream_launch_u4(pl, p, s); break;
    case FNN_DT_U8: e = fnn_stream_launch_u8(pl, p, s); break;
    case FNN_DT_F8: e = fnn_stream_launch_f8(pl, p, s); break;
    case FNN_DT_F8R: e = fnn_stream_launch_f8r(pl, p, s); break;
    case FNN_DT_I4CB: e = fnn_stream_launch_i4cb(pl, p, s); break;
    default: e = fnn_stream_launch_f4(pl, p, s); break;
    }
    if (e != hipSuccess) return fnn_ctx_fail(ctx, FNN_ERR_DISPATCH, hipGetErrorString(e));
    *handled = true;
    return FNN_OK;
}
