// Launch interface of the fragment-major MatMul kernels (qgemm_frag_impl.h; one translation unit per weight type).
#pragma once
#include <cstdint>

#include "common.h"

constexpr int64_t FRAG_OPT_WAVE = 1 << 14;   // FNN_OPT_FRAGMENT names a form of qgemm_wave_impl.h
struct fnn_hip_ctx;
bool fnn_frag_options_untouched(fnn_hip_ctx *ctx);

constexpr int FRAG_NW = 8;        // waves per workgroup, each with an eighth of the workgroup's K range (a segment)

// How K is dealt out: `splits` workgroups of kb_per_split k blocks (64 bytes of a weight row), each in FRAG_NW segments.
struct FragSplit {
    int kblocks, splits, kb_per_split;
    int seg, seg_last;           // k blocks per segment: of the last split (seg_last) and of those before it
    int piece, pieces;           // a segment in `pieces` pieces of `piece` k blocks: what shares a power of two per row
    // segment wv of split z: blocks [b0, b1), empty where b0 >= b1
    __host__ __device__ void segment(int z, int wv, int *b0, int *b1) const
    {
        const int kb0 = z * kb_per_split, kb1 = kb0 + kb_per_split < kblocks ? kb0 + kb_per_split : kblocks;
        const int per = z == splits - 1 ? seg_last : seg;
        *b0 = kb0 + wv * per;
        *b1 = *b0 + per < kb1 ? *b0 + per : kb1;
    }
    // piece i of all pieces, segment by segment
    __host__ __device__ void piece_at(int i, int *b0, int *b1) const
    {
        const int s = i / pieces;
        segment(s / FRAG_NW, s % FRAG_NW, b0, b1);
        *b0 += (i - s * pieces) * piece;
        *b1 = *b0 + piece < *b1 ? *b0 + piece : *b1;
    }
};

// A row's values of a piece of K: the power of two applied to them, and their sum (for the zero-point term).
struct FragRow { int e; float sum; };
__device__ __forceinline__ double frag_sum8(const float(&v)[8])
{
    return (double)(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
}

// The packed words as the kernels read them: the fragment-major copy [row block of 16][k block][q 0..3][row][16 bytes] (kp 0),
// or the registered rows of kp words where there is no copy (the same values, so the same results; a wave load is then 16
// pieces of 64 bytes instead of one contiguous KB).  This: 16 bytes `piece` of row r of row block rb in its first k block (past
// the last of `rows`: that row's; never stored).
__device__ __forceinline__ const uint32_t *frag_row_at(const uint32_t *w, int kp, int rows, int kblocks, int rb, int r, int piece)
{
    const int last_rb = (rows - 1) >> 4;
    if (rb > last_rb) rb = last_rb;
    if (!kp) return w + (int64_t)rb * kblocks * 256 + piece * 64 + r * 4;
    const int last = rows - 1 - rb * 16;
    return w + (int64_t)rb * 16 * kp + (uint32_t)((r < last ? r : last) * kp + piece * 4);
}
typedef uint32_t frag_u32x4 __attribute__((ext_vector_type(4), aligned(4)));   // (registered rows of any length: 4-byte aligned)

struct FragArgs {
    const uint32_t *wf;          // weight words: frag_row_at.  (Fields are dear here: 48 bytes more cost 0.25 us a launch)
    const _Float16 *af;          // activation fragments [row block of 16][step of 32 k][hi, lo][q 0..3][row][8 f16]
    const float *a;              // non-null: the f32 activations [m,k], converted in the kernel (splits == 1; af, rows unused)
    int64_t k;
    const FragRow *rows;         // [segment][piece][m_pad]
    const float *scales, *zeros, *bias;
    float *out;
    float *part;                 // non-null: [split][m][n] sums with scale and zero applied, no bias or activation
    const float *residual;       // non-null (no part): sum_out[m,n] = out[m,n] + residual[m,n] as well
    float *sum_out;
    int64_t m, n, m_pad;
    int act;
    FragSplit ks;
    FastDiv by_mtiles, by_splits;
    int mtiles, ntiles, words_kp;
    int vec4;                    // 16-byte accesses along n: n % 4 == 0 and aligned tensors
};

// mb x 16 activation rows and nb x 16 weight rows per workgroup of eight waves
hipError_t fnn_frag_launch_i8(int mb, int nb, const FragArgs &p, hipStream_t s);
hipError_t fnn_frag_launch_i4(int mb, int nb, const FragArgs &p, hipStream_t s);
hipError_t fnn_frag_launch_u8(int mb, int nb, const FragArgs &p, hipStream_t s);
hipError_t fnn_frag_launch_u4(int mb, int nb, const FragArgs &p, hipStream_t s);
hipError_t fnn_frag_launch_f8(int mb, int nb, const FragArgs &p, hipStream_t s);
hipError_t fnn_frag_launch_f8r(int mb, int nb, const FragArgs &p, hipStream_t s);
hipError_t fnn_frag_launch_f4(int mb, int nb, const FragArgs &p, hipStream_t s);
