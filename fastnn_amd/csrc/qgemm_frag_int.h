// Launch interface of the fragment-major integer MatMul kernels (qgemm_frag_int_impl.h; one translation unit per weight type).
#pragma once
#include "qgemm_frag.h"

// Operands of v_mfma_i32_16x16x64_i8: a step is 64 k-values, a group two steps (128 k-values).
struct FragIntArgs {
    const uint32_t *wf;          // weight fragments as in FragArgs, kblocks blocks of 64 bytes per row of fragments
    const int8_t *af;            // activation fragments [row block of 16][step][plane][q 0..3][row][16 bytes]
    const uint8_t *payload;      // I8 activations: scale, zero, codes [m][k]; with af null the kernel reads the codes itself
    int32_t *qsum;               // I8 activations with part: [split][m_pad] sums of the rows' codes
    const int32_t *wsum;         // I8 activations: [n] sum of the weight row's integers
    const int *rexp;             // digit planes: [m_pad] power of two applied to the row, INT_MIN: a non-finite row
    const float *xsum;           // digit planes: [m_pad] sum_k A[m,k]
    const float *scales, *zeros, *bias;
    float *out;
    int32_t *acc_out;            // I8 activations: the exact sums as well, or null
    int32_t *part;               // non-null: [split][m][n], exact sums (I8 activations) or scaled f32 sums (digit planes)
    const float *residual;       // digit planes, no part: sum_out = out + residual as well
    float *sum_out;
    int64_t m, n, k, m_pad;
    int act;
    FragSplit ks;                // in groups
    int kblocks;
    FastDiv by_mtiles, by_splits;
    int mtiles, ntiles, rblocks;
    int vec4;
};

hipError_t fnn_frag_int_launch_i8(int mb, int nb, bool digits, const FragIntArgs &p, hipStream_t s);
hipError_t fnn_frag_int_launch_i4(int mb, int nb, bool digits, const FragIntArgs &p, hipStream_t s);
hipError_t fnn_frag_int_launch_u4(int mb, int nb, bool digits, const FragIntArgs &p, hipStream_t s);
