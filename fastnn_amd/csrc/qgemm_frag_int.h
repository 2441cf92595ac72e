// Launch interface of the fragment-major integer MatMul kernels (qgemm_frag_int_impl.h; one translation unit per weight type).
#pragma once
#include "qgemm_frag.h"

// Operands of v_mfma_i32_16x16x64_i8: a step is 64 k-values, a group two steps (128 k-values).
struct FragIntArgs {
    const uint32_t *wf;          // weight fragments as in FragArgs, kblocks blocks of 64 bytes per row of fragments
    const int8_t *af;            // activation fragments [row block of 16][step][q 0..3][row][16 bytes]
    const uint8_t *payload;      // scale, zero, codes [m][k]; with af null the kernel reads the codes itself
    int32_t *qsum;               // with part: [split][m_pad] sums of the rows' codes
    const int32_t *wsum;         // [n] sum of the weight row's integers
    const float *scales, *zeros, *bias;
    float *out;
    int32_t *acc_out;            // the exact sums as well, or null
    int32_t *part;               // non-null: [split][m][n], exact sums
    int64_t m, n, k, m_pad;
    int act;
    FragSplit ks;                // in groups
    int kblocks;
    FastDiv by_mtiles, by_splits;
    int mtiles, ntiles, rblocks;
    int vec4;
};

hipError_t fnn_frag_int_launch_i8(int mb, int nb, const FragIntArgs &p, hipStream_t s);
hipError_t fnn_frag_int_launch_i4(int mb, int nb, const FragIntArgs &p, hipStream_t s);
