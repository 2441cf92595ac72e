// Launch interface of the int8 MatMul with large register tiles (qgemm_wave_impl.h; one translation unit per weight type).
#pragma once
#include "qgemm_frag.h"

// steps of 32 k-values in flight per wave: 42 KB (8-bit weights, 7 KB a step) and 40 KB (4-bit, 5 KB); four and six cost 5 to
// 10 %
constexpr int WAVE_RING(bool w8) { return w8 ? 6 : 8; }
constexpr int WAVE_ROWS = 32, WAVE_COLS = 128;   // activation rows (three planes each) and columns of a wave's tile

struct WaveArgs {
    const uint32_t *wf;          // weight words (frag_row_at), kblocks blocks of 64 bytes per row
    const int8_t *af;            // [block of 32 operand rows][step][h 0..1][row][16 bytes]
    const int *rexp;             // [m_pad] power of two applied to the row, INT_MIN: a non-finite row
    const float *xsum;           // [m_pad] sum_k A[m,k]
    const float *scales, *zeros, *bias;
    float *out;
    const float *residual;       // sum_out = out + residual as well
    float *sum_out;
    int64_t m, n;
    int act, kblocks, mtiles, ntiles, words_kp;
    int nsteps;                  // steps per operand row, whole units
    int units, units_per_wave;   // a unit is a ring of steps
    unsigned tiles, main_tiles;  // the tiles behind main_tiles are cut into the smaller ones of `tail` waves
    int tail_units_per_wave;
    FastDiv by_stripe;           // tiles of four row tiles
};

// wk: waves of a workgroup that share an output tile (1, 2, 4); tail: of the tiles behind main_tiles, 0 for none (wk 1: 2, 4, wk 2: 4)
hipError_t fnn_wave_launch_i8(int wk, int tail, const WaveArgs &p, hipStream_t s);
hipError_t fnn_wave_launch_i4(int wk, int tail, const WaveArgs &p, hipStream_t s);
hipError_t fnn_wave_launch_u4(int wk, int tail, const WaveArgs &p, hipStream_t s);

// The form for these sizes by rule, wk + 8 tail, 0 for none; *us: the time expected of it (microseconds).
int fnn_wave_choice(int dtype, int64_t m, int64_t n, int64_t k, float *us);
