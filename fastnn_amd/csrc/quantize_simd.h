// The per-channel weight packers over panels of 32 channels, one SIMD lane per channel: compiled once per instruction
// set (quantize_simd_*.cpp), chosen at run time.
#pragma once
#include <cstdint>

// values: lane l of step k at src[k * ld + l], l < 32.  words: row l at words + l * kp; rows < 32 of them are written.
// scales / zeros: 32 entries, of which `rows` are written.
typedef void (*fnn_quant_panel_fn)(int dtype, const float *src, int64_t ld, int64_t inner, int rows, uint32_t *words, int64_t kp,
                                   float *scales, float *zeros);
// index[i] = the first of the 16 table entries nearest to v[i] (reference order: strictly nearer wins)
typedef void (*fnn_nearest16_fn)(const float *v, int64_t n, const float *table, uint8_t *index);
// dst[k * 32 + l] = src[l * inner + k] for l < rows (0 for the lanes past them)
typedef void (*fnn_panel_from_rows_fn)(const float *src, int64_t inner, int rows, float *dst);
// nearest16, and the values themselves grouped by entry in their order: entry e's are grouped[start[e] .. start[e + 1])
typedef void (*fnn_group16_fn)(const float *v, int64_t n, const float *table, uint8_t *index, float *grouped, int32_t *start);

struct FnnQuantKernels {
    fnn_quant_panel_fn quant_panel;
    fnn_nearest16_fn nearest16;
    fnn_panel_from_rows_fn panel_from_rows;
    fnn_group16_fn group16;
};
extern const FnnQuantKernels fnn_quant_avx512, fnn_quant_avx2, fnn_quant_base;
