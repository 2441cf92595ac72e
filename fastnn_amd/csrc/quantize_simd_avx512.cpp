#define FNN_QUANT_TABLE fnn_quant_avx512
#include "quantize_simd_impl.h"
