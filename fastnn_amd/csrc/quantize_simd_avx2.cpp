#define FNN_QUANT_TABLE fnn_quant_avx2
#include "quantize_simd_impl.h"
