#define FNN_QUANT_TABLE fnn_quant_base
#include "quantize_simd_impl.h"
