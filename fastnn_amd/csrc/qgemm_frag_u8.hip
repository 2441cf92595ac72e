// Fragment-major MatMul (qgemm_frag_impl.h), weight type U8.
#include "mfma.h"
#include "qgemm_frag_impl.h"
hipError_t fnn_frag_launch_u8(int mb, int nb, const FragArgs &p, hipStream_t s) { return frag_launch<FNN_DT_U8>(mb, nb, p, s); }
