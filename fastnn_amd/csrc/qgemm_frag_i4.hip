// Fragment-major MatMul (qgemm_frag_impl.h), weight type I4.
#include "mfma.h"
#include "qgemm_frag_impl.h"
hipError_t fnn_frag_launch_i4(int mb, int nb, const FragArgs &p, hipStream_t s) { return frag_launch<FNN_DT_I4>(mb, nb, p, s); }
