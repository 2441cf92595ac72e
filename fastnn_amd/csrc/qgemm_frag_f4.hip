// Fragment-major MatMul (qgemm_frag_impl.h), weight type F4.
#include "mfma.h"
#include "qgemm_frag_impl.h"
hipError_t fnn_frag_launch_f4(int mb, int nb, const FragArgs &p, hipStream_t s) { return frag_launch<FNN_DT_F4>(mb, nb, p, s); }
