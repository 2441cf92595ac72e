// Fragment-major MatMul on the int8 matrix cores (qgemm_frag_int_impl.h), weight type I4.
#include "mfma.h"
#include "qgemm_frag_int_impl.h"
hipError_t fnn_frag_int_launch_i4(int mb, int nb, const FragIntArgs &p, hipStream_t s) { return frag_int_launch<FNN_DT_I4>(mb, nb, p, s); }
