// Int8 MatMul with large register tiles (qgemm_wave_impl.h), weight type I4.
#include "mfma.h"
#include "qgemm_wave_impl.h"
hipError_t fnn_wave_launch_i4(int wk, const WaveArgs &p, hipStream_t s) { return wave_launch<FNN_DT_I4>(wk, p, s); }
