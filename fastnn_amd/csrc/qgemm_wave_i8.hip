// Int8 MatMul with large register tiles (qgemm_wave_impl.h), weight type I8.
#include "mfma.h"
#include "qgemm_wave_impl.h"
hipError_t fnn_wave_launch_i8(int wk, const WaveArgs &p, hipStream_t s) { return wave_launch<FNN_DT_I8>(wk, p, s); }
