// Int8 MatMul with large register tiles (qgemm_wave_impl.h), weight type U4.
#include "mfma.h"
#include "qgemm_wave_impl.h"
hipError_t fnn_wave_launch_u4(int wk, const WaveArgs &p, hipStream_t s) { return wave_launch<FNN_DT_U4>(wk, p, s); }
