// Lag S/N kernels (lags.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace gxc {

// Series short enough for launch_lag_series, which reads vis in place.  snr and
// peak may be pinned host memory.
bool lag_in_lds(int n);
hipError_t launch_lag_series(const float2 *vis, int n, int nseries, float *snr, int *peak, hipStream_t s);

// a holds nseries series of n (a power of two, >= 2) visibilities and is
// overwritten; b is scratch of the same size.  snr[nseries], peak[nseries]
// are device arrays.
hipError_t launch_lag_snr(float2 *a, float2 *b, int n, int nseries, float *snr, int *peak, hipStream_t s);

}  // namespace gxc
