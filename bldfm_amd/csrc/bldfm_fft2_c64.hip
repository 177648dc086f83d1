#include "bldfm_fft2.h"

template int launch_fft2<float2>(const FftSplit&, int32_t, const FftSplit&, int32_t, int32_t, const float2*, double2*, double2*,
                                 float2*, int32_t, double, int, int, int, hipStream_t);
template void fft2_lds_attr<float2>(int);
