#include "bldfm_fft2.h"

// complex64: compiled in a file of its own, beside this one
extern template int launch_fft2<float2>(const FftSplit&, int32_t, const FftSplit&, int32_t, int32_t, const float2*, double2*,
                                        double2*, float2*, int32_t, double, int, int, int, hipStream_t);
extern template void fft2_lds_attr<float2>(int);

int bldfm_launch_fft2(const FftSplit& A0, int32_t n0, const FftSplit& A1, int32_t n1, int32_t batch, bool single,
                      const void* in, double2* mid, double2* scr, void* out, int32_t sign, double scale,
                      int threads, int lds_bytes, int grid_cap, hipStream_t stream) {
  if (single)
    return launch_fft2(A0, n0, A1, n1, batch, (const float2*)in, mid, scr, (float2*)out, sign, scale, threads, lds_bytes,
                       grid_cap, stream);
  return launch_fft2(A0, n0, A1, n1, batch, (const double2*)in, mid, scr, (double2*)out, sign, scale, threads, lds_bytes,
                     grid_cap, stream);
}

void bldfm_fft2_lds_attr(int bytes) {
  fft2_lds_attr<double2>(bytes);
  fft2_lds_attr<float2>(bytes);
}
