// Mixed-radix transforms of the passes, one workgroup per line.
#include "bldfm_passes.h"

// Single-workgroup transforms of one pass, one line per tile (XCD-swizzled
// so that each XCD works on a contiguous range of lines).
template <int MAXE, int MAXT, int PASS>
__global__ __launch_bounds__(MAXT) void k_pass(PlanDev P, ExecBufs B) {
  const int T = blockDim.x, tid = threadIdx.x;
  const TileRec* recs = PASS == PASS_FWD_ROWS   ? P.t_fwd_rows
                        : PASS == PASS_FWD_COLS ? P.t_fwd_cols
                        : PASS == PASS_INV_COLS ? P.t_inv_cols
                                                : P.t_inv_rows;
  const int64_t tot = PASS == PASS_FWD_ROWS   ? P.tot_fwd_rows
                      : PASS == PASS_FWD_COLS ? P.tot_fwd_cols
                      : PASS == PASS_INV_COLS ? P.tot_inv_cols
                                              : P.tot_inv_rows;
  for (int64_t b = blockIdx.x; b < tot; b += gridDim.x) {
    const int64_t t = gridDim.x >= tot ? xcd_swizzle(b, tot) : b;
    const TileRec tr = tile_rec(recs, t);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    run_pass(PASS, P, B, D, tr.inst, tr.local, [&](const cplan_t& F, auto in, auto out, bool inv) {
      fft_dir<MAXE>(inv, F, P.tw, tid, T, in, out, b != blockIdx.x);
    });
  }
}

int bldfm_launch_pass(const PlanDev& P, const ExecBufs& B, int pass, int64_t tiles, int grid_cap, hipStream_t stream) {
  const unsigned ft = (unsigned)P.fft_threads, g = grid_for(tiles, grid_cap);
  const size_t lds = (size_t)P.fft_lds_bytes;
#define PASS_LAUNCH(PASS)                                                             \
  case PASS:                                                                          \
    if (P.fft_small) k_pass<FFT_SMALL_E, 256, PASS><<<g, ft, lds, stream>>>(P, B);    \
    else k_pass<BLDFM_FFT_MAXE, 1024, PASS><<<g, ft, lds, stream>>>(P, B);            \
    break;
  switch (pass) {
    PASS_LAUNCH(PASS_FWD_ROWS)
    PASS_LAUNCH(PASS_FWD_COLS)
    PASS_LAUNCH(PASS_INV_COLS)
    PASS_LAUNCH(PASS_INV_ROWS)
  }
#undef PASS_LAUNCH
  LAUNCH_CHECK();
  return 0;
}

void bldfm_pass_lds_attr(int bytes) {
  const void* fns[] = {
      (const void*)k_pass<FFT_SMALL_E, 256, PASS_FWD_ROWS>, (const void*)k_pass<FFT_SMALL_E, 256, PASS_FWD_COLS>,
      (const void*)k_pass<FFT_SMALL_E, 256, PASS_INV_COLS>, (const void*)k_pass<FFT_SMALL_E, 256, PASS_INV_ROWS>,
      (const void*)k_pass<BLDFM_FFT_MAXE, 1024, PASS_FWD_ROWS>, (const void*)k_pass<BLDFM_FFT_MAXE, 1024, PASS_FWD_COLS>,
      (const void*)k_pass<BLDFM_FFT_MAXE, 1024, PASS_INV_COLS>, (const void*)k_pass<BLDFM_FFT_MAXE, 1024, PASS_INV_ROWS>};
  for (const void* f : fns) (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}
