// Four-step transforms of the passes of split lengths.
#include "bldfm_passes.h"

// One step of the four-step transforms of the split lines of pass `pass`
// (tile local = line * (n2 or n1) + sub-transform index).
// The pass is a template parameter, as in k_pass: with all four behind a
// run-time switch in one body the compiler took minutes per kernel.
template <int MAXE, int MAXT, bool STEPB, int pass>
__global__ __launch_bounds__(MAXT) void k_long(PlanDev P, ExecBufs B) {
  const int T = blockDim.x, tid = threadIdx.x;
  const int k = 2 * pass + (STEPB ? 1 : 0);
  const TileRec* recs = P.t_long[k];
  const int64_t tot = P.tot_long[k];
  for (int64_t b = blockIdx.x; b < tot; b += gridDim.x) {
    const TileRec tr = tile_rec(recs, b);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    const bool x_axis = pass == PASS_FWD_ROWS || pass == PASS_INV_ROWS;
    const cplan_t& FL = *(const cplan_t*)(P.plans + (x_axis ? D.plan_x : D.plan_y));
    const int n = FL.n, n1 = FL.n1, n2 = FL.n2;
    const int64_t per = STEPB ? n1 : n2;
    const int64_t line = (int64_t)tr.local / per;
    const int sub = (int)((int64_t)tr.local % per);
    double2* scr = B.ws + D.off_long + line * n;
    const bool reuse = b != blockIdx.x;
    run_pass(pass, P, B, D, tr.inst, line, [&](const cplan_t&, auto in, auto out, bool inv) {
      if constexpr (!STEPB) {
        const cplan_t& F1 = *(const cplan_t*)(P.plans + FL.plan1);
        fft_dir<MAXE>(inv, F1, P.tw, tid, T, SubIn<decltype(in)>{in, n2, sub},
                      TwiddleOut{scr + (int64_t)sub * n1, P.tw + FL.tw_off, sub, inv}, reuse);
      } else {
        const cplan_t& F2 = *(const cplan_t*)(P.plans + FL.plan2);
        fft_dir<MAXE>(inv, F2, P.tw, tid, T, ScrIn{scr + sub, n1}, SubOut<decltype(out)>{out, n1, sub}, reuse);
      }
    });
  }
}

template <int PASS>
static int launch_long(const PlanDev& P, const ExecBufs& B, int grid_cap, hipStream_t stream) {
  const unsigned ft = (unsigned)P.fft_threads;
  const size_t lds = (size_t)P.fft_lds_bytes;
  for (int st = 0; st < 2; ++st) {
    const int64_t tl = P.tot_long[2 * PASS + st];
    if (tl <= 0) continue;
    const unsigned g = grid_for(tl, grid_cap);
    if (P.fft_small) {
      if (st) k_long<FFT_SMALL_E, 256, true, PASS><<<g, ft, lds, stream>>>(P, B);
      else k_long<FFT_SMALL_E, 256, false, PASS><<<g, ft, lds, stream>>>(P, B);
    } else {
      if (st) k_long<BLDFM_FFT_MAXE, 1024, true, PASS><<<g, ft, lds, stream>>>(P, B);
      else k_long<BLDFM_FFT_MAXE, 1024, false, PASS><<<g, ft, lds, stream>>>(P, B);
    }
    LAUNCH_CHECK();
  }
  return 0;
}

int bldfm_launch_long(const PlanDev& P, const ExecBufs& B, int pass, int grid_cap, hipStream_t stream) {
  switch (pass) {
    case PASS_FWD_ROWS: return launch_long<PASS_FWD_ROWS>(P, B, grid_cap, stream);
    case PASS_FWD_COLS: return launch_long<PASS_FWD_COLS>(P, B, grid_cap, stream);
    case PASS_INV_COLS: return launch_long<PASS_INV_COLS>(P, B, grid_cap, stream);
    default: return launch_long<PASS_INV_ROWS>(P, B, grid_cap, stream);
  }
}

template <int PASS>
static void set_long_attr(int bytes) {
  const void* fns[] = {(const void*)k_long<FFT_SMALL_E, 256, false, PASS>, (const void*)k_long<FFT_SMALL_E, 256, true, PASS>,
                       (const void*)k_long<BLDFM_FFT_MAXE, 1024, false, PASS>,
                       (const void*)k_long<BLDFM_FFT_MAXE, 1024, true, PASS>};
  for (const void* f : fns) (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

void bldfm_long_lds_attr(int bytes) {
  set_long_attr<PASS_FWD_ROWS>(bytes);
  set_long_attr<PASS_FWD_COLS>(bytes);
  set_long_attr<PASS_INV_COLS>(bytes);
  set_long_attr<PASS_INV_ROWS>(bytes);
}
