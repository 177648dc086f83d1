// Chirp transforms of the forward rows (dispersion: surface flux rows onto the retained columns).
#include "bldfm_line.h"

int bldfm_lines_pass0(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int grid_cap, hipStream_t stream, int lds_attr) {
  return launch_lines<PASS_FWD_ROWS>(P, L, B, grid_cap, stream, lds_attr);
}
