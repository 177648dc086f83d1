// Chirp transforms of the forward columns (dispersion: onto the retained modes).
#include "bldfm_line.h"

int bldfm_lines_pass1(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int grid_cap, hipStream_t stream, int lds_attr) {
  return launch_lines<PASS_FWD_COLS>(P, L, B, grid_cap, stream, lds_attr);
}
