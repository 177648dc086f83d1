// Chirp transforms of the inverse x-pass (cropped rows onto conc and flx).
#include "bldfm_line.h"

int bldfm_lines_pass3(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int grid_cap, hipStream_t stream, int lds_attr) {
  return launch_lines<PASS_INV_ROWS>(P, L, B, grid_cap, stream, lds_attr);
}
