// Chirp transforms of the inverse y-pass (band columns onto the cropped rows).
#include "bldfm_line.h"

int bldfm_lines_pass2(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int grid_cap, hipStream_t stream, int lds_attr) {
  return launch_lines<PASS_INV_COLS>(P, L, B, grid_cap, stream, lds_attr);
}
