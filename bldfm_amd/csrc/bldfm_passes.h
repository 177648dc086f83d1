// Mixed-radix transform passes of the solver: sources, sinks and the four
// passes as factories of (plan, source, sink, direction) for one line.
#pragma once
#include "bldfm_internal.h"
#include "bldfm_fft.h"
#include "bldfm_march.h"

#define FFT_SMALL_E 8     // values per thread per stage, 256-thread FFT kernels (n <= 2048)

// ---------------------------------------------------------------- FFT passes
extern __shared__ double2 smem[];

// Sources (first stage) and sinks (last stage) of the transforms.  A band of
// nb compact values (truncated order: f >= 0 first, then f < 0) occupies
// padded indices [0, lo) and [n - (nb - lo), n) with lo = (nb + 1)/2; the
// gap between the two halves is zero.
struct Band {
  int lo, hi_start, nb;
  __device__ __forceinline__ Band(int nb_, int n) : lo((nb_ + 1) / 2), hi_start(n - (nb_ - (nb_ + 1) / 2)), nb(nb_) {}
  // compact index of padded index i, or -1 in the gap
  __device__ __forceinline__ int compact(int i) const { return i < lo ? i : (i >= hi_start ? i - hi_start + lo : -1); }
};

// Compact band at element stride `stride` in global memory.
struct BandIn {
  const double2* __restrict__ src;
  int64_t stride;
  Band band;
  __device__ __forceinline__ double2 operator()(int i) const {
    const int c = band.compact(i);
    return c < 0 ? cmk(0.0, 0.0) : src[(int64_t)c * stride];
  }
};

// Band of the spectrum, scaled, to a compact array.
struct BandOut {
  double2* __restrict__ dst;
  double fct;
  Band band;
  __device__ __forceinline__ void operator()(int o, double2 v) const {
    const int c = band.compact(o);
    if (c >= 0) dst[c] = cscale(fct, v);
  }
};

// cnt values (element stride `stride`) placed at [off, off + cnt), zeros
// elsewhere; real input when `re` is set.
template <class T_>
struct PadIn {
  const T_* __restrict__ src;
  int64_t stride;
  int off, cnt;
  __device__ __forceinline__ double2 operator()(int i) const {
    const unsigned t = (unsigned)(i - off);
    if (t >= (unsigned)cnt) return cmk(0.0, 0.0);
    if constexpr (sizeof(T_) == sizeof(double)) return cmk(src[(int64_t)t * stride], 0.0);
    else return src[(int64_t)t * stride];
  }
};

// Outputs [off, off + cnt) to an array with element stride `stride`.
struct CropOut {
  double2* __restrict__ dst;
  int64_t stride;
  int off, cnt;
  __device__ __forceinline__ void operator()(int o, double2 v) const {
    const unsigned t = (unsigned)(o - off);
    if (t < (unsigned)cnt) dst[(int64_t)t * stride] = v;
  }
};

// Outputs [off, off + cnt) split into conc = cm * Re and flx = Im.
template <class T_>
struct SplitOut {
  T_* __restrict__ conc;
  T_* __restrict__ flx;
  double cm;
  int off, cnt;
  __device__ __forceinline__ void operator()(int o, double2 v) const {
    const unsigned t = (unsigned)(o - off);
    if (t < (unsigned)cnt) {
      conc[t] = (T_)(cm * v.x);
      flx[t] = (T_)v.y;
    }
  }
};

// One transform of a tile loop; `reuse`: not the workgroup's first tile.
template <int MAXE, class In, class Out>
__device__ __forceinline__ void fft_dir(bool inv, const cplan_t& F, const double2* __restrict__ tw, int tid, int T,
                                        In in, Out out, bool reuse) {
  const bldfm_fft::Lds buf = bldfm_fft::lds_view(smem, F.n);
  if (inv) bldfm_fft::lds_fft<MAXE, true>(buf, smem + F.n, (const FftPlan*)&F, tw + F.tw_off, tid, T, in, out, reuse);
  else bldfm_fft::lds_fft<MAXE, false>(buf, smem + F.n, (const FftPlan*)&F, tw + F.tw_off, tid, T, in, out, reuse);
}

// The four passes, each as a factory of (plan, source, sink, direction) for
// one line of one instance: the single-workgroup kernels below and the
// four-step kernels (k_long) of split lengths run the same definitions.

// Forward, rows: one surface-flux row y placed at [px, px+nx) of nxe points,
// e^{-i} DFT, scale 1/nxe (numpy norm="forward"), keep the nlx retained
// columns in truncated order.
template <class Fn>
__device__ __forceinline__ void pass_fwd_rows(const PlanDev& P, const ExecBufs& B, const cdesc_t& D, int64_t line,
                                              Fn&& fn) {
  const cplan_t& F = *(const cplan_t*)(P.plans + D.plan_x);
  const int y = (int)line;
  fn(F, PadIn<double>{B.src + D.off_src + (int64_t)y * D.nx, 1, D.px, D.nx},
     BandOut{B.ws + D.off_aw + (int64_t)y * D.nlx, 1.0 / (double)F.n, Band(D.nlx, F.n)}, false);
}

// Forward, columns: retained column jx over y placed at [py, py+ny) of nye
// points, e^{-i} DFT, scale 1/nye, keep the nly retained rows -> q^0 (x-major).
template <class Fn>
__device__ __forceinline__ void pass_fwd_cols(const PlanDev& P, const ExecBufs& B, const cdesc_t& D, int64_t line,
                                              Fn&& fn) {
  const cplan_t& F = *(const cplan_t*)(P.plans + D.plan_y);
  const int jx = (int)line;
  fn(F, PadIn<double2>{B.ws + D.off_aw + jx, D.nlx, D.py, D.ny},
     BandOut{B.ws + D.off_q0 + (int64_t)jx * D.nly, 1.0 / (double)F.n, Band(D.nly, F.n)}, false);
}

// Inverse, y-pass: band column cx of slot s (line s*nxb + cx; compact rows
// scattered to their padded indices), unnormalised DFT (e^{-i} footprint,
// e^{+i} dispersion), keep the cropped rows [py, py+ny).
template <class Fn>
__device__ __forceinline__ void pass_inv_cols(const PlanDev& P, const ExecBufs& B, const cdesc_t& D, int64_t line,
                                              Fn&& fn) {
  const cplan_t& F = *(const cplan_t*)(P.plans + D.plan_y);
  const BandIn in{B.ws + D.off_z + line * D.nyb, 1, Band(D.nyb, F.n)};
  // layout 1: column cx of slot s lands at v[s][y][cx]
  const int64_t s = line / D.nxb, cx = line % D.nxb;
  const CropOut out = P.xlayout == 1 ? CropOut{B.ws + D.off_v + s * D.ny * D.nxb + cx, D.nxb, D.py, D.ny}
                                     : CropOut{B.ws + D.off_v + line * D.ny, 1, D.py, D.ny};
  fn(F, in, out, !D.footprint);
}

// Inverse, x-pass: cropped row y of slot s (line s*ny + y) over the band
// columns, DFT, keep [px, px+nx); conc = Re, flx = Im.  Instances served by
// the surrogate carry no concentration spectrum (conc 0).
template <class Fn>
__device__ __forceinline__ void pass_inv_rows(const PlanDev& P, const ExecBufs& B, const cdesc_t& D, int inst,
                                              int64_t line, Fn&& fn) {
  const int s = (int)(line / D.ny), y = (int)(line % D.ny);
  const cplan_t& F = *(const cplan_t*)(P.plans + D.plan_x);
  const BandIn in = P.xlayout == 0
                        ? BandIn{B.ws + D.off_v + (int64_t)s * D.nxb * D.ny + y, D.ny, Band(D.nxb, F.n)}
                        : BandIn{B.ws + (P.xlayout == 1 ? D.off_v : D.off_vt) + ((int64_t)s * D.ny + y) * D.nxb,
                                 1, Band(D.nxb, F.n)};
  const int64_t o = D.off_out + line * D.nx;
  const double cm = (B.mode && B.mode[inst] == 0) ? 0.0 : 1.0;
  if (D.out_f32)
    fn(F, in, SplitOut<float>{(float*)B.conc + o, (float*)B.flx + o, cm, D.px, D.nx}, !D.footprint);
  else
    fn(F, in, SplitOut<double>{(double*)B.conc + o, (double*)B.flx + o, cm, D.px, D.nx}, !D.footprint);
}

template <class Fn>
__device__ __forceinline__ void run_pass(int pass, const PlanDev& P, const ExecBufs& B, const cdesc_t& D, int inst,
                                         int64_t line, Fn&& fn) {
  switch (pass) {
    case PASS_FWD_ROWS: pass_fwd_rows(P, B, D, line, fn); break;
    case PASS_FWD_COLS: pass_fwd_cols(P, B, D, line, fn); break;
    case PASS_INV_COLS: pass_inv_cols(P, B, D, line, fn); break;
    default: pass_inv_rows(P, B, D, inst, line, fn); break;
  }
}

// Four-step sources and sinks: step A reads the strided sub-sequence
// in(j1 n2 + j2) and stores the twiddled length-n1 result at scr[j2 n1 + k1];
// step B reads scr[j2 n1 + k1] over j2 and writes X[k1 + n1 k2] through the
// pass's own sink.
template <class In>
struct SubIn {
  In in;
  int n2, j2;
  __device__ __forceinline__ double2 operator()(int j1) const { return in(j1 * n2 + j2); }
};
struct TwiddleOut {
  double2* __restrict__ dst;      // scr + j2 n1
  const double2* __restrict__ w;  // W_n^t, t < n
  int j2;
  bool inv;
  __device__ __forceinline__ void operator()(int k1, double2 v) const {
    double2 t = w[j2 * k1];  // j2 k1 < n: no reduction modulo n
    if (inv) t.y = -t.y;
    dst[k1] = cmul(v, t);
  }
};
struct ScrIn {
  const double2* __restrict__ src;  // scr + k1
  int n1;
  __device__ __forceinline__ double2 operator()(int j2) const { return src[(int64_t)j2 * n1]; }
};
template <class Out>
struct SubOut {
  Out out;
  int n1, k1;
  __device__ __forceinline__ void operator()(int k2, double2 v) const { out(k1 + n1 * k2, v); }
};
