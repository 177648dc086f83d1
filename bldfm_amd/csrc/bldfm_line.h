// Chirp transforms of the solver's passes on compile-time power-of-two lengths.
//
// A pass needs, of a length-N DFT, only a window of the outputs of a window
// of the inputs:
//   X[o0 + v] = sum_{u < nin} x[u] W_N^{(i0 + u)(o0 + v)},  v < nout,
// W_N = e^{-2 pi i/N} (the e^{+i} transform conjugates input and output).  With
// 2 i o = i^2 + o^2 - (o - i)^2 (L. Bluestein, IEEE Trans. Audio Electroacoust.
// 18:451, 1970) that is a convolution of length M >= nin + nout - 1: two
// transforms of length M and three tables.  What it costs depends on the
// windows, a third of N each at the default halo, and not on N's factors, where
// the mixed-radix passes run a prime p > 5 as p products a point.  Windows of more
// than 2048 values (above 1024 cells an axis at the default halo) stay there.
//
// One workgroup of 256 threads takes 2048/M lines; a line's T = M/8 lanes sit
// in one wave up to M = 512, so its exchanges through LDS need no barrier.  At
// 100 registers and 41 KB of LDS a workgroup (three to four waves a SIMD) the
// two transforms' vector work and its LDS latency bound it, not its traffic:
// the y-pass of 256 footprints with 374-point lines (2 * 11 * 17) takes 47 us
// against 278 us in the mixed-radix kernel, 1.4 TB/s.
#pragma once
#include "bldfm_fft.h"
#include "bldfm_march.h"

namespace bldfm_line {

using bldfm_fft::butterfly;

// LDS positions of an exchange buffer: i ^ ((i >> 3) & 7) (see bldfm_fft.h).
__device__ __forceinline__ int phys(int i) { return i ^ ((i >> 3) & 7); }

template <bool WAVE>
__device__ __forceinline__ void line_sync() {
  if constexpr (WAVE) {  // a wave's LDS operations execute in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// Stage twiddles of the length-M transform in LDS, [r-1][k] per stage so that
// a wave's lanes read consecutive entries: W_64^{kr} (k < 8, r < 8), then what
// line_tw_len counts.  w: the M-entry table W_M^t (global).
__device__ __forceinline__ void fill_twiddles(double2* tw, int lm, const double2* __restrict__ w, int tid) {
  const int M = 1 << lm, n = line_tw_len(lm);
  for (int i = tid; i < n; i += 256) {
    int j = i, t;
    if (j < 56) {
      t = ((j & 7) * ((j >> 3) + 1)) << (lm - 6);
    } else if (lm < 9) {  // last stage, radix M/64: W_M^{kr}, k < 64
      j -= 56;
      t = (j & 63) * ((j >> 6) + 1);
    } else if (j < 504) {  // radix 8 at Ns = 64: W_512^{kr}
      j -= 56;
      t = ((j & 63) * ((j >> 6) + 1)) << (lm - 9);
    } else {  // last stage, radix M/512: W_M^{kr}, k < 512
      j -= 504;
      t = (j & 511) * ((j >> 9) + 1);
    }
    tw[i] = w[t & (M - 1)];
  }
}

// Length-M DFT (e^{-i}) of the values x[r] = element t + T r, in place (same
// order out): Stockham stages of radix 8, 8, ... with one of 2, 4 or 8 last.
template <int LM>
__device__ __forceinline__ void fft_regs(double2 (&x)[8], double2* ex, const double2* tw, int t) {
  constexpr int M = 1 << LM, T = M / 8;
  constexpr bool W = T <= 64;
  auto gather = [&] {
    line_sync<W>();
    if constexpr (T >= 64) {
      const int p = phys(t);
#pragma unroll
      for (int r = 0; r < 8; ++r) x[r] = ex[p + T * r];
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r) x[r] = ex[phys(t + T * r)];
    }
    line_sync<W>();
  };
  butterfly<8>(x, false);
  {
    const int b = 8 * t, m = t & 7;
#pragma unroll
    for (int r = 0; r < 8; ++r) ex[b + (r ^ m)] = x[r];
  }
  gather();
  const int k1 = t & 7;
#pragma unroll
  for (int r = 1; r < 8; ++r) x[r] = cmul(x[r], tw[(r - 1) * 8 + k1]);
  butterfly<8>(x, false);
  if constexpr (LM == 6) return;
  {
    const int b = (t - k1) * 8;
#pragma unroll
    for (int r = 0; r < 8; ++r) ex[b + 8 * r + (k1 ^ r)] = x[r];
  }
  gather();
  const double2* tw2 = tw + 56;
  if constexpr (LM == 7) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const double2 c = cmul(x[b + 4], tw2[t + T * b]);
      x[b + 4] = csub(x[b], c);
      x[b] = cadd(x[b], c);
    }
  } else if constexpr (LM == 8) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      double2 y[4] = {x[b], x[b + 2], x[b + 4], x[b + 6]};
#pragma unroll
      for (int r = 1; r < 4; ++r) y[r] = cmul(y[r], tw2[(r - 1) * 64 + t + T * b]);
      butterfly<4>(y, false);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[b + 2 * r] = y[r];
    }
  } else {
    const int k2 = t & 63;
#pragma unroll
    for (int r = 1; r < 8; ++r) x[r] = cmul(x[r], tw2[(r - 1) * 64 + k2]);
    butterfly<8>(x, false);
    if constexpr (LM > 9) {
      const int b = (t - k2) * 8 + (k2 ^ ((k2 >> 3) & 7));
#pragma unroll
      for (int r = 0; r < 8; ++r) ex[b + 64 * r] = x[r];
      gather();
      const double2* tw3 = tw + 504;
      if constexpr (LM == 10) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double2 c = cmul(x[q + 4], tw3[t + T * q]);
          x[q + 4] = csub(x[q], c);
          x[q] = cadd(x[q], c);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          double2 y[4] = {x[q], x[q + 2], x[q + 4], x[q + 6]};
#pragma unroll
          for (int r = 1; r < 4; ++r) y[r] = cmul(y[r], tw3[(r - 1) * 512 + t + T * q]);
          butterfly<4>(y, false);
#pragma unroll
          for (int r = 0; r < 4; ++r) x[q + 2 * r] = y[r];
        }
      }
    }
  }
}

// One line of a tile.  load(u): input u < nin (conjugated by the caller for
// e^{+i}), zero on the lanes of a line that does not exist, so that every wave
// runs the same code; store(v, X): output v < nout, nothing for such a line.
// STAGED: load reads LDS where other waves' exchanges go.
template <int LM, bool STAGED = false, class Load, class Store>
__device__ __forceinline__ void run_line(const LineAlg& A, const double2* __restrict__ twp, int t, double2* ex,
                                         const double2* tw, Load load, Store store) {
  constexpr int M = 1 << LM, T = M / 8;
  const double2* __restrict__ tab = twp + A.tab;  // A (nin), B (nout), H (M)
  double2 x[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int e = t + T * r;
    x[r] = e < A.nin ? cmul(load(e), tab[e]) : cmk(0.0, 0.0);
  }
  if constexpr (STAGED) __syncthreads();  // every wave has its inputs
#pragma unroll 1
  for (int it = 0; it < 2; ++it) {
    int to = t;
    asm volatile("" : "+v"(to));  // index arithmetic stays inside the loop: hoisted, it costs registers
    fft_regs<LM>(x, ex, tw, to);
    if (it == 0) {
#pragma unroll
      for (int r = 0; r < 8; ++r) x[r] = cconj(cmul(x[r], tab[A.nin + A.nout + to + T * r]));
    }
  }
#pragma unroll
  for (int r = 0; r < 8; ++r) {
    const int v = t + T * r;
    if (v < A.nout) store(v, cmul(cconj(x[r]), tab[A.nin + v]));
  }
}

}  // namespace bldfm_line

extern __shared__ double2 line_smem[];

// ---------------------------------------------------------------- chirp passes
// One tile (line_per_wg(lm) lines) of a pass.  Lines whose elements are
// strided in memory (the x-pass over v[s][cx][y], the forward columns) are
// neighbours there, so the workgroup reads them together, NL consecutive
// values at a time, and hands them over through LDS.
template <int LM, int PASS>
__device__ __forceinline__ void line_tile(const PlanDev& P, const ExecBufs& B, const cdesc_t& D, int inst, int local,
                                          double2* ex0, const double2* tw) {
  constexpr int M = 1 << LM, T = M / 8, NL = 256 / T;
  const int tid = (int)threadIdx.x, l = tid / T, t = tid % T;
  const LineAlg A = [&] {
    const auto& a = D.line[PASS];
    LineAlg r;
    r.lm = a.lm; r.N = a.N; r.nin = a.nin; r.i0 = a.i0; r.nout = a.nout; r.o0 = a.o0;
    r.tw = a.tw; r.tab = a.tab;
    return r;
  }();
  double2* ex = ex0 + l * M;
  const double sg = (PASS >= PASS_INV_COLS && !D.footprint) ? -1.0 : 1.0;  // e^{+i}: conjugate in and out
  // band position of input u (inverse) or output v (forward)
  auto band_in = [&](int u) { const int f = A.i0 + u; return f < 0 ? f + A.nin : f; };
  auto band_out = [&](int v) { const int f = A.o0 + v; return f < 0 ? f + A.nout : f; };
  if constexpr (PASS == PASS_FWD_ROWS) {
    const int y = local * NL + l;
    const bool live = y < D.ny;
    const double* src = B.src + D.off_src + (int64_t)y * D.nx;
    double2* dst = B.ws + D.off_aw + (int64_t)y * D.nlx;
    const double sc = 1.0 / (double)A.N;
    bldfm_line::run_line<LM>(A, P.tw, t, ex, tw,
                             [&](int u) { return live ? cmk(src[u], 0.0) : cmk(0.0, 0.0); },
                             [&](int v, double2 X) { if (live) dst[band_out(v)] = cscale(sc, X); });
  } else if constexpr (PASS == PASS_INV_COLS) {
    const int64_t line = (int64_t)local * NL + l;
    const bool live = line < (int64_t)D.nslot * D.nxb;
    const double2* src = B.ws + D.off_z + line * D.nyb;
    const int64_t s = line / D.nxb, cx = line % D.nxb;
    double2* dst = P.xlayout == 1 ? B.ws + D.off_v + s * D.ny * D.nxb + cx : B.ws + D.off_v + line * D.ny;
    const int64_t st = P.xlayout == 1 ? D.nxb : 1;
    bldfm_line::run_line<LM>(A, P.tw, t, ex, tw,
                             [&](int u) {
                               if (!live) return cmk(0.0, 0.0);
                               const double2 z = src[band_in(u)];
                               return cmk(z.x, sg * z.y);
                             },
                             [&](int v, double2 X) { if (live) dst[(int64_t)v * st] = cmk(X.x, sg * X.y); });
  } else {
    const int lines = PASS == PASS_FWD_COLS ? D.nlx : D.ny;  // per slot
    const int per = (lines + NL - 1) / NL;
    const int s = local / per, line0 = (local % per) * NL, line = line0 + l;
    const bool live = line < lines;
    const bool rows = PASS == PASS_INV_ROWS && P.xlayout != 0;  // v is already row-major
    const double2* src;
    if (PASS == PASS_FWD_COLS) src = B.ws + D.off_aw;
    else if (!rows) src = B.ws + D.off_v + (int64_t)s * D.nxb * D.ny;
    else src = B.ws + (P.xlayout == 1 ? D.off_v : D.off_vt) + ((int64_t)s * D.ny + line) * D.nxb;
    const int pitch = line_pitch(LM, A.nin);
    if (!rows) {
      for (int i = tid; i < NL * A.nin; i += 256) {
        const int q = i % NL, u = i / NL;
        double2 z = cmk(0.0, 0.0);
        if (line0 + q < lines)
          z = src[(int64_t)(PASS == PASS_FWD_COLS ? u : band_in(u)) * lines + line0 + q];
        ex0[q * pitch + u] = z;
      }
      __syncthreads();
    }
    auto load = [&](int u) {
      double2 z = cmk(0.0, 0.0);
      if (!rows) z = ex0[l * pitch + u];
      else if (live) z = src[band_in(u)];
      return cmk(z.x, sg * z.y);
    };
    if constexpr (PASS == PASS_FWD_COLS) {
      double2* dst = B.ws + D.off_q0 + (int64_t)line * D.nly;
      const double sc = 1.0 / (double)A.N;
      bldfm_line::run_line<LM, true>(A, P.tw, t, ex, tw, load,
                                     [&](int v, double2 X) { if (live) dst[band_out(v)] = cscale(sc, X); });
    } else {
      const int64_t o = D.off_out + ((int64_t)s * D.ny + line) * D.nx;
      const double cm = (B.mode && B.mode[inst] == 0) ? 0.0 : 1.0;
      if (D.out_f32) {
        float *c = (float*)B.conc + o, *f = (float*)B.flx + o;
        bldfm_line::run_line<LM, true>(A, P.tw, t, ex, tw, load, [&](int v, double2 X) {
          if (live) { c[v] = (float)(cm * X.x); f[v] = (float)(sg * X.y); }
        });
      } else {
        double *c = (double*)B.conc + o, *f = (double*)B.flx + o;
        bldfm_line::run_line<LM, true>(A, P.tw, t, ex, tw, load, [&](int v, double2 X) {
          if (live) { c[v] = cm * X.x; f[v] = sg * X.y; }
        });
      }
    }
  }
}

// One kernel per pass and length: with a switch over the lengths inside this
// loop the compiler kept every length's indices live and spilled 500 registers.
template <int PASS, int LM>
__global__ __launch_bounds__(256, 4) void k_line(PlanDev P, ExecBufs B, const TileRec* recs, int64_t tot) {
  double2* ex0 = line_smem + line_tw_len(LM);
  for (int64_t b = blockIdx.x; b < tot; b += gridDim.x) {
    const int64_t t = gridDim.x >= tot ? xcd_swizzle(b, tot) : b;
    const TileRec tr = tile_rec(recs, t);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    if (b == blockIdx.x) bldfm_line::fill_twiddles(line_smem, LM, P.tw + D.line[PASS].tw, (int)threadIdx.x);
    __syncthreads();  // the tables are there, and the previous tile is done
    line_tile<LM, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem);
  }
}

// The tiles of all lengths of one pass in one launch, a workgroup each: length
// 2^(LINE_MIN_LM + k) has the workgroups first[k] .. first[k + 1] - 1.  A launch a
// length cost each further length 4 to 5 us of a tail that fills no CU: whole
// batches of three to seven instances with windows of 28 to 208 values took 68 to 83
// us, 10 to 17 more than all in the mixed radix, and take 43 to 44.  The switch
// stands outside any loop: inside the tile loop every length's indices were hoisted
// out of it (500 registers spilled); so it takes 92 and 108, as the kernels of one
// length do.
//
// Up to LINE_MERGE_TILES: where the tiles fill the chip many times over, all lengths
// having the longest's LDS (65 KB, two workgroups a CU) costs more than the tails
// (seven instances of M = 64 .. 2048 each k times, about 950 k tiles a pass, launched
// apart and together: k = 4 419 and 373 us, 16 1352 and 1342, 24 1995 and 1989, 32 2592
// and 2673; three of M = 256 .. 1024 each 64 times, 12000 tiles, 675 and 675).
#define LINE_MERGE_TILES 8192
struct LineTiles {
  const TileRec* recs[LINE_NLM];
  int32_t first[LINE_NLM + 1];
};
template <int PASS>
__global__ __launch_bounds__(256, 4) void k_lines(PlanDev P, ExecBufs B, LineTiles L) {
  const int b = (int)blockIdx.x;
  int k = 0;
  while (b >= L.first[k + 1]) ++k;
  const TileRec tr = tile_rec(L.recs[k], b - L.first[k]);
  const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
  const int lm = LINE_MIN_LM + k;
  bldfm_line::fill_twiddles(line_smem, lm, P.tw + D.line[PASS].tw, (int)threadIdx.x);
  __syncthreads();
  double2* ex0 = line_smem + line_tw_len(lm);
  switch (lm) {
    case 6: line_tile<6, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem); break;
    case 7: line_tile<7, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem); break;
    case 8: line_tile<8, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem); break;
    case 9: line_tile<9, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem); break;
    case 10: line_tile<10, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem); break;
    default: line_tile<11, PASS>(P, B, D, tr.inst, tr.local, ex0, line_smem); break;
  }
}
// Launches a plan's lines of one pass, or (lds_attr > 0) only allows that much
// dynamic LDS in the pass's kernels.
template <int PASS>
static int launch_lines(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int grid_cap, hipStream_t stream, int lds_attr) {
  auto one = [&](auto* fn, int k) {
    if (lds_attr > 0) {
      (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds_attr);
      return 0;
    }
    const int64_t n = L.tot[PASS][k];
    if (n <= 0) return 0;
    fn<<<(unsigned)(n < grid_cap ? n : grid_cap), 256, (size_t)L.lds[PASS][k], stream>>>(P, B, L.recs[PASS][k], n);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : -(int)e - 1000;
  };
  int lengths = 0, lds = 0;
  int64_t tiles = 0;
  for (int k = 0; k < LINE_NLM; ++k)
    if (L.tot[PASS][k] > 0) {
      ++lengths;
      tiles += L.tot[PASS][k];
      lds = L.lds[PASS][k] > lds ? L.lds[PASS][k] : lds;
    }
  if (lds_attr > 0) {
    (void)hipFuncSetAttribute((const void*)&k_lines<PASS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_attr);
  } else if (lengths > 1 && tiles <= LINE_MERGE_TILES) {
    LineTiles T;
    for (int k = 0, at = 0; k <= LINE_NLM; ++k) {
      T.first[k] = at;
      if (k == LINE_NLM) break;
      T.recs[k] = L.recs[PASS][k];
      at += (int)L.tot[PASS][k];
    }
    k_lines<PASS><<<(unsigned)tiles, 256, (size_t)lds, stream>>>(P, B, T);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : -(int)e - 1000;
  }
  int rc = one(&k_line<PASS, 6>, 0);
  if (!rc) rc = one(&k_line<PASS, 7>, 1);
  if (!rc) rc = one(&k_line<PASS, 8>, 2);
  if (!rc) rc = one(&k_line<PASS, 9>, 3);
  if (!rc) rc = one(&k_line<PASS, 10>, 4);
  if (!rc) rc = one(&k_line<PASS, 11>, 5);
  return rc;
}
