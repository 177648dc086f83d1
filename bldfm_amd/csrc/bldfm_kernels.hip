// HIP kernels of the BLDFM steady-state solver for gfx950 (MI355X).
//
// Pipeline per solve instance (all FP64):
//   k_level_table  per-step constants of the vertical march (profiles from
//                  caller arrays, or evaluated here from met scalars)
//   k_fwd_rows/cols  dispersion mode only: pruned forward 2-D DFT of the
//                  halo-padded surface flux onto the retained modes
//   k_shoot_*      one lane per Fourier mode: two initial-value problems,
//                  radiation condition, shooting, (0,0) trapezoid, phase
//                  shift, Hermitian packing of p^ and q^ into Z = Hp + i Hq
//   k_nyq_fix      Hermitian part on the unpaired Nyquist row/column where a
//                  Nyquist mode's mirror is retained too (modes = padded grid)
//   k_inv_cols/rows  pruned inverse 2-D DFT of Z: y-pass over the band
//                  columns, x-pass over the cropped rows; Re -> conc, Im -> flx
//
// Work of a batch of instances is laid out as tiles with per-kernel prefix
// sums; every kernel is a grid-stride loop over its tiles.
#include "bldfm_internal.h"
#include "bldfm_march.h"

// ---------------------------------------------------------------- level table
// Entry i < nz-1 (step from z_i to z_{i+1}, coefficients of the LOWER level,
// src/bldfm/solver.py:357-364), with kappa = 1/Kz_i, h = z_{i+1} - z_i:
//   [0..3]  Kx, Ky, u, v
//   [4..11] the reference's scalar sub-expressions, rounded as numba rounds
//           them: sa = 0.5*kappa, h2 = h*h, b0 = (-kappa)*h,
//           sb = (1/6)*(kappa*kappa), h3 = h*(h*h), h, sc = (1/6)*kappa,
//           W = 0.5/Kz_i + 0.5/Kz_{i+1}  (trapezoid weight of the (0,0) mode)
//   [12..14] fused-path coefficients A = sa*h2, B1 = sb*h3, C = sc*h3; [15] 2 sc
// so that T = -(Kx lx^2 + Ky ly^2) - i(u lx + v ly), a = d = 1 - sa T h2,
// b = b0 - sb T h3, c = T h - sc T^2 h3.
// Entry nz-1 (top, src/bldfm/solver.py:164-174):
//   {Kx/Kz, Ky/Kz, u/Kz, v/Kz, Kz, 1/Kz} (products with 1/Kz as the reference forms them)
// One level-table row from the profile values (z,u,v,Kx,Ky,Kz) of level i
// (cur) and level i+1 (nxt, unused for the top row).
__device__ __forceinline__ void fill_level_row(const double* cur, const double* nxt, bool top,
                                               double* __restrict__ T) {
#pragma clang fp contract(off)
  const double kz = cur[5];
  const double kinv = 1.0 / kz;
  if (!top) {
    const double h = nxt[0] - cur[0];
    const double h2 = h * h;
    const double h3 = h * h2;
    const double sixth = 1.0 / 6.0;
    const double sa = 0.5 * kinv, sb = sixth * (kinv * kinv), sc = sixth * kinv;
    T[0] = cur[3];
    T[1] = cur[4];
    T[2] = cur[1];
    T[3] = cur[2];
    T[4] = sa;
    T[5] = h2;
    T[6] = -kinv * h;
    T[7] = sb;
    T[8] = h3;
    T[9] = h;
    T[10] = sc;
    T[11] = 0.5 / kz + 0.5 / nxt[5];
    T[12] = sa * h2;
    T[13] = sb * h3;
    T[14] = sc * h3;
    T[15] = sc + sc;
  } else {
    T[0] = cur[3] * kinv;
    T[1] = cur[4] * kinv;
    T[2] = cur[1] * kinv;
    T[3] = cur[2] * kinv;
    T[4] = kz;
    T[5] = kinv;
    for (int c = 6; c < BLDFM_LEVEL_STRIDE; ++c) T[c] = 0.0;
  }
}

// Profiles of up to 256 levels i0 + tid by a workgroup of 4 x 256 threads,
// same values as prof_point.  A level's correctly rounded functions are one
// long serial chain (about nine logarithms), and a plan has few levels, so the
// four groups evaluate what does not depend on each other: z, then log(z/z0),
// xi and phi, then psi's two logarithms and its arctangent; the chain is about
// half as long.  A wave issues one of its dependent FP64 operations every eight
// cycles, so the groups' waves of the same levels go to different SIMDs
// (on one SIMD they took as long as one wave): the unstable profiles of 26
// levels take 12.5 us instead of 27, k_level_table of 96 footprints 16.4 instead
// of 32.7.
// Leaves out = {z, u, v, Kx, Ky, Kz} in the registers of group 0.
struct GroupSlot {
  int grp, tid;
};
__device__ __forceinline__ GroupSlot group_slot() {
  const int wave = (int)threadIdx.x >> 6, grp = wave >> 2;  // wave w runs on SIMD w mod 4
  return GroupSlot{grp, ((wave + grp) & 3) * 64 + (int)(threadIdx.x & 63)};
}
__device__ __forceinline__ void prof_group(const ProfSetup& S, int i, bool live, double (*sh)[256], double out[6]) {
#pragma clang fp contract(off)
  const int tid = group_slot().tid, grp = group_slot().grp;
  const bool most = S.closure == CL_MOST || S.closure == CL_MOSTM;
  __syncthreads();  // the last call's values (and its caller's) are read
  if (!most) {
    // z and at most one logarithm of it, one after the other: nothing to share out
    if (grp == 0 && live) {
      const double z = prof_z(S, i);
      prof_combine(S, z, S.closure == CL_CONSTANT ? 0.0 : cr_log(z / S.z0), 0.0, 1.0, out);
    }
    return;
  }
  if (grp == 0 && live) sh[0][tid] = prof_z(S, i);
  __syncthreads();
  const double z = sh[0][tid], x = z / S.mol;
  if (live) {
    if (grp == 0) sh[1][tid] = cr_log(z / S.z0);
    if (grp == 1 && !(x > 0.0)) sh[2][tid] = gl_cpow_real(1.0 - 16.0 * x, 0.25);
    if (grp == 2) sh[3][tid] = most_phi(x);
  }
  __syncthreads();
  if (live && !(x > 0.0)) {
    const double xi = sh[2][tid];
    if (grp == 1) sh[4][tid] = cr_log(0.5 * (1.0 + xi));
    if (grp == 2) sh[5][tid] = cr_log(0.5 * (1.0 + xi * xi));
    if (grp == 3) sh[6][tid] = cr_atan(xi);
  }
  __syncthreads();
  if (grp == 0 && live)
    prof_combine(S, z, sh[1][tid], x > 0.0 ? 5.0 * x : psi_of(sh[4][tid], sh[5][tid], sh[6][tid]), sh[3][tid], out);
}

__global__ __launch_bounds__(1024) void k_level_table(PlanDev P, ExecBufs B) {
#pragma clang fp contract(off)
  // levels evaluated from met in this tile: 256 of them and the one above
  __shared__ double lev[6][257];
  __shared__ double sh[7][256];
  for (int64_t t = blockIdx.x; t < P.tot_tab; t += gridDim.x) {
    const TileRec tr = tile_rec(P.t_tab, t);
    const int inst = tr.inst;
    const cdesc_t& D = *(const cdesc_t*)(P.desc + inst);
    const int nz = D.nz;
    const int tid = group_slot().tid, grp = group_slot().grp;
    const int i = tr.local * 256 + tid;
    double* prof = B.prof + D.off_prof;
    double cur[6], nxt[6];
    if (P.met_flag[inst]) {  // uniform over the workgroup (one instance per tile)
      // every level once: group 0 its level, and where the tile ends inside the
      // grid one thread of group 3 the next tile's first
      const ProfSetup& S = P.met[inst];
      prof_group(S, i, i < nz, sh, cur);
      if (grp == 0 && i < nz)
        for (int c = 0; c < 6; ++c) {
          prof[(int64_t)c * nz + i] = cur[c];
          lev[c][tid] = cur[c];
        }
      if (grp == 3 && tid == 255 && i + 1 < nz) {
        prof_point(S, i + 1, nxt);
        for (int c = 0; c < 6; ++c) lev[c][256] = nxt[c];
      }
      __syncthreads();
      if (i + 1 < nz)
        for (int c = 0; c < 6; ++c) nxt[c] = lev[c][tid + 1];
    } else {
      if (i < nz)
        for (int c = 0; c < 6; ++c) cur[c] = prof[(int64_t)c * nz + i];
      if (i + 1 < nz)
        for (int c = 0; c < 6; ++c) nxt[c] = prof[(int64_t)c * nz + i + 1];
    }
    if (grp == 0 && i < nz)
      fill_level_row(cur, nxt, i == nz - 1, B.tab + D.off_tab + (int64_t)i * BLDFM_LEVEL_STRIDE);
  }
}

// Value of `v` in lane j (uniform) of the wave.
__device__ __forceinline__ double lane_value(double v, int j) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), j);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), j);
  return __hiloint2double(hi, lo);
}

// Degenerate mode (0,0): flux conserved, p by the trapezoid rule in z
// (src/bldfm/solver.py:190-191, 239-251): p00 <- p00 - (q00*dz)*W.  The whole
// wave that holds the origin lane runs this: each lane loads one row and forms
// its term, and only the subtractions stay serial.  As one lane's loop with
// dependent loads in every row it held back its wave's march (k_shoot of a
// 64x128 footprint 16.9 -> 12.5 us, of a 512^2 one 43.6 -> 41.5 us).
__device__ void origin_numeric(const cdesc_t& D, const double* __restrict__ tab,
                               const int32_t* __restrict__ slot, double2* __restrict__ ws) {
#pragma clang fp contract(off)
  const int l = (int)(threadIdx.x & 63);
  const double q00 = D.footprint ? D.q00 : ws[D.off_q0].x;
  double p00 = D.p000;
  for (int i0 = 0; i0 < D.nz; i0 += 64) {
    const int i = i0 + l;
    double term = 0.0, mine = 0.0;
    if (i < D.nz - 1) {
      const double* T = tab + (int64_t)i * BLDFM_LEVEL_STRIDE;
      term = (q00 * T[9]) * T[11];
    }
    const int n = D.nz - i0 < 64 ? D.nz - i0 : 64;
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
      if (l == j) mine = p00;
      p00 = p00 - lane_value(term, j);
    }
    const int sl = i < D.nz ? slot[i] : -1;
    if (sl >= 0) emit_origin(D, ws, sl, mine, q00);
  }
  if (l == 0)
    for (int s = D.nfilled; s < D.nslot; ++s) emit_origin(D, ws, s, s == 0 ? D.p000 : 0.0, q00);
}

// Numerical branch.  MAXS register snapshots (RECOMP == false), or a second
// march from the bottom after the shooting coefficient is known
// (RECOMP == true) for many output levels.  Both give the same values.
template <int MAXS, bool RECOMP, bool EXACT, int BLOCK>
__global__ __launch_bounds__(BLOCK, MAXS == 1 ? 5 : 3) void k_shoot(PlanDev P, ExecBufs B, int variant) {
  for (int64_t t = blockIdx.x; t < P.tot_shoot; t += gridDim.x) {
    const TileRec tr = tile_rec(P.t_shoot, t);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    if (D.variant != variant || D.exact != (int)EXACT || D.pair) continue;
    if (B.mode && B.mode[tr.inst] == 0) continue;  // accepted surrogate instance
    Lane L;
    const int lane = tr.local * BLOCK + (int)threadIdx.x;
    const double* __restrict__ tab = B.tab + D.off_tab;
    const int wave0 = __builtin_amdgcn_readfirstlane(lane);  // the wave's lanes are wave0 .. wave0 + 63
    const int o = origin_lane(D.nlx, D.nly) - wave0;
    if (o >= 0 && o < 64) origin_numeric(D, tab, P.ints + D.off_slot, B.ws);
    if (!lane_setup(D, lane, L) || L.kind == LANE_ORIGIN) continue;
    ctab_t* __restrict__ ctab = (ctab_t*)tab;
    cint_t* __restrict__ slot = (cint_t*)(P.ints + D.off_slot);
    const int nz = D.nz;
    const double lx = L.lx, ly = L.ly, lx2 = xmul(lx, lx), ly2 = xmul(ly, ly);
    const double2 q0 = ivp2_init(D, L, B.ws);
    double2 p1 = cmk(1.0, 0.0), q1 = cmk(0.0, 0.0), p2 = cmk(0.0, 0.0), q2 = q0;
    double2 sp1[MAXS], sq1[MAXS], sp2[MAXS], sq2[MAXS];
#pragma unroll
    for (int s = 0; s < MAXS; ++s) sp1[s] = sq1[s] = sp2[s] = sq2[s] = cmk(0.0, 0.0);
    // the next row is fetched while the current step computes; unrolled by
    // two so the prefetched row and the (p, q) state alternate between two
    // register sets instead of being copied every step.  The snapshot levels
    // come from the descriptor (uniform compares), so no step waits on a
    // load issued in the same step.
    int snap[MAXS];
#pragma unroll
    for (int s = 0; s < MAXS; ++s) snap[s] = D.snap_level[s];
    Row nxt = load_row(ctab);
#pragma unroll 2
    for (int i = 0; i < nz - 1; ++i) {
      if (!RECOMP) {
#pragma unroll
        for (int s = 0; s < MAXS; ++s)
          if (i == snap[s]) { sp1[s] = p1; sq1[s] = q1; sp2[s] = p2; sq2[s] = q2; }
      }
      const Row cur = nxt;
      if (i + 1 < nz - 1) nxt = load_row(ctab + (int64_t)(i + 1) * BLDFM_LEVEL_STRIDE);
      march_step<EXACT>(cur, lx, ly, lx2, ly2, p1, q1, p2, q2);
    }
    if (!RECOMP) {
#pragma unroll
      for (int s = 0; s < MAXS; ++s)
        if (nz - 1 == snap[s]) { sp1[s] = p1; sq1[s] = q1; sp2[s] = p2; sq2[s] = q2; }
    }
    const double* tt = tab + (int64_t)(nz - 1) * BLDFM_LEVEL_STRIDE;
    const double2 alpha = shoot_alpha(tt, top_lambda(tt, lx, ly, lx2, ly2), p1, q1, p2, q2);
    const double2 sh = phase_shift(D, L);
    if (!RECOMP) {
#pragma unroll
      for (int s = 0; s < MAXS; ++s)
        if (s < D.nfilled)
          emit_mode(D, L, B.ws, s, xcadd(ncmul(alpha, sp1[s]), sp2[s]),
                    xcadd(ncmul(alpha, sq1[s]), sq2[s]), sh);
    } else {
      p1 = cmk(1.0, 0.0); q1 = cmk(0.0, 0.0); p2 = cmk(0.0, 0.0); q2 = q0;
      Row nxt2 = load_row(ctab);
      for (int i = 0; i <= D.max_level; ++i) {
        const int sl = slot[i];
        if (sl >= 0)
          emit_mode(D, L, B.ws, sl, xcadd(ncmul(alpha, p1), p2), xcadd(ncmul(alpha, q1), q2), sh);
        if (i < D.max_level) {
          const Row cur = nxt2;
          if (i + 1 < D.max_level) nxt2 = load_row(ctab + (int64_t)(i + 1) * BLDFM_LEVEL_STRIDE);
          march_step<EXACT>(cur, lx, ly, lx2, ly2, p1, q1, p2, q2);
        }
      }
    }
    for (int s = D.nfilled; s < D.nslot; ++s) emit_mode(D, L, B.ws, s, cmk(0.0, 0.0), cmk(0.0, 0.0), sh);
  }
}

// The numerical branch with a mode and its mirror in x per lane (exact
// rounding; one register snapshot, or the second march).  The march is bound
// by FP64 issue (95% of the slots) and by the clock the card holds under it,
// so the operations that a pair shares are its gain: 128 footprints of 512^2 x
// 64 take 1.44e9 vector instructions instead of 1.57e9 and 10% fewer cycles, of
// which the lower clock (1.83 against 1.99 GHz) takes half: 2.74 -> 2.64 ms.
// With one snapshot it is at its 128 registers (four waves a SIMD) and spills two
// to four, stored and reloaded once a tile outside the march: 593 MB of traffic
// for 539, where the one-mode march has 570.
template <bool RECOMP, int BLOCK>
__global__ __launch_bounds__(BLOCK, 4) void k_shoot_pair(PlanDev P, ExecBufs B, int variant) {
  for (int64_t t = blockIdx.x; t < P.tot_shoot; t += gridDim.x) {
    const TileRec tr = tile_rec(P.t_shoot, t);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    if (D.variant != variant || !D.pair) continue;
    if (B.mode && B.mode[tr.inst] == 0) continue;  // accepted surrogate instance
    const int lane = tr.local * BLOCK + (int)threadIdx.x;
    const double* __restrict__ tab = B.tab + D.off_tab;
    const int wave0 = __builtin_amdgcn_readfirstlane(lane);
    const int o = pair_origin_lane(D.nlx, D.nly) - wave0;
    if (o >= 0 && o < 64) origin_numeric(D, tab, P.ints + D.off_slot, B.ws);
    if (lane >= D.plane) continue;
    Lane L;
    L.fx = L.fy = 0;
    int two, nidx2;
    L.kind = decode_pair(lane, D.nlx, D.nly, &L.fx, &L.fy, &L.nidx, &two, &nidx2);
    if (L.kind == LANE_IDLE || L.kind == LANE_ORIGIN) continue;
    L.lx = xmul(D.sx, xmul((double)L.fx, D.vx));
    L.ly = xmul(D.sy, xmul((double)L.fy, D.vy));
    Lane L2 = L;
    if (two) {
      L2.fx = -L.fx;
      L2.lx = -L.lx;
      L2.nidx = nidx2;
    }
    ctab_t* __restrict__ ctab = (ctab_t*)tab;
    cint_t* __restrict__ slot = (cint_t*)(P.ints + D.off_slot);
    const int nz = D.nz;
    const double lx = L.lx, ly = L.ly, lx2 = xmul(lx, lx), ly2 = xmul(ly, ly);
    const double2 one = cmk(1.0, 0.0), zero = cmk(0.0, 0.0);
    double2 p1[2] = {one, one}, q1[2] = {zero, zero}, p2[2] = {zero, zero};
    double2 q2[2] = {ivp2_init(D, L, B.ws), ivp2_init(D, L2, B.ws)};
    double2 sp1[2], sq1[2], sp2[2], sq2[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) sp1[m] = sq1[m] = sp2[m] = sq2[m] = zero;
    const int snap = D.snap_level[0];
    Row nxt = load_row(ctab);
#pragma unroll 2
    for (int i = 0; i < nz - 1; ++i) {
      if (!RECOMP && i == snap) {
#pragma unroll
        for (int m = 0; m < 2; ++m) { sp1[m] = p1[m]; sq1[m] = q1[m]; sp2[m] = p2[m]; sq2[m] = q2[m]; }
      }
      const Row cur = nxt;
      if (i + 1 < nz - 1) nxt = load_row(ctab + (int64_t)(i + 1) * BLDFM_LEVEL_STRIDE);
      march_pair(cur, lx, ly, lx2, ly2, p1, q1, p2, q2);
    }
    if (!RECOMP && nz - 1 == snap) {
#pragma unroll
      for (int m = 0; m < 2; ++m) { sp1[m] = p1[m]; sq1[m] = q1[m]; sp2[m] = p2[m]; sq2[m] = q2[m]; }
    }
    const double* tt = tab + (int64_t)(nz - 1) * BLDFM_LEVEL_STRIDE;
    double2 alpha[2], sh[2];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const Lane& M = m ? L2 : L;
      alpha[m] = shoot_alpha(tt, top_lambda(tt, M.lx, M.ly, lx2, ly2), p1[m], q1[m], p2[m], q2[m]);
      sh[m] = phase_shift(D, M);
    }
    if (!RECOMP) {
      if (D.nfilled > 0) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
          if (m == 0 || two)
            emit_mode(D, m ? L2 : L, B.ws, 0, xcadd(ncmul(alpha[m], sp1[m]), sp2[m]),
                      xcadd(ncmul(alpha[m], sq1[m]), sq2[m]), sh[m]);
      }
    } else {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        p1[m] = one; q1[m] = zero; p2[m] = zero;
        q2[m] = ivp2_init(D, m ? L2 : L, B.ws);
      }
      Row nxt2 = load_row(ctab);
      for (int i = 0; i <= D.max_level; ++i) {
        const int sl = slot[i];
        if (sl >= 0) {
#pragma unroll
          for (int m = 0; m < 2; ++m)
            if (m == 0 || two)
              emit_mode(D, m ? L2 : L, B.ws, sl, xcadd(ncmul(alpha[m], p1[m]), p2[m]),
                        xcadd(ncmul(alpha[m], q1[m]), q2[m]), sh[m]);
        }
        if (i < D.max_level) {
          const Row cur = nxt2;
          if (i + 1 < D.max_level) nxt2 = load_row(ctab + (int64_t)(i + 1) * BLDFM_LEVEL_STRIDE);
          march_pair(cur, lx, ly, lx2, ly2, p1, q1, p2, q2);
        }
      }
    }
    for (int s = D.nfilled; s < D.nslot; ++s)
#pragma unroll
      for (int m = 0; m < 2; ++m)
        if (m == 0 || two) emit_mode(D, m ? L2 : L, B.ws, s, zero, zero, sh[m]);
  }
}

// Analytic branch for constant profiles (src/bldfm/solver.py:193-202):
// q^ = q^0 e^{-lambda h}, p^ = (q^ / Kz) / lambda, p^00 = p000 - (q^00 / Kz) h.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_shoot_analytic(PlanDev P, ExecBufs B, int variant) {
#pragma clang fp contract(off)
  for (int64_t t = blockIdx.x; t < P.tot_shoot; t += gridDim.x) {
    const TileRec tr = tile_rec(P.t_shoot, t);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    if (D.variant != variant) continue;
    if (B.mode && B.mode[tr.inst] == 0) continue;
    Lane L;
    const int lane = tr.local * BLOCK + (int)threadIdx.x;
    if (!lane_setup(D, lane, L)) continue;
    const int nz = D.nz;
    const double* tt = B.tab + D.off_tab + (int64_t)(nz - 1) * BLDFM_LEVEL_STRIDE;
    const double kinv = tt[5];
    const double* z = B.prof + D.off_prof;
    const int32_t* lvidx = P.ints + D.off_slot + nz;
    if (L.kind == LANE_ORIGIN) {
      const double q00 = D.footprint ? D.q00 : B.ws[D.off_q0].x;
      for (int s = 0; s < D.nslot; ++s) {
        const double h = z[lvidx[s]] - z[0];
        emit_origin(D, B.ws, s, D.p000 - (q00 * kinv) * h, q00);
      }
      continue;
    }
    const double lx = L.lx, ly = L.ly;
    const double2 lam = top_lambda(tt, lx, ly, lx * lx, ly * ly);
    const double2 q0 = ivp2_init(D, L, B.ws);
    const double2 sh = phase_shift(D, L);
    for (int s = 0; s < D.nslot; ++s) {
      const double h = z[lvidx[s]] - z[0];
      double2 Xq = ncmul(q0, cexp_(cmk(-lam.x * h, -lam.y * h)));
      if (D.single) Xq = round_c64(Xq);
      const double2 Xp = cdiv(xcscale(kinv, Xq), lam);
      emit_mode(D, L, B.ws, s, Xp, Xq, sh);
    }
  }
}

// Hermitian part on the Nyquist row/column:
// Z(c) = (X(c) + conj X(-c))/2 packed as Hp + i Hq.
__global__ __launch_bounds__(256) void k_nyq_fix(PlanDev P, ExecBufs B) {
  for (int64_t t = blockIdx.x; t < P.tot_nyq; t += gridDim.x) {
    const TileRec tr = tile_rec(P.t_nyq, t);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    const int cnt = nyq_fix_count(D.nlx, D.nly, D.nxb, D.nyb);
    const int bps = (cnt + 255) / 256;
    const int local = tr.local;
    const int s = local / bps;
    const int p = (local % bps) * 256 + threadIdx.x;
    if (p >= cnt) continue;
    int cx, cy;
    nyq_fix_decode(p, D.nlx, D.nly, D.nxb, D.nyb, &cx, &cy);
    const int mx = compact_mirror(cx, D.nxb), my = compact_mirror(cy, D.nyb);
    const int n1 = nyq_index_at(cx, cy, D.nlx, D.nly, D.nxb, D.nyb);
    const int n2 = nyq_index_at(mx, my, D.nlx, D.nly, D.nxb, D.nyb);
    const double2* N = B.ws + D.off_nyq + (int64_t)s * (D.nlx + D.nly) * 2;
    double2 A = cmk(0.0, 0.0), Q = cmk(0.0, 0.0);
    if (n1 >= 0) { A = N[2 * n1]; Q = N[2 * n1 + 1]; }
    if (n2 >= 0) { A = cadd(A, cconj(N[2 * n2])); Q = cadd(Q, cconj(N[2 * n2 + 1])); }
    B.ws[D.off_z + ((int64_t)s * D.nxb + cx) * D.nyb + cy] = cmk(0.5 * (A.x - Q.y), 0.5 * (A.y + Q.x));
  }
}

// ---------------------------------------------------------------- point solver
// Level tables of nmet met samples for the point solver, `rows` rows per
// sample (rows >= the sample's level count).
__global__ __launch_bounds__(256) void k_tables_met(const ProfSetup* __restrict__ S, int nmet, int rows,
                                                    double* __restrict__ tab) {
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= (int64_t)nmet * rows) return;
  const int m = (int)(g / rows), i = (int)(g % rows);
  const ProfSetup& s = S[m];
  const int nz = s.nlev;
  if (i >= nz) return;
  double cur[6], nxt[6];
  prof_point(s, i, cur);
  if (i + 1 < nz) prof_point(s, i + 1, nxt);
  fill_level_row(cur, nxt, i == nz - 1, tab + g * BLDFM_LEVEL_STRIDE);
}

// Flux transfer G = q^(z_lvl) / q^(0) of single modes: the shooting solve
// of the footprint mode (both IVPs, radiation condition, shooting
// coefficient) for a unit surface flux.  Blocks of 256 points share one met
// sample (its table rows are uniform, read through scalar loads).  Invalid
// block metadata yields NaN instead of an out-of-range read.
template <bool EXACT>
__global__ __launch_bounds__(256) void k_transfer(const double* __restrict__ tab, int rows,
                                                  const int32_t* __restrict__ nzs,
                                                  const int32_t* __restrict__ lvls, int nmet,
                                                  const int32_t* __restrict__ blk_met, int nblk,
                                                  const double2* __restrict__ kxy, double2* __restrict__ g) {
  for (int b = blockIdx.x; b < nblk; b += gridDim.x) {
    const int64_t p = (int64_t)b * 256 + threadIdx.x;
    const int m = blk_met[b];
    const int nz = (m >= 0 && m < nmet) ? nzs[m] : 0;
    const int lvl = (m >= 0 && m < nmet) ? lvls[m] : -1;
    if (nz < 2 || nz > rows || lvl < 0 || lvl >= nz) {
      g[p] = cmk(__builtin_nan(""), __builtin_nan(""));
      continue;
    }
    const double* T = tab + (int64_t)m * rows * BLDFM_LEVEL_STRIDE;
    ctab_t* ct = (ctab_t*)T;
    const double2 k = kxy[p];
    const double lx = k.x, ly = k.y, lx2 = xmul(lx, lx), ly2 = xmul(ly, ly);
    double2 p1 = cmk(1.0, 0.0), q1 = cmk(0.0, 0.0), p2 = cmk(0.0, 0.0), q2 = cmk(1.0, 0.0);
    double2 sq1 = q1, sq2 = q2;
    Row nxt = load_row(ct);
    for (int i = 0; i < nz - 1; ++i) {
      if (i == lvl) { sq1 = q1; sq2 = q2; }
      const Row cur = nxt;
      if (i + 1 < nz - 1) nxt = load_row(ct + (int64_t)(i + 1) * BLDFM_LEVEL_STRIDE);
      march_step<EXACT>(cur, lx, ly, lx2, ly2, p1, q1, p2, q2);
    }
    if (lvl == nz - 1) { sq1 = q1; sq2 = q2; }
    const double* tt = T + (int64_t)(nz - 1) * BLDFM_LEVEL_STRIDE;
    const double2 alpha = shoot_alpha(tt, top_lambda(tt, lx, ly, lx2, ly2), p1, q1, p2, q2);
    g[p] = (lx == 0.0 && ly == 0.0) ? cmk(1.0, 0.0) : xcadd(ncmul(alpha, sq1), sq2);
  }
}

// ---------------------------------------------------------------- surrogate gate
// Per-instance gate state before the surrogate runs: sums cleared, accepted
// (mode 0) if flagged and inside the training hull, else solved (mode 1).
__global__ __launch_bounds__(256) void k_sur_clear(PlanDev P, ExecBufs B) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P.ninst) return;
  B.gate[i] = cmk(0.0, 0.0);
  B.mode[i] = P.sur_ok[i] ? 0 : 1;
}

// Spot check: every sur_stride-th lane of an accepted instance is solved in
// FP64 and compared with the surrogate's packed output X_q = -i Z(k).
template <bool EXACT>
__global__ __launch_bounds__(256) void k_sur_spot(PlanDev P, ExecBufs B) {
  __shared__ double sd[4], ss[4];
  for (int64_t t = blockIdx.x; t < P.tot_spot; t += gridDim.x) {
    const TileRec tr = tile_rec(P.t_spot, t);
    const int inst = tr.inst;
    const cdesc_t& D = *(const cdesc_t*)(P.desc + inst);
    if (B.mode[inst] != 0 || D.exact != (int)EXACT) continue;  // uniform over the workgroup
    const int off = (int)((inst * 61LL) % P.sur_stride);
    const int lane = off + (tr.local * 256 + (int)threadIdx.x) * P.sur_stride;
    double d2 = 0.0, s2 = 0.0;
    Lane L;
    if (lane_setup(D, lane, L) && L.kind == LANE_HALF) {
      const double* __restrict__ tab = B.tab + D.off_tab;
      ctab_t* __restrict__ ctab = (ctab_t*)tab;
      const int nz = D.nz, lvl = D.max_level;
      const double lx = L.lx, ly = L.ly, lx2 = xmul(lx, lx), ly2 = xmul(ly, ly);
      double2 p1 = cmk(1.0, 0.0), q1 = cmk(0.0, 0.0), p2 = cmk(0.0, 0.0), q2 = cmk(D.q00, 0.0);
      double2 sq1 = q1, sq2 = q2;
      Row nxt = load_row(ctab);
      for (int i = 0; i < nz - 1; ++i) {
        if (i == lvl) { sq1 = q1; sq2 = q2; }
        const Row cur = nxt;
        if (i + 1 < nz - 1) nxt = load_row(ctab + (int64_t)(i + 1) * BLDFM_LEVEL_STRIDE);
        march_step<EXACT>(cur, lx, ly, lx2, ly2, p1, q1, p2, q2);
      }
      if (lvl == nz - 1) { sq1 = q1; sq2 = q2; }
      const double* tt = tab + (int64_t)(nz - 1) * BLDFM_LEVEL_STRIDE;
      const double2 alpha = shoot_alpha(tt, top_lambda(tt, lx, ly, lx2, ly2), p1, q1, p2, q2);
      double2 xq = xcadd(ncmul(alpha, sq1), sq2);
      if (D.has_shift) xq = ncmul(xq, phase_shift(D, L));
      const int cx = compact_of_freq(L.fx, D.nxb), cy = compact_of_freq(L.fy, D.nyb);
      const double2 z = B.ws[D.off_z + (int64_t)cx * D.nyb + cy];
      const double er = z.y - xq.x, ei = -z.x - xq.y;
      d2 = er * er + ei * ei;
      s2 = xq.x * xq.x + xq.y * xq.y;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      d2 += __shfl_xor(d2, o);
      s2 += __shfl_xor(s2, o);
    }
    if ((threadIdx.x & 63) == 0) { sd[threadIdx.x >> 6] = d2; ss[threadIdx.x >> 6] = s2; }
    __syncthreads();
    if (threadIdx.x == 0) {
      atomicAdd(&B.gate[inst].x, sd[0] + sd[1] + sd[2] + sd[3]);
      atomicAdd(&B.gate[inst].y, ss[0] + ss[1] + ss[2] + ss[3]);
    }
    __syncthreads();
  }
}

// Gate decision: an accepted instance whose spot-check relative L2 error
// exceeds sur_tol (or is not finite) falls back to the FP64 solver.
__global__ __launch_bounds__(256) void k_sur_gate(PlanDev P, ExecBufs B) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= P.ninst || B.mode[i] != 0) return;
  const double2 s = B.gate[i];
  // no checked lane (or a zero reference) is no evidence: the solver serves it
  const double err = s.y > 0.0 ? sqrt(s.x / s.y) : INFINITY;
  if (!(err <= P.sur_tol)) B.mode[i] = 1;
}

// ---------------------------------------------------------------- KM01
// Kormann & Meixner (2001) analytic footprint on a regular grid
// (src/bldfm/ffm_kormann_meixner.py:110-330, Eqs. 9 and 21): one thread per
// cell, blockIdx.y = footprint.  Cell (j, i) sits at x = xmin + res/2 + i res,
// y = ymax - res/2 - j res (numpy arange order), is shifted to the receptor
// and, with a wind direction, rotated into the along/cross-wind frame.
__global__ __launch_bounds__(256) void k_km01(const Km01Dev* __restrict__ P, double* __restrict__ out) {
  const Km01Dev& D = P[blockIdx.y];
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c >= (int64_t)D.nx * D.ny) return;
  const int j = (int)(c / D.nx), i = (int)(c % D.nx);
  double x = (D.xmin + 0.5 * D.res + i * D.res) - D.mx;
  double y = (D.ymax - 0.5 * D.res - j * D.res) - D.my;
  if (D.has_wd) {
    const double rho = sqrt(x * x + y * y);
    const double th = atan2(y, x) + D.wd_rad - 0.5 * BLDFM_PI;
    x = rho * cos(th);
    y = rho * sin(th);
  }
  double f = 0.0;
  if (D.valid && x > 0.0) {
    const double g = D.gA * y * pow(x, D.e2);
    f = D.scale * pow(x, D.e1) * exp(-D.Xi / x - 0.5 * (g * g));
  }
  out[D.off + c] = f;
}

// x-pass layout 2: v[s][cx][y] -> vt[s][y][cx] in 32 x 32 tiles through LDS.
// Reads run along y and writes along cx, both coalesced; the padding column
// makes the transposed LDS reads (stride 33 x 16 bytes) conflict free.
__global__ __launch_bounds__(256) void k_transpose_v(PlanDev P, ExecBufs B) {
  __shared__ double2 tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int64_t b = blockIdx.x; b < P.tot_tr; b += gridDim.x) {
    const TileRec tr = tile_rec(P.t_tr, b);
    const cdesc_t& D = *(const cdesc_t*)(P.desc + tr.inst);
    const int tcx = (D.nxb + 31) >> 5, tcy = (D.ny + 31) >> 5;
    const int s = tr.local / (tcx * tcy), r = tr.local % (tcx * tcy);
    const int cx0 = (r / tcy) * 32, y0 = (r % tcy) * 32;
    const double2* src = B.ws + D.off_v + (int64_t)s * D.nxb * D.ny;
    double2* dst = B.ws + D.off_vt + (int64_t)s * D.ny * D.nxb;
    if (b != blockIdx.x) __syncthreads();  // the previous tile's reads of `tile` are done
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int cx = cx0 + ty + 8 * k, y = y0 + tx;
      if (cx < D.nxb && y < D.ny) tile[ty + 8 * k][tx] = src[(int64_t)cx * D.ny + y];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int y = y0 + ty + 8 * k, cx = cx0 + tx;
      if (cx < D.nxb && y < D.ny) dst[(int64_t)y * D.nxb + cx] = tile[tx][ty + 8 * k];
    }
  }
}

// ---------------------------------------------------------------- launcher
int bldfm_launch_lines(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int pass, int grid_cap, hipStream_t stream) {
  switch (pass) {
    case PASS_FWD_ROWS: return bldfm_lines_pass0(P, L, B, grid_cap, stream, 0);
    case PASS_FWD_COLS: return bldfm_lines_pass1(P, L, B, grid_cap, stream, 0);
    case PASS_INV_COLS: return bldfm_lines_pass2(P, L, B, grid_cap, stream, 0);
    default: return bldfm_lines_pass3(P, L, B, grid_cap, stream, 0);
  }
}

int bldfm_launch_all(const PlanDev& P, const LinePlan& L, const ExecBufs& B, int grid_cap, hipStream_t stream,
                     hipEvent_t* ev) {
#define MARK(k)                                            \
  if (ev) {                                                \
    if (hipEventRecord(ev[k], stream) != hipSuccess) return -1999; \
  }
  MARK(0)
  if (P.tot_tab > 0) {
    k_level_table<<<grid_for(P.tot_tab, grid_cap), 1024, 0, stream>>>(P, B);
    LAUNCH_CHECK();
  }
  MARK(1)
  // chirp lines of a pass, then single-workgroup lines, then split (four-step) lines
#define FFT_LAUNCH(PASS, tiles)                                                     \
  {                                                                                 \
    int rc_ = bldfm_launch_lines(P, L, B, PASS, grid_cap, stream);                  \
    if (!rc_ && (tiles) > 0) rc_ = bldfm_launch_pass(P, B, PASS, tiles, grid_cap, stream); \
    if (!rc_) rc_ = bldfm_launch_long(P, B, PASS, grid_cap, stream);                \
    if (rc_) return rc_;                                                            \
  }
  if (P.any_dispersion) {
    FFT_LAUNCH(PASS_FWD_ROWS, P.tot_fwd_rows)
    FFT_LAUNCH(PASS_FWD_COLS, P.tot_fwd_cols)
  }
  MARK(2)
  const bool sur = P.sur_net != nullptr && B.mode != nullptr && P.tot_sur > 0;
  if (sur) {
    const unsigned gi = (unsigned)((P.ninst + 255) / 256);
    k_sur_clear<<<gi, 256, 0, stream>>>(P, B);
    LAUNCH_CHECK();
    const int rc = bldfm_launch_sur_plan(P, B, grid_cap, stream);
    if (rc) return rc;
    if (P.tot_spot > 0) {
      // a launch over instances of the other rounding alone costs 4.6 us
      bool used[2] = {false, false};  // fused, exact
      for (int v = 0; v < 4; ++v) {
        used[0] |= P.variant_used[v][0] != 0;
        used[1] |= P.variant_used[v][1] || P.pair_used[v];
      }
      if (used[1]) k_sur_spot<true><<<grid_for(P.tot_spot, grid_cap), 256, 0, stream>>>(P, B);
      LAUNCH_CHECK();
      if (used[0]) k_sur_spot<false><<<grid_for(P.tot_spot, grid_cap), 256, 0, stream>>>(P, B);
      LAUNCH_CHECK();
    }
    k_sur_gate<<<gi, 256, 0, stream>>>(P, B);
    LAUNCH_CHECK();
  }
  MARK(3)
  const unsigned gs = grid_for(P.tot_shoot, grid_cap);
#define SHOOT(V, MAXS, RECOMP, EX)                                                           \
  if (P.variant_used[V][EX]) {                                                               \
    if (P.shoot_block == 64) k_shoot<MAXS, RECOMP, EX, 64><<<gs, 64, 0, stream>>>(P, B, V);     \
    else if (P.shoot_block == 128) k_shoot<MAXS, RECOMP, EX, 128><<<gs, 128, 0, stream>>>(P, B, V); \
    else k_shoot<MAXS, RECOMP, EX, 256><<<gs, 256, 0, stream>>>(P, B, V);                     \
    LAUNCH_CHECK();                                                                          \
  }
  SHOOT(0, 1, false, true)
  SHOOT(1, 4, false, true)
  SHOOT(2, 1, true, true)
  SHOOT(0, 1, false, false)
  SHOOT(1, 4, false, false)
  SHOOT(2, 1, true, false)
#undef SHOOT
#define SHOOT_PAIR(V, RECOMP)                                                             \
  if (P.pair_used[V]) {                                                                   \
    if (P.shoot_block == 64) k_shoot_pair<RECOMP, 64><<<gs, 64, 0, stream>>>(P, B, V);    \
    else if (P.shoot_block == 128) k_shoot_pair<RECOMP, 128><<<gs, 128, 0, stream>>>(P, B, V); \
    else k_shoot_pair<RECOMP, 256><<<gs, 256, 0, stream>>>(P, B, V);                      \
    LAUNCH_CHECK();                                                                       \
  }
  SHOOT_PAIR(0, false)
  SHOOT_PAIR(2, true)
#undef SHOOT_PAIR
  if (P.variant_used[3][0] || P.variant_used[3][1]) {
    if (P.shoot_block == 64) k_shoot_analytic<64><<<gs, 64, 0, stream>>>(P, B, 3);
    else if (P.shoot_block == 128) k_shoot_analytic<128><<<gs, 128, 0, stream>>>(P, B, 3);
    else k_shoot_analytic<256><<<gs, 256, 0, stream>>>(P, B, 3);
    LAUNCH_CHECK();
  }
  MARK(4)
  if (P.tot_nyq > 0) {
    k_nyq_fix<<<grid_for(P.tot_nyq, grid_cap), 256, 0, stream>>>(P, B);
    LAUNCH_CHECK();
  }
  MARK(5)
  FFT_LAUNCH(PASS_INV_COLS, P.tot_inv_cols)
  MARK(6)
  if (P.xlayout == 2 && P.tot_tr > 0) {
    k_transpose_v<<<grid_for(P.tot_tr, grid_cap), 256, 0, stream>>>(P, B);
    LAUNCH_CHECK();
  }
  FFT_LAUNCH(PASS_INV_ROWS, P.tot_inv_rows)
  MARK(7)
#undef FFT_LAUNCH
#undef MARK
  return 0;
}

// ---------------------------------------------------------------- profiles
// Array part of vertical_profiles (src/bldfm/pbl_model.py:127-182):
// out = [z | u | v | Kx | Ky | Kz], nlev each.
__global__ __launch_bounds__(1024) void k_profiles(ProfSetup S, double* __restrict__ out) {
  __shared__ double sh[7][256];
  const int i = blockIdx.x * 256 + group_slot().tid;
  double o[6];
  prof_group(S, i, i < S.nlev, sh, o);
  if (group_slot().grp == 0 && i < S.nlev)
    for (int c = 0; c < 6; ++c) out[(int64_t)c * S.nlev + i] = o[c];
}

int bldfm_launch_profiles(const ProfSetup& S, double* out, hipStream_t stream) {
  // one group where the closure has no chains to share out: 5.2 and 7.2 us (CONSTANT,
  // OAAHOC) instead of 5.7 and 7.7 with four
  const bool most = S.closure == CL_MOST || S.closure == CL_MOSTM;
  k_profiles<<<(S.nlev + 255) / 256, most ? 1024 : 256, 0, stream>>>(S, out);
  LAUNCH_CHECK();
  return 0;
}

// Allow dynamic LDS beyond the default per-workgroup cap for the FFT kernels.
void bldfm_set_line_lds_attr(int bytes) {
  const PlanDev P{};
  const LinePlan L{};
  const ExecBufs B{};
  (void)bldfm_lines_pass0(P, L, B, 0, nullptr, bytes);
  (void)bldfm_lines_pass1(P, L, B, 0, nullptr, bytes);
  (void)bldfm_lines_pass2(P, L, B, 0, nullptr, bytes);
  (void)bldfm_lines_pass3(P, L, B, 0, nullptr, bytes);
}

void bldfm_set_fft_lds_attr(int bytes) {
  bldfm_pass_lds_attr(bytes);
  bldfm_long_lds_attr(bytes);
  bldfm_fft2_lds_attr(bytes);
}

// ---------------------------------------------------------------- elementwise
// psi(x), phi(x) of MOST (src/bldfm/pbl_model.py:207-250).
__global__ __launch_bounds__(256) void k_stability(const double* __restrict__ x, int64_t n,
                                                   double* __restrict__ psi, double* __restrict__ phi) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double v = x[i];
    if (psi) psi[i] = most_psi(v);
    if (phi) phi[i] = most_phi(v);
  }
}

// Met wind (speed, direction blowing FROM, degrees) -> (u, v)
// (src/bldfm/utils.py:23-27): u = -U sin(theta), v = -U cos(theta).
__global__ __launch_bounds__(256) void k_wind(const double* __restrict__ spd, const double* __restrict__ dir,
                                              int64_t n, double* __restrict__ u, double* __restrict__ v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    wind_uv(spd[i], dir[i], &u[i], &v[i]);
  }
}

int bldfm_launch_stability(const double* x, int64_t n, double* psi, double* phi, hipStream_t stream) {
  if (n <= 0) return 0;
  k_stability<<<grid_for((n + 255) / 256, 4096), 256, 0, stream>>>(x, n, psi, phi);
  LAUNCH_CHECK();
  return 0;
}

int bldfm_launch_wind(const double* spd, const double* dir, int64_t n, double* u, double* v, hipStream_t stream) {
  if (n <= 0) return 0;
  k_wind<<<grid_for((n + 255) / 256, 4096), 256, 0, stream>>>(spd, dir, n, u, v);
  LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------- math probe
// Evaluates the device math helpers on n inputs for bitwise checks:
// op 0 hypot_borges(a, b); op 1 csqrt_exact(a + ib) -> (out[2i], out[2i+1]);
// op 2 cdiv((a0 + i a1), (b0 + i b1)) with a, b holding complex pairs;
// op 3 ncmul of complex pairs; op 4 xcmul of complex pairs; op 5 sqrt(a).
__global__ __launch_bounds__(256) void k_math_probe(int op, const double* __restrict__ a,
                                                    const double* __restrict__ b, int64_t n,
                                                    double* __restrict__ out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    if (op == 0) {
      out[i] = hypot_borges(a[i], b[i]);
    } else if (op == 1) {
      const double2 r = csqrt_exact(cmk(a[i], b[i]));
      out[2 * i] = r.x;
      out[2 * i + 1] = r.y;
    } else if (op == 5) {
      out[i] = sqrt(a[i]);
    } else {
      const double2 x = cmk(a[2 * i], a[2 * i + 1]), y = cmk(b[2 * i], b[2 * i + 1]);
      const double2 r = op == 2 ? cdiv(x, y) : (op == 3 ? ncmul(x, y) : xcmul(x, y));
      out[2 * i] = r.x;
      out[2 * i + 1] = r.y;
    }
  }
}

int bldfm_launch_math_probe(int op, const double* a, const double* b, int64_t n, double* out, hipStream_t stream) {
  if (n <= 0) return 0;
  k_math_probe<<<grid_for((n + 255) / 256, 4096), 256, 0, stream>>>(op, a, b, n, out);
  LAUNCH_CHECK();
  return 0;
}

int bldfm_launch_tables(const ProfSetup* S, int nmet, int rows, double* tab, hipStream_t stream) {
  const int64_t n = (int64_t)nmet * rows;
  k_tables_met<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(S, nmet, rows, tab);
  LAUNCH_CHECK();
  return 0;
}

int bldfm_launch_transfer(const double* tab, int rows, const int32_t* nzs, const int32_t* lvls, int nmet,
                          const int32_t* blk_met, int nblk, const double2* kxy, double2* g, int exact,
                          hipStream_t stream) {
  const unsigned grid = (unsigned)(nblk < (1 << 20) ? nblk : (1 << 20));
  if (exact)
    k_transfer<true><<<grid, 256, 0, stream>>>(tab, rows, nzs, lvls, nmet, blk_met, nblk, kxy, g);
  else
    k_transfer<false><<<grid, 256, 0, stream>>>(tab, rows, nzs, lvls, nmet, blk_met, nblk, kxy, g);
  LAUNCH_CHECK();
  return 0;
}

int bldfm_launch_km01(const Km01Dev* P, int n, int64_t max_cells, double* out, hipStream_t stream) {
  if (n <= 0 || max_cells <= 0) return 0;
  dim3 grid((unsigned)((max_cells + 255) / 256), (unsigned)n);
  k_km01<<<grid, 256, 0, stream>>>(P, out);
  LAUNCH_CHECK();
  return 0;
}
