#pragma once
#include <type_traits>

#include "bldfm_passes.h"

// ---------------------------------------------------------------- plain 2-D FFT
// numpy fft2/ifft2 on `batch` contiguous (n0, n1) complex arrays: x-pass
// over the rows into the workspace, then y-pass over the columns, output
// multiplied by `scale`.
//
// T is the caller's element, double2 or float2: complex64 fields are widened by
// the first pass's loads and rounded by the last one's stores, the arithmetic and
// the field between the passes stay FP64.  Converting whole fields before and
// after cost 76 us of the 180 of a 4 x 1001 x 1386 inverse (95 without).
__device__ __forceinline__ double2 widen(double2 v) { return v; }
__device__ __forceinline__ double2 widen(float2 v) { return cmk(v.x, v.y); }
__device__ __forceinline__ void store_as(double2* p, double2 v) { *p = v; }
__device__ __forceinline__ void store_as(float2* p, double2 v) { *p = make_float2((float)v.x, (float)v.y); }

template <class T>
struct StridedIn {
  const T* __restrict__ src;
  int64_t stride;
  __device__ __forceinline__ double2 operator()(int i) const { return widen(src[(int64_t)i * stride]); }
};
template <class T>
struct StridedOut {
  T* __restrict__ dst;
  int64_t stride;
  double scale;
  __device__ __forceinline__ void operator()(int o, double2 v) const { store_as(dst + (int64_t)o * stride, cscale(scale, v)); }
};

// PRIMES: with the butterflies of 7, 11 and 13, for lengths that have such a
// factor.  They take 109 to 116 registers, the others' kernels 81 to 103; where
// every length ran them, a small field took longer than it does without:
// 48 x 64 replayed from a graph 8.5 us against 8.0, 60 x 100 9.5 against 8.3,
// 512 x 512 14.1 against 13.2.
inline bool fft2_primes(int n) { return n % 7 == 0 || n % 11 == 0 || n % 13 == 0; }

// How they take their twiddles, by the caller's element.
template <bool PRIMES, class E>
constexpr bldfm_fft::Primes prime_mode() {
  return !PRIMES ? bldfm_fft::PRIME_NONE : sizeof(E) == sizeof(double2) ? bldfm_fft::PRIME_LOOKUP : bldfm_fft::PRIME_POWERS;
}

template <int MAXE, bldfm_fft::Primes PRIMES, class In, class Out>
__device__ __forceinline__ void fft_plain(bool inv, const FftPlan* F, int n, const double2* __restrict__ tw, int tid,
                                          int T, In in, Out out, bool reuse) {
  const bldfm_fft::Lds buf = bldfm_fft::lds_view(smem, n);
  if (inv) bldfm_fft::lds_fft<MAXE, true, PRIMES>(buf, smem + n, F, tw, tid, T, in, out, reuse);
  else bldfm_fft::lds_fft<MAXE, false, PRIMES>(buf, smem + n, F, tw, tid, T, in, out, reuse);
}

template <int MAXE, int MAXT, bool PRIMES, class E>
__global__ __launch_bounds__(MAXT) void k_fft2_rows(const FftPlan* F, const double2* __restrict__ tw,
                                                  const E* __restrict__ in, double2* __restrict__ mid,
                                                  int32_t n, int64_t nrows, bool inv) {
  const int T = blockDim.x, tid = threadIdx.x;
  for (int64_t r = blockIdx.x; r < nrows; r += gridDim.x)
    fft_plain<MAXE, prime_mode<PRIMES, E>()>(inv, F, n, tw, tid, T, StridedIn<E>{in + r * n, 1}, StridedOut<double2>{mid + r * n, 1, 1.0},
                    r != blockIdx.x);
}

template <int MAXE, int MAXT, bool PRIMES, class E>
__global__ __launch_bounds__(MAXT) void k_fft2_cols(const FftPlan* F, const double2* __restrict__ tw,
                                                  const double2* __restrict__ mid, E* __restrict__ out,
                                                  int32_t n0, int32_t n1, int64_t ncols, double scale, bool inv) {
  const int T = blockDim.x, tid = threadIdx.x;
  for (int64_t w = blockIdx.x; w < ncols; w += gridDim.x) {
    // eight neighbouring columns share every 128-byte line: each XCD takes a
    // contiguous range of them, so a line is fetched into one L2 and not into
    // eight (both passes of 2 x 2048^2 complex128, before its
    // columns ran in tiles: 302 -> 212 us)
    const int64_t c = gridDim.x >= ncols ? xcd_swizzle(w, ncols) : w;
    const int64_t b = c / n1, col = c % n1;
    const int64_t o = b * (int64_t)n0 * n1 + col;
    fft_plain<MAXE, prime_mode<PRIMES, E>()>(inv, F, n0, tw, tid, T, StridedIn<double2>{mid + o, n1}, StridedOut<E>{out + o, n1, scale},
                    w != blockIdx.x);
  }
}

// C neighbouring columns per workgroup (ncols rounded up to tiles of C within
// an array): neighbouring lanes hold neighbouring columns, so loads and stores
// move C * 16 consecutive bytes.  One column per workgroup wrote 2.6 times the
// result's bytes (16-byte pieces of lines that left the L2 before the seven
// other columns came).  2 x 2048^2, both passes: 212 -> 134 us; 4 x 1024^2: 156 -> 70.
struct TileIn {
  const double2* __restrict__ src;
  int64_t stride;
  bool live;
  __device__ __forceinline__ double2 operator()(int i) const { return live ? src[(int64_t)i * stride] : cmk(0.0, 0.0); }
};
template <class E>
struct TileOut {
  E* __restrict__ dst;
  int64_t stride;
  double scale;
  bool live;
  __device__ __forceinline__ void operator()(int o, double2 v) const {
    if (live) store_as(dst + (int64_t)o * stride, cscale(scale, v));
  }
};
template <int C, bool PRIMES, class E>
__global__ __launch_bounds__(1024) void k_fft2_col_tiles(const FftPlan* F, const double2* __restrict__ tw,
                                                       const double2* __restrict__ mid, E* __restrict__ out,
                                                       int32_t n0, int32_t n1, int64_t ntiles, double scale, bool inv) {
  const int c = (int)threadIdx.x % C, t = (int)threadIdx.x / C, T = (int)blockDim.x / C;
  const int per = (n1 + C - 1) / C;
  for (int64_t w = blockIdx.x; w < ntiles; w += gridDim.x) {
    const int64_t tile = gridDim.x >= ntiles ? xcd_swizzle(w, ntiles) : w;
    const int64_t b = tile / per;
    const int col = (int)(tile % per) * C + c;
    const int64_t o = b * (int64_t)n0 * n1 + col;
    const bool live = col < n1;
    const bldfm_fft::LdsT<C> buf = bldfm_fft::lds_view<C>(smem + c, n0);
    const TileIn in{mid + o, n1, live};
    const TileOut<E> dst{out + o, n1, scale, live};
    if (inv) bldfm_fft::lds_fft<FFT_SMALL_E, true, prime_mode<PRIMES, E>()>(buf, smem + n0 * C, F, tw, t, T, in, dst, w != blockIdx.x);
    else bldfm_fft::lds_fft<FFT_SMALL_E, false, prime_mode<PRIMES, E>()>(buf, smem + n0 * C, F, tw, t, T, in, dst, w != blockIdx.x);
  }
}

// Split (four-step) lines of the plain 2-D FFT: `rows` selects the rows of
// the (n0, n1) arrays (line r at r*n1, stride 1), else their columns (line c
// at (c / n1)*n0*n1 + c % n1, stride n1); scr holds nlines x n values.
// E is the element of `in` in step A and of `out` in step B.
template <int MAXE, int MAXT, bool STEPB, class E>
__global__ __launch_bounds__(MAXT) void k_fft2_long(FftSplit S, const E* __restrict__ in,
                                                  E* __restrict__ out, double2* __restrict__ scr, int rows,
                                                  int32_t n0, int32_t n1, int64_t nlines, double scale, bool inv) {
  const int T = blockDim.x, tid = threadIdx.x;
  const int n = S.F->n, s1 = S.F->n1, s2 = S.F->n2;
  const int64_t per = STEPB ? s1 : s2;
  for (int64_t b = blockIdx.x; b < nlines * per; b += gridDim.x) {
    const int64_t line = b / per;
    const int sub = (int)(b % per);
    const int64_t base = rows ? line * n1 : (line / n1) * (int64_t)n0 * n1 + line % n1;
    const int64_t stride = rows ? 1 : n1;
    double2* sc = scr + line * n;
    const bldfm_fft::Lds buf0 = bldfm_fft::lds_view(smem, STEPB ? s2 : s1);
    if constexpr (!STEPB) {
      const SubIn<StridedIn<E>> src{StridedIn<E>{in + base, stride}, s2, sub};
      const TwiddleOut dst{sc + (int64_t)sub * s1, S.tw, sub, inv};
      if (inv) bldfm_fft::lds_fft<MAXE, true>(buf0, smem + (STEPB ? s2 : s1), S.F1, S.tw1, tid, T, src, dst, b != blockIdx.x);
      else bldfm_fft::lds_fft<MAXE, false>(buf0, smem + (STEPB ? s2 : s1), S.F1, S.tw1, tid, T, src, dst, b != blockIdx.x);
    } else {
      const ScrIn src{sc + sub, s1};
      const SubOut<StridedOut<E>> dst{StridedOut<E>{out + base, stride, scale}, s1, sub};
      if (inv) bldfm_fft::lds_fft<MAXE, true>(buf0, smem + (STEPB ? s2 : s1), S.F2, S.tw2, tid, T, src, dst, b != blockIdx.x);
      else bldfm_fft::lds_fft<MAXE, false>(buf0, smem + (STEPB ? s2 : s1), S.F2, S.tw2, tid, T, src, dst, b != blockIdx.x);
    }
  }
}

template <class E>
int launch_fft2(const FftSplit& A0, int32_t n0, const FftSplit& A1, int32_t n1, int32_t batch,
                       const E* in, double2* mid, double2* scr, E* out, int32_t sign, double scale,
                       int threads, int lds_bytes, int grid_cap, hipStream_t stream) {
  const bool inv = sign > 0;
  const int64_t nrows = (int64_t)batch * n0, ncols = (int64_t)batch * n1;
  // kernel family by the longest LDS transform (a split axis runs its two
  // factors): the 256-thread kernels hold 8 values per thread, so they take
  // lengths up to BLDFM_FFT_SMALL_N; a longer transform may still run on 256
  // threads (10 values each) in the other family
  auto lds_n = [](const FftSplit& A, int32_t n) { return A.F1 ? (A.n1 > A.n2 ? A.n1 : A.n2) : n; };
  const int nmax = lds_n(A0, n0) > lds_n(A1, n1) ? lds_n(A0, n0) : lds_n(A1, n1);
  const bool small = nmax <= BLDFM_FFT_SMALL_N;
  if ((small && threads > 256) || threads > 1024 ||
      (int64_t)threads * (small ? FFT_SMALL_E : BLDFM_FFT_MAXE) < nmax)
    return -1000 - (int)hipErrorInvalidConfiguration;
  // a one-workgroup pass, its kernel by whether the length has a prime butterfly
  auto by_primes = [](int n, auto launch) { fft2_primes(n) ? launch(std::true_type()) : launch(std::false_type()); };
  // rows (axis 1, length n1): in -> mid
  if (A1.F1) {
    const unsigned ga = grid_for(nrows * A1.n2, grid_cap), gb = grid_for(nrows * A1.n1, grid_cap);
    if (small) {
      k_fft2_long<FFT_SMALL_E, 256, false, E><<<ga, threads, lds_bytes, stream>>>(A1, in, nullptr, scr, 1, n0, n1, nrows, 1.0, inv);
      LAUNCH_CHECK();
      k_fft2_long<FFT_SMALL_E, 256, true, double2><<<gb, threads, lds_bytes, stream>>>(A1, nullptr, mid, scr, 1, n0, n1, nrows, 1.0, inv);
    } else {
      k_fft2_long<BLDFM_FFT_MAXE, 1024, false, E><<<ga, threads, lds_bytes, stream>>>(A1, in, nullptr, scr, 1, n0, n1, nrows, 1.0, inv);
      LAUNCH_CHECK();
      k_fft2_long<BLDFM_FFT_MAXE, 1024, true, double2><<<gb, threads, lds_bytes, stream>>>(A1, nullptr, mid, scr, 1, n0, n1, nrows, 1.0, inv);
    }
  } else {
    by_primes(n1, [&](auto pr) {
      const unsigned g = grid_for(nrows, grid_cap);
      if (small) k_fft2_rows<FFT_SMALL_E, 256, pr, E><<<g, threads, lds_bytes, stream>>>(A1.F, A1.tw, in, mid, n1, nrows, inv);
      else k_fft2_rows<BLDFM_FFT_MAXE, 1024, pr, E><<<g, threads, lds_bytes, stream>>>(A1.F, A1.tw, in, mid, n1, nrows, inv);
    });
  }
  LAUNCH_CHECK();
  // columns (axis 0, length n0): mid -> out, scaled
  if (A0.F1) {
    const unsigned ga = grid_for(ncols * A0.n2, grid_cap), gb = grid_for(ncols * A0.n1, grid_cap);
    if (small) {
      k_fft2_long<FFT_SMALL_E, 256, false, double2><<<ga, threads, lds_bytes, stream>>>(A0, mid, nullptr, scr, 0, n0, n1, ncols, 1.0, inv);
      LAUNCH_CHECK();
      k_fft2_long<FFT_SMALL_E, 256, true, E><<<gb, threads, lds_bytes, stream>>>(A0, nullptr, out, scr, 0, n0, n1, ncols, scale, inv);
    } else {
      k_fft2_long<BLDFM_FFT_MAXE, 1024, false, double2><<<ga, threads, lds_bytes, stream>>>(A0, mid, nullptr, scr, 0, n0, n1, ncols, 1.0, inv);
      LAUNCH_CHECK();
      k_fft2_long<BLDFM_FFT_MAXE, 1024, true, E><<<gb, threads, lds_bytes, stream>>>(A0, nullptr, out, scr, 0, n0, n1, ncols, scale, inv);
    }
  } else if (fft2_tile(n0, n1, batch)) {
    const int c = fft2_tile(n0, n1, batch);
    const int64_t tiles = (int64_t)batch * ((n1 + c - 1) / c);
    const int t = (n0 + FFT_SMALL_E - 1) / FFT_SMALL_E;                     // lanes of a column
    const unsigned nt = (unsigned)((t * c + 63) / 64 * 64);
    const size_t lds = ((size_t)n0 * c + tw_table_len(n0)) * 16;
    by_primes(n0, [&](auto pr) {
      const unsigned g = grid_for(tiles, grid_cap);
      if (c == 8) k_fft2_col_tiles<8, pr, E><<<g, nt, lds, stream>>>(A0.F, A0.tw, mid, out, n0, n1, tiles, scale, inv);
      else k_fft2_col_tiles<4, pr, E><<<g, nt, lds, stream>>>(A0.F, A0.tw, mid, out, n0, n1, tiles, scale, inv);
    });
  } else {
    by_primes(n0, [&](auto pr) {
      const unsigned g = grid_for(ncols, grid_cap);
      if (small) k_fft2_cols<FFT_SMALL_E, 256, pr, E><<<g, threads, lds_bytes, stream>>>(A0.F, A0.tw, mid, out, n0, n1, ncols, scale, inv);
      else k_fft2_cols<BLDFM_FFT_MAXE, 1024, pr, E><<<g, threads, lds_bytes, stream>>>(A0.F, A0.tw, mid, out, n0, n1, ncols, scale, inv);
    });
  }
  LAUNCH_CHECK();
  return 0;
}

template <bool PRIMES, class E>
void fft2_lds_attr_of(int bytes) {
  const void* fns[] = {
      (const void*)k_fft2_rows<FFT_SMALL_E, 256, PRIMES, E>, (const void*)k_fft2_rows<BLDFM_FFT_MAXE, 1024, PRIMES, E>,
      (const void*)k_fft2_cols<FFT_SMALL_E, 256, PRIMES, E>, (const void*)k_fft2_cols<BLDFM_FFT_MAXE, 1024, PRIMES, E>,
      (const void*)k_fft2_col_tiles<4, PRIMES, E>, (const void*)k_fft2_col_tiles<8, PRIMES, E>};
  for (const void* f : fns) (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <class E>
void fft2_lds_attr(int bytes) {
  const void* fns[] = {
      (const void*)k_fft2_long<FFT_SMALL_E, 256, false, E>, (const void*)k_fft2_long<FFT_SMALL_E, 256, true, E>,
      (const void*)k_fft2_long<BLDFM_FFT_MAXE, 1024, false, E>, (const void*)k_fft2_long<BLDFM_FFT_MAXE, 1024, true, E>};
  for (const void* f : fns) (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  fft2_lds_attr_of<false, E>(bytes);
  fft2_lds_attr_of<true, E>(bytes);
}
