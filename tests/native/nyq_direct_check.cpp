// Direct emission of the unpaired Nyquist modes: with D.nyq_direct every
// position of the packed band is written exactly once by the shooting lanes
// (paired modes, Nyquist modes with their mirrors, the origin with the two
// corners) and holds what the Hermitian fix-up writes there.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../bldfm_amd/csrc/bldfm_types.h"

#define CHECK(c, ...) do { if (!(c)) { printf(__VA_ARGS__); printf("\n"); exit(1); } } while (0)

struct C { double re, im; };

int main() {
  int cases = 0, direct = 0;
  const int nls[] = {1, 2, 3, 4, 6, 7, 8, 16, 32};
  for (int nlx : nls) for (int nly : nls) for (int ex = 0; ex <= 3; ++ex) for (int ey = 0; ey <= 3; ++ey) {
    const int nxb = band_len(nlx, nlx + ex), nyb = band_len(nly, nly + ey);
    ++cases;
    // an unretained mirror of every Nyquist mode is what the rule claims
    bool none = true;
    const int lanes = shoot_lanes(nlx, nly);
    for (int lane = 0; lane < lanes; ++lane) {
      int fx = 0, fy = 0, nidx = -1;
      const int kind = decode_lane(lane, nlx, nly, &fx, &fy, &nidx);
      if (kind == LANE_ORIGIN) CHECK(lane == origin_lane(nlx, nly), "origin lane %d", lane);
      if (kind != LANE_NYQ) continue;
      const int cx = compact_of_freq(fx, nxb), cy = compact_of_freq(fy, nyb);
      if (nyq_index_at(compact_mirror(cx, nxb), compact_mirror(cy, nyb), nlx, nly, nxb, nyb) >= 0) none = false;
    }
    const bool d = nyq_is_direct(nlx, nly, nxb, nyb);
    CHECK(!d || none, "direct but a mirror is retained: %d %d %d %d", nlx, nly, nxb, nyb);
    if (!d) continue;
    ++direct;
    std::vector<int> cnt((size_t)nxb * nyb, 0);
    std::vector<C> Z((size_t)nxb * nyb, C{-1, -1}), N(2 * (size_t)(nlx + nly));
    for (int lane = 0; lane < lanes; ++lane) {
      int fx = 0, fy = 0, nidx = -1;
      const int kind = decode_lane(lane, nlx, nly, &fx, &fy, &nidx);
      if (kind == LANE_IDLE) continue;
      if (kind == LANE_ORIGIN) {
        cnt[0]++;
        if (nxb > nlx && nyb > nly) {
          const size_t a = (size_t)(nlx / 2) * nyb + compact_of_freq(-nly / 2, nyb);
          const size_t b = (size_t)compact_of_freq(-nlx / 2, nxb) * nyb + nly / 2;
          cnt[a]++; cnt[b]++;
          Z[a] = Z[b] = C{0, 0};
        }
        continue;
      }
      const C p{1.0 + lane, 0.25 * lane - 3.0}, q{0.5 * lane + 2.0, 7.0 - lane};
      const int cx = compact_of_freq(fx, nxb), cy = compact_of_freq(fy, nyb);
      const int mx = compact_mirror(cx, nxb), my = compact_mirror(cy, nyb);
      const double f = kind == LANE_HALF ? 1.0 : 0.5;
      const size_t a = (size_t)cx * nyb + cy, b = (size_t)mx * nyb + my;
      CHECK(a != b, "mode is its own mirror");
      cnt[a]++; cnt[b]++;
      Z[a] = C{f * (p.re - q.im), f * (p.im + q.re)};
      Z[b] = C{f * (p.re + q.im), f * (q.re - p.im)};
      if (kind == LANE_NYQ) { N[2 * nidx] = p; N[2 * nidx + 1] = q; }
    }
    for (int v : cnt) CHECK(v == 1, "band position written %d times (%d %d %d %d)", v, nlx, nly, nxb, nyb);
    for (int pfix = 0; pfix < nyq_fix_count(nlx, nly, nxb, nyb); ++pfix) {
      int cx, cy;
      nyq_fix_decode(pfix, nlx, nly, nxb, nyb, &cx, &cy);
      const int n1 = nyq_index_at(cx, cy, nlx, nly, nxb, nyb);
      const int n2 = nyq_index_at(compact_mirror(cx, nxb), compact_mirror(cy, nyb), nlx, nly, nxb, nyb);
      C A{0, 0}, Q{0, 0};
      if (n1 >= 0) { A = N[2 * n1]; Q = N[2 * n1 + 1]; }
      if (n2 >= 0) { A.re += N[2 * n2].re; A.im -= N[2 * n2].im; Q.re += N[2 * n2 + 1].re; Q.im -= N[2 * n2 + 1].im; }
      const C want{0.5 * (A.re - Q.im), 0.5 * (A.im + Q.re)}, got = Z[(size_t)cx * nyb + cy];
      CHECK(want.re == got.re && want.im == got.im, "fix-up differs at (%d,%d)", cx, cy);
    }
  }
  printf("%d shapes, %d direct\n", cases, direct);
  return 0;
}
