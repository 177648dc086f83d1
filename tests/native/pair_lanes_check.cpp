// Pair lanes of the march: every mode that decode_lane gives, exactly once,
// with the same kind and Nyquist index; the origin where pair_origin_lane says.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <utility>

#include "../../bldfm_amd/csrc/bldfm_types.h"

#define CHECK(c, ...) do { if (!(c)) { printf(__VA_ARGS__); printf("\n"); exit(1); } } while (0)

int main() {
  int cases = 0;
  for (int nlx = 1; nlx <= 18; ++nlx)
    for (int nly = 1; nly <= 18; ++nly) {
      ++cases;
      std::map<std::pair<int, int>, std::pair<int, int>> want, got;
      for (int lane = 0; lane < shoot_lanes(nlx, nly); ++lane) {
        int fx = 0, fy = 0, n = -1;
        const int k = decode_lane(lane, nlx, nly, &fx, &fy, &n);
        if (k != LANE_IDLE) want[{fx, fy}] = {k, n};
      }
      for (int lane = 0; lane < pair_lanes(nlx, nly) + 3; ++lane) {
        int fx = 0, fy = 0, n = -1, two = 0, n2 = -1;
        const int k = decode_pair(lane, nlx, nly, &fx, &fy, &n, &two, &n2);
        CHECK((lane < pair_lanes(nlx, nly)) == (k != LANE_IDLE), "lane %d of %d kind %d", lane, pair_lanes(nlx, nly), k);
        if (k == LANE_IDLE) continue;
        CHECK((k == LANE_ORIGIN) == (lane == pair_origin_lane(nlx, nly)), "origin at %d", lane);
        CHECK(got.insert({{fx, fy}, {k, n}}).second, "mode twice");
        if (two) CHECK(fx > 0 && got.insert({{-fx, fy}, {k, n2}}).second, "mirror twice");
      }
      CHECK(got == want, "modes differ at %d x %d: %zu and %zu", nlx, nly, got.size(), want.size());
    }
  printf("%d shapes\n", cases);
  return 0;
}
