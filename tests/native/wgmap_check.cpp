// Host check of rmx_wgmap.h: every (problem, group, tile) is some workgroup's exactly once and
// the rest are invalid; balanced maps give XCD bid % 8 an eighth of each problem, shared groups
// stay on one XCD; sets run their tiles in order. Exit status 0 when all agree.
#include <cstdio>
#include <set>
#include <tuple>
#include <vector>

#include "rmx_wgmap.h"

int main() {
  long bad = 0, maps = 0;
  for (int groups : {1, 3, 8, 16, 24, 32, 40, 64})
    for (int share : {1, 2, 4, 8})
      for (int uneven = 0; uneven < 2; ++uneven)
        for (const std::vector<int>& nt : std::vector<std::vector<int>>{
                 {1}, {5}, {16}, {31}, {32}, {70}, {300}, {0}, {7, 7, 3}, {16, 16, 1, 0}, {64, 2}}) {
          if (groups % share) continue;
          rmx::WgMapParams m;
          const int n = (int)nt.size();
          const int grid = rmx::plan_workgroups(m, n, groups, share, nt.data(), uneven);
          std::set<std::tuple<int, int, int>> seen;
          std::vector<int> xcd(groups, -1);
          ++maps;
          for (int b = 0; b < grid; ++b) {
            const rmx::WgCoord c = rmx::map_workgroup(m, b);
            if (!c.valid) continue;
            const bool in = c.p >= 0 && c.p < n && c.group >= 0 && c.group < groups && c.tile >= 0 &&
                            c.tile < nt[c.p];
            if (!in || !seen.insert({c.p, c.group, c.tile}).second) ++bad;
            if (in && m.balanced) {
              if (xcd[c.group] >= 0 && xcd[c.group] != b % 8) ++bad;
              xcd[c.group] = b % 8;
            }
          }
          long want = 0;
          for (int t : nt) want += (long)groups * t;
          if ((long)seen.size() != want) ++bad;
          if (m.balanced && m.share > 1 && want)
            for (int g = 0; g < groups; ++g)
              if (xcd[g] != xcd[g / m.share * m.share]) ++bad;
        }
  std::printf("wgmap: %ld maps, %ld mismatches\n", maps, bad);
  return bad != 0;
}
