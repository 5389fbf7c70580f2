// Host check of xcd_tile_run (i8conv_device.hpp): over tile counts 1..2100
// and every grid limit of the persistent kernels, each tile is walked exactly
// once and no workgroup walks more than ceil(tiles / workgroups).
#include <algorithm>
#include <cstdio>
#include <vector>

#include "i8conv_device.hpp"

int main() {
  long bad = 0, checked = 0;
  for (int limit : {256, 512, 768, 1024})
    for (int tiles = 1; tiles <= 2100; ++tiles) {
      const int groups = std::min(tiles, limit), most = (tiles + groups - 1) / groups;
      std::vector<int> seen(tiles, 0);
      int longest = 0;
      for (int b = 0; b < groups; ++b) {
        const i8conv::TileRun r = i8conv::xcd_tile_run(tiles, groups, b);
        int walked = 0;
        for (int t = r.first; t < r.last; t += r.step, ++walked)
          if (t >= 0 && t < tiles) ++seen[t];
        longest = std::max(longest, walked);
      }
      ++checked;
      const bool once = std::all_of(seen.begin(), seen.end(), [](int n) { return n == 1; });
      if (once && longest <= most) continue;
      if (++bad <= 5)
        std::printf("%d tiles, %d workgroups: %s, a workgroup walks %d tiles (at most %d)\n", tiles,
                    groups, once ? "each once" : "NOT each once", longest, most);
    }
  if (bad) return 1;
  std::printf("ok %ld\n", checked);
  return 0;
}
