// Walks the z-sum's groups of planes on the CPU: every row that a sample of a
// regular group asks for is a plane of the volume, and the rows and weights are
// those of the group's LORs. Prints samples, samples of partial groups at the
// volume's last plane, groups that are not regular, and failures.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "gfr_internal.h"

using namespace gfr;

int main() {
  srand(1);
  auto in = [](int lo, int hi) { return lo + (int)(rand() / (RAND_MAX + 1.0) * (hi - lo + 1)); };
  long long samples = 0, ends = 0, irregular = 0, bad = 0;
  for (int i = 0; i < 400; i++) {
    gfr_geometry g{in(4, 40), in(1, 70), 8, 4, 2 * in(0, 5) + 1, 1, 1, 1.f, 0.f, 40.f};
    g.diam_det = (float)in(40, 90);
    g.nseg = 1 + 2 * in(0, g.nzs / (2 * g.span));
    GeomHost h;
    if (derive_geometry(&g, &h, nullptr, true) != GFR_OK) continue;
    const int nl = h.info.lambda1 - h.info.lambda0 + 1, ns = h.info.nsinogs;
    for (int sg : {4, 6, 8}) {
      const auto& groups = h.zgrp[zg_index(sg)];
      const int n = (int)groups.size();
      for (int q = 0; q < n; q++) {
        const int2 e = groups[q];
        bool reg = true;  // as the device marks the groups
        for (int li = 0; li < nl; li++) reg = reg && zg_regular(&h.ztab[(size_t)li * ns + e.x], e.y);
        bool consecutive = true;
        for (int li = 0; li < nl; li++) {
          const uint2* t = &h.ztab[(size_t)li * ns + e.x];
          const int z = (int)(t[0].x & 0xffffu);
          for (int k = 0; k < e.y; k++)
            consecutive = consecutive && (int)(t[k].x & 0xffffu) == z + k &&
                          (int)(t[k].x >> 16) == z + k + 1;
          if (!reg || e.y == 0) continue;  // each LOR's two rows
          samples++;
          ends += e.y < sg && z + e.y == g.nzs - 1;
          for (int k = 0; k <= sg; k++) bad += z + zg_row(k, e.y) > g.nzs - 1;
        }
        irregular += !reg;
        bad += reg != consecutive;
      }
    }
  }
  printf("%lld %lld %lld %lld\n", samples, ends, irregular, bad);
  return bad != 0;
}
