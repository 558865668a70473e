// Walks tilts, sizes and tunings on the CPU: a backprojector that reads through
// LDS windows has room for every plane that a tile's samples touch, and loads
// that many rows (16 a load, two loads where one view is taken at a time).
// Prints shapes with windows, shapes of several views at a time, gathering
// shapes, and failures.
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "gfr_internal.h"

using namespace gfr;

int main() {
  long long win = 0, views = 0, gather = 0, bad = 0;
  Tune asked[14];
  const int shapes[13][3] = {{1, 4, 1}, {1, 5, 1}, {1, 6, 1}, {1, 8, 1}, {1, 16, 1},
                             {0, 1, 1}, {0, 1, 2}, {0, 1, 4}, {0, 2, 1}, {0, 4, 1},
                             {0, 6, 1}, {0, 8, 1}, {0, 16, 1}};
  for (int i = 0; i < 13; i++) {
    asked[i].tuned = true;
    asked[i].back_lds = shapes[i][0];
    asked[i].back_zb = shapes[i][1];
    asked[i].back_ahead = shapes[i][2];
  }
  for (int res : {8, 16, 48, 64, 96, 128, 200}) {
    for (int nzs : {3, 16, 65, 127, 159, 300}) {
      for (float tilt = 0.f; tilt < 5.f; tilt += 0.07f) {
        for (float bins : {0.5f, 1.f, 1.3f, 1.4f}) {
          DevGeom G{};
          G.res = res;
          G.nzs = nzs;
          G.fzb_absmax = tilt;
          G.fxb = bins;
          for (const Tune& t : asked) {  // the last one: not measured
            const BackShape b = back_shape(G, t);
            win += b.win;
            views += b.nv > 1;
            gather += !b.win;
            if (!b.win) {
              bad += b.nv != 1 || b.split;
              continue;
            }
            // positions of a tile span this many planes; their floors and the
            // interpolation partner
            const double span = 7.0 * sqrt(2.0) * tilt + b.zb - 1;
            const int planes = (int)ceil(span) + 2;
            const int loaded = b.nv > 1 ? 16 : 32;
            if (planes > b.rows || b.rows > loaded || 7.0 * sqrt(2.0) * bins + 2 > 15.0 ||
                (b.zb != 1 && b.zb < 4) || (b.zb == 1) != (b.nv > 1)) {
              if (bad++ < 5)
                printf("res %d nzs %d tilt %g bins %g: %d slices, %d views, %d planes, %d rows\n",
                       res, nzs, tilt, bins, b.zb, b.nv, planes, b.rows);
            }
          }
        }
      }
    }
  }
  printf("%lld %lld %lld %lld\n", win, views, gather, bad);
  return bad != 0;
}
