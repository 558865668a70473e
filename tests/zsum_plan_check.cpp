// Walks geometries, subset counts and tile shapes on the CPU and compares the
// log-likelihood partials of each forward pass with the capacity of the buffer
// they are written to. Prints passes, passes of narrow waves with shorter
// subsets, passes with chunks cut at 4 GiB, and failures.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "gfr_internal.h"

using namespace gfr;

namespace {

long long passes = 0, narrow_short = 0, cut = 0, bad = 0;

// End of the partials that the launches of one pass write: chunks of plan.chunk
// angles, each at a whole number of full chunks' blocks.
long long written(const ZsumDims& d, const ZsumPlan& p, int nav) {
  const bool wide = p.kind != kZsumNarrow;
  const long long ngb = wide ? (d.ngroups[zg_index(p.kind)] + 3) / 4 : (d.nsinogs + 7) / 8;
  auto blocks = [&](int na) {
    const long long items = (long long)na * (wide ? (d.nrad + 3) / 4 : d.nrad);
    return ngb * ((items + 63) / 64);
  };
  long long end = 0;
  for (int a0 = 0; a0 < nav; a0 += p.chunk)
    end = std::max(end, blocks(p.chunk) * (a0 / p.chunk) + blocks(std::min(p.chunk, nav - a0)));
  return end;
}

// Buffers are made for `made` subsets and serve passes of `made` or more.
void walk(const gfr_geometry& g, int made) {
  GeomHost h;
  if (derive_geometry(&g, &h, nullptr) != GFR_OK || made > g.nang) return;
  const ZsumDims d = zsum_dims(h);
  const int cap = llh_capacity(h, made);
  const size_t r_cap = d.per * std::min((g.nang + made - 1) / made, kRotChunk);
  Tune shapes[5];
  for (int k = 0; k < 4; k++) {
    shapes[k].tuned = true;
    shapes[k].zsum_sg = k < 3 ? 4 + 2 * k : kZsumNarrow;
  }
  for (const Tune& t : shapes) {  // the last one: not measured
    for (int nsub : {made, made + 1, made + 3, 2 * made, 3 * made}) {
      if (nsub > g.nang) continue;
      // refused by gfr_tuning_set, and not a candidate of the tuner
      if (t.tuned && t.zsum_sg == kZsumNarrow && !zsum_narrow_serves(d, nsub)) continue;
      const int longest = zsum_plan(d, t, 0, nsub, r_cap).kind;
      for (int s : {0, nsub / 2, nsub - 1}) {
        const int nav = (g.nang - s + nsub - 1) / nsub;
        const ZsumPlan p = zsum_plan(d, t, s, nsub, r_cap);
        passes++;
        narrow_short += p.kind == kZsumNarrow && nav < (g.nang + nsub - 1) / nsub;
        cut += p.chunk < std::min(nav, kRotChunk);
        if (p.chunk < 1) continue;  // refused by the launcher
        const long long n = written(d, p, nav);
        if (p.kind != longest || n != p.blocks || n > cap) {
          if (bad++ < 5)
            printf("res %d nzs %d nrad %d nang %d span %d nseg %d made %d nsub %d subset %d: "
                   "kind %d of %d, %lld partials, plan %d, room %d\n", g.res, g.nzs, g.nrad,
                   g.nang, g.span, g.nseg, made, nsub, s, p.kind, longest, n, p.blocks, cap);
        }
      }
    }
  }
}

}  // namespace

int main(int argc, char** argv) {
  const int count = argc > 1 ? atoi(argv[1]) : 1000;
  // long subsets above the narrow kernel's range and short ones below it
  walk({77, 149, 84, 60, 3, 51, 1, 1.f, 100.f, 77.f}, 16);
  walk({83, 121, 89, 151, 5, 19, 1, 1.f, 100.f, 83.f}, 16);
  walk({64, 145, 124, 51, 5, 29, 1, 1.f, 100.f, 64.f}, 12);
  // frames with more subsets than the lanes' buffers were made for
  walk({64, 157, 124, 96, 9, 17, 1, 1.f, 100.f, 64.f}, 8);
  // rotations of 16 angles beyond 4 GiB
  walk({256, 399, 655, 144, 3, 21, 1, 1.f, 400.f, 256.f}, 4);
  walk({512, 511, 512, 64, 3, 21, 1, 1.f, 900.f, 512.f}, 2);
  walk({1023, 200, 300, 40, 3, 1, 1, 1.f, 1600.f, 1023.f}, 2);
  walk({4095, 1201, 300, 40, 3, 1, 1, 1.f, 6000.f, 4095.f}, 2);  // less than one angle
  srand(1);
  auto in = [](int lo, int hi) { return lo + (int)(rand() / (RAND_MAX + 1.0) * (hi - lo + 1)); };
  for (int i = 0; i < count; i++) {
    gfr_geometry g{in(8, 128), in(3, 159), in(1, 147), in(1, 168), 2 * in(0, 5) + 1, 1, 1,
                   1.f, 200.f, 100.f};
    const int most = g.nzs / (2 * g.span);  // segments of each sign that have planes
    g.nseg = 1 + 2 * in(0, most);
    walk(g, in(1, std::min(24, g.nang)));
  }
  printf("%lld %lld %lld %lld\n", passes, narrow_short, cut, bad);
  return bad != 0;
}
