// gfr_back_window.hip — backprojector (BACKWPROJ_K, GFIRST_GPU_Kernels.cu:
// 109-164) that reads each view's rows through a small LDS window per wave.
//
// A wave owns an 8x8 tile of voxel columns and ZB slices. In one view the
// tile's samples fall into a window of at most 16 bins x 32 planes, whose
// bounds are exact: every coordinate is a monotone (correctly rounded)
// function of the column and the slice, so its extremes are at the tile's
// corners. The wave copies the window with one 16-byte load per lane (4 lanes
// a row, 16 rows an instruction; the next view's load is in flight while the
// current view is summed) and its lanes then read their bin pairs from LDS.
// Nothing is shared between waves but the angle table, so there is no barrier
// in the view loop.
//
// What bounds it: gathers straight from the rows cost 16-32 cycles of the
// CU's vector-memory path per wave load, whatever the load's width (each lane
// quad of a tilted tile touches its own lines), which is what bound the
// kernel this one replaces; the same pair from LDS rows 20 dwords apart costs
// 4-6. The rest is VALU issue, where fma, add, sub and mul with VGPR operands
// issue at about 1.55 a CU-cycle and compares, min/max, conversions and
// operands in SGPRs at about 0.85, so the sums are written with the former:
//   e = clamp(fma(A, 2^127, 1))   1 where A >= 0, 0 where A < 0
//   n = fma(A, e, n), d = d + e   n + A and d + 1, or both unchanged
// (exactly rounded like the additions they stand for).
//
// Measured (pack and backprojection of one subset, before and after): 128x128x
// 159 voxels, 530 views of 128 bins: 604 -> 289 us; the same image, 210 views of
// 147 bins with detector gaps: 254 -> 202 us; 64x64x32, 176 views: 190 -> 45 us
// (57 with one wave per tile and slice).
//
// Where the calibration went: the calibration of a bin is 1 or -1000, and the
// interpolated calibration B of four valid bins is exactly 1. Rows therefore
// hold one float per bin, the ratio where the calibration is valid and
// kInvalid (about -2^126) where it is not (also outside the segment's planes),
// so a sample that gives an invalid bin the weight W > 0 comes out near
// W * kInvalid, far below every sample without one. If W > 1/1001, B is
// negative and the view is dropped: A < 0 does that. Smaller W (samples between
// -kDrop and -kTouch) may still count with B < 1; such a view of a tile is
// summed by the reference's own expression from the rows and the side array,
// which holds the ratios of the invalid bins. So is every view when a ratio
// of the pass is out of the range that these steps are exact for
// (PackedRows::bad).
#include "gfr_device.h"

namespace gfr {

namespace {

constexpr int kWinStride = 20;  // dwords per window row: 16 bins and 4 of padding, so that
                                // a tile's rows and bins spread over the LDS banks
constexpr int kWinRows = 32;    // two loads of 16 rows
constexpr float kTouch = 0x1p70f;         // |regular samples| stay below 2^61
constexpr float kDrop = 0x1.89374cp116f;  // 0.0015 * 2^126: W > 1.1e-3 > 1/1001

// Radial part of a column in an angle (GFIRST_GPU_Kernels.cu:133-147).
struct Radial {
  float yr, au;
  int iq;  // clamp(floor(u - 0.5), -1, NRAD-1): packed entries iq + 1 and iq + 2
};

__device__ __forceinline__ Radial radial(const DevGeom& G, float xv, float yv, float st, float ct) {
  Radial r;
  r.yr = fmaf(yv, ct, -(xv * st));
  const float xr = fmaf(yv, st, xv * ct);
  const float u = fmaf(xr, G.fxb, G.RADM) + 0.5f;
  const float t = u - 0.5f;
  const float f = floorf(t);
  r.au = t - f;
  r.iq = min(max((int)f, -1), G.nrad - 1);
  return r;
}

// The reference's expression for one sample from its four taps (rows hold
// kInvalid where the calibration is -1000 and the ratio is in the side array)
// and the gap rule (GFIRST_GPU_Kernels.cu:150-160): x what it adds to the
// numerator, y to the denominator (zeros where the view is dropped).
__device__ __forceinline__ float2 exact_sample(float r00, float r01, float r10, float r11,
                                               __amdgpu_buffer_rsrc_t rs, unsigned o,
                                               unsigned rowb, float au, float al, bool want) {
  auto cal = [&](float& ratio, unsigned off) {
    const bool inv = ratio == kInvalid;
    if (inv && want) ratio = ld_f1(rs, off, 0);
    return inv ? -1000.f : 1.f;
  };
  const float q00 = cal(r00, o), q01 = cal(r01, o + 4u);
  const float q10 = cal(r10, o + rowb), q11 = cal(r11, o + rowb + 4u);
  const float A = lerp1(lerp1(r00, r01, au), lerp1(r10, r11, au), al);
  const float B = lerp1(lerp1(q00, q01, au), lerp1(q10, q11, au), al);
  const bool ok = want && !(B < 0.f || A < 0.f);
  return make_float2(ok ? A : 0.f, ok ? B : 0.f);
}

// The reference's expression for one view, every lane of the wave: plane
// position per slice, four taps (GFIRST_GPU_Kernels.cu:140-160).
template <int ZB>
__device__ __forceinline__ void exact_view(const DevGeom& G, __amdgpu_buffer_rsrc_t rv,
                                           __amdgpu_buffer_rsrc_t rs, const SegEntry& se,
                                           unsigned vrow, const Radial& rd, int zb, bool act,
                                           float* n, float* d) {
  const unsigned rowb = (unsigned)packed_row_len(G.nrad) * 4u;
  const float fzm = (float)se.zmin, fzhi = (float)(G.nzs - se.zmin);
  float z = (float)zb;
  asm("" : "+v"(z));  // not kept for every slice in a register of its own
#pragma unroll
  for (int j = 0; j < ZB; j++) {
    const float w = fmaf(rd.yr, se.fzb, z + (float)j) + 0.5f;
    float2 r = make_float2(0.f, 0.f);
    if (act && w >= fzm && w < fzhi) {
      const float t = w - 0.5f;
      const float f = floorf(t);
      const unsigned o = (vrow + (unsigned)(int)f) * rowb + (unsigned)(rd.iq + 1) * 4u;
      r = exact_sample(ld_f1(rv, o, 0), ld_f1(rv, o + 4u, 0), ld_f1(rv, o + rowb, 0),
                       ld_f1(rv, o + rowb + 4u, 0), rs, o, rowb, rd.au, t - f, true);
    }
    n[j] += r.x;
    d[j] += r.y;
  }
}

// One slice per wave, for small images, where a wave's walk over the views, a
// chain of instructions and round trips, sets the time (windows of at most 16
// rows). NV views are taken at a time: their windows are loaded together and
// the next NV are in flight meanwhile.
// SPLIT: the four waves of a block share a tile and slice and take NV views each
// a turn. They leave their samples in LDS, and one wave after the other adds a
// turn's samples to the sums in the order of the views.
// TAB: the radial part of every angle of the subset is kept in LDS (few
// angles), else it is computed per view.
// WIN false: the same sums with every pair gathered from the rows, for
// geometries whose tiles need wider windows.
template <int ZB, int NV, bool TAB, bool WIN, bool SPLIT>
__global__ __launch_bounds__(256, ZB * NV <= 8 ? 5 : 3) void k_back_window(
    DevGeom G, BackFrames F, int nf, int subset, int nsub, const int* __restrict__ dsub, int tabf,
    int wrows) {
  // [angle][3][64]: yr, au, entry offset in bytes; then per wave NV windows of
  // wrows rows
  extern __shared__ __align__(16) float tab[];
  if (dsub) subset = *dsub;
  const int nav = (G.nang - subset + nsub - 1) / nsub;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int bx, by, bz;
  xcd_region(bx, by, bz);
  const int fr = __builtin_amdgcn_readfirstlane(bz % nf);  // every frame's heavy slabs first
  bz /= nf;
  const PackedRows P = F.rows[fr];
  // The four waves of a block take the same columns and neighbouring slabs,
  // counted from the middle of the volume outwards: the middle slabs see the
  // most views, so the heaviest blocks start first and the last ones are light.
  // (the waves of a split block take one slab)
  const int ns = (G.nzs + ZB - 1) / ZB, sk = SPLIT ? bz : bz * 4 + wv;
  const int zb = ((sk & 1) ? (ns - 1) / 2 + (sk + 1) / 2 : (ns - 1) / 2 - sk / 2) * ZB;
  const int ix = bx * 8 + (lane & 7), iy = by * 8 + (lane >> 3);
  const bool act = ix < G.res && iy < G.res;
  const float xv = (float)min(ix, G.res - 1) - G.RESM, yv = (float)min(iy, G.res - 1) - G.RESM;
  const float cx0 = (float)(bx * 8) - G.RESM, cx1 = (float)min(bx * 8 + 7, G.res - 1) - G.RESM;
  const float cy0 = (float)(by * 8) - G.RESM, cy1 = (float)min(by * 8 + 7, G.res - 1) - G.RESM;
  if constexpr (TAB) {
    for (int a = wv; a < nav; a += 4) {
      const int it = subset + a * nsub;
      const Radial r = radial(G, xv, yv, G.sin_t[it], G.cos_t[it]);
      float* t = tab + a * 192 + lane;
      t[0] = r.yr;
      t[64] = r.au;
      t[128] = (float)((r.iq + 1) * 4);
    }
    __syncthreads();
  }
  if (sk >= ns) return;  // of four slabs: no barrier follows
  const bool bad = *P.bad == P.epoch;
  const unsigned rowb = (unsigned)packed_row_len(G.nrad) * 4u;
  const unsigned nr = (unsigned)(G.nsinogs + 2 * G.nseg);
  const __amdgpu_buffer_rsrc_t rv = rsrc(P.v, P.bytes);
  const __amdgpu_buffer_rsrc_t rs = rsrc(P.side, P.bytes);
  float* const win = tab + tabf;
  constexpr int kRowB = kWinStride * 4;
  const int wbytes = wv * (NV * wrows * kRowB);
  const float fz0 = (float)zb, fzl = (float)(zb + ZB - 1);
  float n[ZB], d[ZB];
#pragma unroll
  for (int j = 0; j < ZB; j++) n[j] = d[j] = 0.f;
  float big = 0x1p127f;
  asm("" : "+v"(big));  // in a VGPR: an SGPR operand halves the issue rate
  // Plane positions are rounded twice, by at most 2^-23 of their size each
  // time: two slices' fractions differ by less than this.
  const float apart = (float)G.nzs * 0x1p-20f;

  // this lane's 16 bytes of a window: row lane / 4 (and + 16), bins 4 (lane % 4) ...
  const int lrow = lane >> 2;
  const unsigned lcol = (unsigned)(lane & 3) * 16u;
  char* const wst = (char*)win + wbytes + lrow * kRowB + lcol;
  const bool second = lrow + 16 < wrows;
  // rows of the window past the rows that exist repeat the extra rows
  auto fetch = [&](unsigned base, unsigned clamp, int up) -> float4 {
    const unsigned p = min(__builtin_elementwise_sub_sat((unsigned)(lrow + up), clamp & 0xffffu),
                           clamp >> 16);
    return ld_f4(rv, __umul24(p, rowb) + lcol, base);
  };
  auto lane_of = [&](auto v, int k) {
    return __builtin_bit_cast(decltype(v), __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
  };
  // The lane's bin pairs of planes f, f + 1, ...: from the window (col: bytes of
  // its column less the window's origin), or from the rows (col: bytes of its
  // entry; row, clamp: of the view).
  auto pairs = [&](float f, float col, unsigned row, unsigned clamp, auto& q) {
    constexpr int K = sizeof(q) / sizeof(q[0]);
    if constexpr (WIN) {
      const float* p = (const float*)((const char*)win + (int)fmaf(f, (float)kRowB, col));
#pragma unroll
      for (int k = 0; k < K; k++) q[k] = make_float2(p[k * kWinStride], p[k * kWinStride + 1]);
    } else {
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int p = min(max((int)f + 1 + k, (int)(clamp & 0xffffu)), (int)(clamp >> 16));
        q[k] = ld_f2(rv, (row + (unsigned)p) * rowb + (unsigned)(int)col, 0);
      }
    }
  };
  auto planes = [&](float f, float col, float au, unsigned row, unsigned clamp,
                    float (&c)[ZB + 1]) {
    float2 q[ZB + 1];
    pairs(f, col, row, clamp, q);
#pragma unroll
    for (int k = 0; k <= ZB; k++) c[k] = lerp1(q[k].x, q[k].y, au);
  };
  auto add_view = [&](const float (&A)[ZB]) {
#pragma unroll
    for (int j = 0; j < ZB; j++) {
      const float e = __builtin_amdgcn_fmed3f(fmaf(A[j], big, 1.f), 0.f, 1.f);
      n[j] = fmaf(A[j], e, n[j]);
      d[j] += e;
    }
  };

  // split blocks: samples of two turns, what they count where that is not 1 or
  // 0, sums, and per wave the views of a turn that have such samples
  constexpr int kTurn = 4 * NV;
  float* const smp = win + 4 * NV * wrows * kWinStride;
  float* const cts = smp + 2 * kTurn * 64;
  float* const sums = cts + 2 * kTurn * 64;
  int* const rare = (int*)(sums + 128);
  int turn = 0;
  if constexpr (SPLIT) {
    if (wv == 0) {
      sums[lane] = sums[64 + lane] = 0.f;
    }
    __syncthreads();
  }

  const int nviews = G.nseg * nav;  // view v: segment v / nav, angle v % nav
  for (int c0 = 0; c0 < nviews; c0 += 64) {
    // lane k sets up view c0 + k; `m` marks the views that meet the tile's slices
    float r_fzb = 0.f, r_st = 0.f, r_ct = 0.f;
    float r_off = 0.f;     // bytes: window address - 80 * first plane - 4 * first entry
    unsigned r_base = 0;   // bytes: row of the window's first plane that exists, first entry
    unsigned r_clamp = 0;  // window rows before that plane | rows from it to the last << 16
    int r_view = 0;        // angle << 2 | (1: slices share the fraction) | (2: over 16 rows)
    bool used = false;
    {
      const int vi = c0 + lane;
      if (vi < nviews) {
        const int si = vi / nav, a = vi - si * nav;
        const SegEntry se = G.seg[si];
        const int it = subset + a * nsub;
        const float st = G.sin_t[it], ct = G.cos_t[it];
        const float ya = fmaf(cy0, ct, -(cx0 * st)), yb = fmaf(cy0, ct, -(cx1 * st));
        const float yc = fmaf(cy1, ct, -(cx0 * st)), yd = fmaf(cy1, ct, -(cx1 * st));
        const float ymn = fminf(fminf(ya, yb), fminf(yc, yd));
        const float ymx = fmaxf(fmaxf(ya, yb), fmaxf(yc, yd));
        const float smn = fminf(fmaf(ymn, se.fzb, fz0), fmaf(ymx, se.fzb, fz0));
        const float smx = fmaxf(fmaf(ymn, se.fzb, fzl), fmaf(ymx, se.fzb, fzl));
        const float wmn = smn + 0.5f, wmx = smx + 0.5f;
        used = wmx >= (float)se.zmin && wmn < (float)(G.nzs - se.zmin);
        const int lo = (int)floorf(wmn - 0.5f), hi = (int)floorf(wmx - 0.5f) + 1;
        const int e0 = min(min(radial(G, cx0, cy0, st, ct).iq, radial(G, cx1, cy0, st, ct).iq),
                           min(radial(G, cx0, cy1, st, ct).iq, radial(G, cx1, cy1, st, ct).iq)) + 1;
        // slices share one fraction: every plane position is >= 1 and in one
        // binade (see accumulate_view), or the segment has no tilt
        const bool shared = se.fzb == 0.f || (smn >= 1.f && (__float_as_uint(smn) >> 23) ==
                                                                (__float_as_uint(wmx) >> 23));
        r_fzb = se.fzb;
        r_st = st;
        r_ct = ct;
        if constexpr (WIN) {
          r_off = (float)(wbytes - lo * kRowB - e0 * 4);
          const int p0 = max(lo, se.zmin - 1);
          r_base = ((unsigned)a * nr + (unsigned)(se.nza + 2 * si + 1 - se.zmin + p0)) * rowb +
                   (unsigned)e0 * 4u;
          r_clamp = (unsigned)(p0 - lo) | (unsigned)max(G.nzs - se.zmin - p0, 0) << 16;
        } else {  // row of plane -1, planes that exist + 1
          r_base = (unsigned)a * nr + (unsigned)(se.nza + 2 * si - se.zmin);
          r_clamp = (unsigned)se.zmin | (unsigned)(G.nzs - se.zmin + 1) << 16;
        }
        r_view = a * 4 + (shared ? 1 : 0) + (hi - lo >= 16 ? 2 : 0);
      }
    }
    const unsigned long long m_shared = __builtin_amdgcn_ballot_w64((r_view & 1) != 0);
    unsigned long long m = __builtin_amdgcn_ballot_w64(used);
    if (m == 0) continue;

    // column of the lane in view k of the chunk, window u
    auto column = [&](int k, int u, int fl, float& yr, float& au, float& col) {
      if constexpr (TAB) {
        const float* t = tab + (fl >> 2) * 192 + lane;
        yr = t[0];
        au = t[64];
        col = t[128];
      } else {
        const Radial r = radial(G, xv, yv, lane_of(r_st, k), lane_of(r_ct, k));
        yr = r.yr;
        au = r.au;
        col = (float)((r.iq + 1) * 4);
      }
      if constexpr (WIN) col += lane_of(r_off, k);
      if constexpr (NV > 1) col += (float)(u * wrows * kRowB);
    };
    // Samples of a view that a bin without calibration has touched: exact sums
    // for those that still count, the others drop by themselves.
    auto touched = [&](int k, int fl, float yr, float au, float col, float fzb, unsigned row,
                       unsigned clamp, float (&A)[ZB]) {
      bool few = false;
#pragma unroll
      for (int j = 0; j < ZB; j++) few |= A[j] < -kTouch && A[j] > -kDrop;
      if (__builtin_amdgcn_ballot_w64(few) == 0 && !bad) return;
      const int a = fl >> 2, si = (c0 + k) / nav;
      const SegEntry se = G.seg[si];
      const unsigned vrow = (unsigned)a * nr + (unsigned)(se.nza + 2 * si + 1 - se.zmin);
      const int it = subset + a * nsub;
      const Radial r = radial(G, xv, yv, G.sin_t[it], G.cos_t[it]);
      if (bad) {
        exact_view<ZB>(G, rv, rs, se, vrow, r, zb, act, n, d);
#pragma unroll
        for (int j = 0; j < ZB; j++) A[j] = -1.f;
        return;
      }
      float z = fz0;
      asm("" : "+v"(z));
#pragma unroll
      for (int j = 0; j < ZB; j++) {
        const bool fw = A[j] < -kTouch && A[j] > -kDrop;
        if (__builtin_amdgcn_ballot_w64(fw) != 0) {
          const float t = (fmaf(yr, fzb, z + (float)j) + 0.5f) - 0.5f;
          const float f = floorf(t);
          const unsigned o = (vrow + (unsigned)(int)f) * rowb + (unsigned)(r.iq + 1) * 4u;
          float2 q[2];
          pairs(f, col, row, clamp, q);
          const float2 x = exact_sample(q[0].x, q[0].y, q[1].x, q[1].y, rs, o, rowb, au, t - f, fw);
          n[j] += x.x;
          d[j] += x.y;
          A[j] = fw ? -1.f : A[j];
        }
      }
    };
    // samples of one view of the chunk, window u
    auto sample = [&](int k, int u, int fl, float fzb, unsigned row, unsigned clamp, float& yr,
                      float& au, float& col, float (&A)[ZB]) {
      float c[ZB + 1];
      column(k, u, fl, yr, au, col);
      const float s0 = fmaf(yr, fzb, fz0);
      if (fl & 1) {
        const float f0 = floorf(s0);
        planes(f0, col, au, row, clamp, c);
#pragma unroll
        for (int j = 0; j < ZB; j++) A[j] = lerp1(c[j], c[j + 1], s0 - f0);
      } else {
        const float t0 = (s0 + 0.5f) - 0.5f;
        const float f0 = floorf(t0);
        float z = fz0;
        asm("" : "+v"(z));  // not kept for every slice in a register of its own
        // Slice j reads planes f0 + j and f0 + j + 1 unless rounding carries a
        // position across a plane.
        if (ZB == 1 ||
            __builtin_amdgcn_ballot_w64(!(fabsf((t0 - f0) - 0.5f) < 0.5f - apart)) == 0) {
          planes(f0, col, au, row, clamp, c);
          const float g0 = f0 + 0.5f;
#pragma unroll
          for (int j = 0; j < ZB; j++) {
            const float w = fmaf(yr, fzb, z + (float)j) + 0.5f;
            A[j] = lerp1(c[j], c[j + 1], w - (g0 + (float)j));  // (w - 0.5) - (f0 + j), exact
          }
        } else {
#pragma unroll
          for (int j = 0; j < ZB; j++) {
            const float t = (fmaf(yr, fzb, z + (float)j) + 0.5f) - 0.5f;
            const float f = floorf(t);
            float2 q[2];
            pairs(f, col, row, clamp, q);
            A[j] = lerp1(lerp1(q[0].x, q[0].y, au), lerp1(q[1].x, q[1].y, au), t - f);
          }
        }
      }
    };
    auto one_view = [&](int k, int u) {
      const int fl = lane_of(r_view, k);
      const float fzb = lane_of(r_fzb, k);
      const unsigned row = WIN ? 0 : lane_of(r_base, k), clamp = WIN ? 0 : lane_of(r_clamp, k);
      float yr, au, col, A[ZB];
      sample(k, u, fl, fzb, row, clamp, yr, au, col, A);
      // a touched sample is below -2^70, the others' sum within 16 * 2^61
      float sum = A[0];
#pragma unroll
      for (int j = 1; j < ZB; j++) sum += A[j];
      if (__builtin_amdgcn_ballot_w64(sum < -0.5f * kTouch) != 0 || bad)
        touched(k, fl, yr, au, col, fzb, row, clamp, A);
      add_view(A);
    };

    if constexpr (!WIN) {
      for (; m; m &= m - 1) one_view(__builtin_ctzll(m), 0);
    } else if constexpr (NV == 1) {
      int k = __builtin_ctzll(m);
      int flags = lane_of(r_view, k);
      float4 w0, w1 = make_float4(0.f, 0.f, 0.f, 0.f);
      {
        const unsigned base = lane_of(r_base, k);
        const unsigned cl = lane_of(r_clamp, k);
        w0 = fetch(base, cl, 0);
        if (flags & 2) w1 = fetch(base, cl, 16);
      }
      while (m) {
        *(float4*)wst = w0;
        if ((flags & 2) && second) *(float4*)(wst + 16 * kRowB) = w1;
        const int kc = k;
        m &= m - 1;
        if (m) {
          k = __builtin_ctzll(m);
          flags = lane_of(r_view, k);
          const unsigned base = lane_of(r_base, k);
          const unsigned cl = lane_of(r_clamp, k);
          w0 = fetch(base, cl, 0);
          if (flags & 2) w1 = fetch(base, cl, 16);
        }
        wave_sync();
        one_view(kc, 0);
        wave_sync();  // the window may be overwritten
      }
    } else if constexpr (!SPLIT) {
      int kk[NV];
      float4 w[NV];
      int left = __popcll(m);
      auto take = [&]() {  // the next NV views (the last one again past the end)
#pragma unroll
        for (int u = 0; u < NV; u++) {
          if (m) {
            kk[u] = __builtin_ctzll(m);
            m &= m - 1;
          } else if (u) {
            kk[u] = kk[u - 1];
          }
          w[u] = fetch(lane_of(r_base, kk[u]), lane_of(r_clamp, kk[u]), 0);
        }
      };
      take();
      while (left > 0) {
        int kc[NV];
        bool all = left >= NV && !bad;
#pragma unroll
        for (int u = 0; u < NV; u++) {
          kc[u] = kk[u];
          all = all && ((m_shared >> kk[u]) & 1) != 0;
          *(float4*)(wst + u * wrows * kRowB) = w[u];
        }
        if (left > NV) take();
        wave_sync();
        bool done = false;
        if (all) {
          float A[NV][ZB], sum = 0.f;
#pragma unroll
          for (int u = 0; u < NV; u++) {
            float yr, au, col, c[ZB + 1];
            column(kc[u], u, lane_of(r_view, kc[u]), yr, au, col);
            const float s0 = fmaf(yr, lane_of(r_fzb, kc[u]), fz0);
            const float f0 = floorf(s0);
            planes(f0, col, au, 0, 0, c);
#pragma unroll
            for (int j = 0; j < ZB; j++) {
              A[u][j] = lerp1(c[j], c[j + 1], s0 - f0);
              sum += A[u][j];
            }
          }
          if (__builtin_amdgcn_ballot_w64(sum < -0.5f * kTouch) == 0) {
#pragma unroll
            for (int u = 0; u < NV; u++) add_view(A[u]);
            done = true;
          }
        }
        if (!done) {
          const int g = min(left, NV);
          int mk = kc[0] | kc[1] << 6 | (NV > 2 ? kc[NV > 2 ? 2 : 0] << 12 | kc[NV > 3 ? 3 : 0] << 18 : 0);
          for (int u = 0; u < g; u++, mk >>= 6) one_view(mk & 63, u);
        }
        wave_sync();
        left -= NV;
      }
    } else {
      // lane k: the chunk's k-th view that meets the slice
      const int cnt = __popcll(m);
      const int below = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
      const int order = __builtin_amdgcn_ds_permute((used ? below : cnt + lane - below) * 4, lane);
      int kk[NV];
      float4 w[NV];
      auto take = [&](int p0) {  // this wave's views of the turn at p0 (the last one past the end)
#pragma unroll
        for (int u = 0; u < NV; u++) {
          kk[u] = lane_of(order, min(p0 + wv * NV + u, cnt - 1));
          w[u] = fetch(lane_of(r_base, kk[u]), lane_of(r_clamp, kk[u]), 0);
        }
      };
      take(0);
      for (int p0 = 0; p0 < cnt; p0 += kTurn, turn++) {
        int kc[NV];
        bool all = true;
#pragma unroll
        for (int u = 0; u < NV; u++) {
          kc[u] = kk[u];
          all = all && ((m_shared >> kk[u]) & 1) != 0;
          *(float4*)(wst + u * wrows * kRowB) = w[u];
        }
        if (p0 + kTurn < cnt) take(p0 + kTurn);
        wave_sync();
        float A[NV][ZB], sum = 0.f;
        float yr[NV], au[NV], col[NV];
        if (all) {
#pragma unroll
          for (int u = 0; u < NV; u++) {
            float c[ZB + 1];
            column(kc[u], u, lane_of(r_view, kc[u]), yr[u], au[u], col[u]);
            const float s0 = fmaf(yr[u], lane_of(r_fzb, kc[u]), fz0);
            const float f0 = floorf(s0);
            planes(f0, col[u], au[u], 0, 0, c);
            A[u][0] = lerp1(c[0], c[1], s0 - f0);
          }
        } else {
#pragma unroll
          for (int u = 0; u < NV; u++)
            sample(kc[u], u, lane_of(r_view, kc[u]), lane_of(r_fzb, kc[u]), 0, 0, yr[u], au[u],
                   col[u], A[u]);
        }
        const int at = ((turn & 1) * kTurn + wv * NV) * 64 + lane;
#pragma unroll
        for (int u = 0; u < NV; u++) {
          smp[at + u * 64] = A[u][0];
          sum += A[u][0];
        }
        int exact = bad ? (1 << NV) - 1 : 0;
        if (__builtin_amdgcn_ballot_w64(sum < -0.5f * kTouch) != 0 || bad) {
#pragma unroll
          for (int u = 0; u < NV; u++) {
            const bool few = A[u][0] < -kTouch && A[u][0] > -kDrop;
            if (__builtin_amdgcn_ballot_w64(few) == 0 && !bad) continue;
            exact |= 1 << u;
            const int a = lane_of(r_view, kc[u]) >> 2, si = (c0 + kc[u]) / nav;
            const SegEntry se = G.seg[si];
            const unsigned vrow = (unsigned)a * nr + (unsigned)(se.nza + 2 * si + 1 - se.zmin);
            const int it = subset + a * nsub;
            const Radial r = radial(G, xv, yv, G.sin_t[it], G.cos_t[it]);
            float x[ZB] = {0.f}, ct[ZB] = {0.f};
            if (bad) {
              exact_view<ZB>(G, rv, rs, se, vrow, r, zb, act, x, ct);
            } else {
              const float t = (fmaf(yr[u], se.fzb, fz0) + 0.5f) - 0.5f;
              const float f = floorf(t);
              const unsigned o = (vrow + (unsigned)(int)f) * rowb + (unsigned)(r.iq + 1) * 4u;
              float2 q[2];
              pairs(f, col[u], 0, 0, q);
              const float2 e = exact_sample(q[0].x, q[0].y, q[1].x, q[1].y, rs, o, rowb, au[u],
                                            t - f, few);
              x[0] = few ? e.x : A[u][0] < 0.f ? 0.f : A[u][0];
              ct[0] = few ? e.y : A[u][0] < 0.f ? 0.f : 1.f;
            }
            smp[at + u * 64] = x[0];
            cts[at + u * 64] = ct[0];
          }
        }
        rare[(turn & 1) * 4 + wv] = exact << (wv * NV);
        __syncthreads();
        if ((turn & 3) == wv) {  // the others take the next turn meanwhile
          const int nt = min(kTurn, cnt - p0);
          const float* from = smp + (turn & 1) * kTurn * 64 + lane;
          n[0] = sums[lane];
          d[0] = sums[64 + lane];
          const int4 rw = *(const int4*)(rare + (turn & 1) * 4);
          const int rm = __builtin_amdgcn_readfirstlane(rw.x | rw.y | rw.z | rw.w);
          if (rm) {
            for (int v = 0; v < nt; v++) {
              if ((rm >> v) & 1) {
                n[0] += from[v * 64];
                d[0] += from[(2 * kTurn + v) * 64];
              } else {
                const float x[ZB] = {from[v * 64]};
                add_view(x);
              }
            }
          } else {
#pragma unroll 4
            for (int v = 0; v < nt; v++) {
              const float x[ZB] = {from[v * 64]};
              add_view(x);
            }
          }
          sums[lane] = n[0];
          sums[64 + lane] = d[0];
        }
      }
    }
  }
  if constexpr (SPLIT) {
    __syncthreads();
    if (wv != 0) return;
    n[0] = sums[lane];
    d[0] = sums[64 + lane];
  }
  if (!act) return;
#pragma unroll
  for (int j = 0; j < ZB; j++) {
    const int iz = zb + j;
    if (iz < G.nzs) {
      const size_t iV = ((size_t)iz * G.res + iy) * G.res + ix;
      if (F.denom[fr]) {
        F.numer[fr][iV] = n[j];
        F.denom[fr][iV] = d[j];
      } else {
        F.numer[fr][iV] = update_ratio(n[j], d[j]);
      }
    }
  }
}

constexpr int kTabAngles = 24;  // radial tables up to 18 KB a block

// Rows of a window: 7 columns further in x and in y move a plane position by
// at most 7 sqrt(2) |fzb| planes; 2 more for the position between planes and
// the interpolation partner, and rounding.
int window_rows(const DevGeom& G, int zb) {
  return (int)ceilf(9.9f * G.fzb_absmax + (float)(zb - 1) + 0.01f) + 2;
}

template <int ZB, int NV, bool WIN, bool SPLIT>
hipError_t launch_zb(const DevGeom& G, const BackFrames& F, int nf, int subset, int nsub,
                     const int* dsub, int nav, int rows, hipStream_t st) {
  const unsigned nt = (G.res + 7) / 8, ns = (G.nzs + ZB - 1) / ZB;
  const dim3 grid(nt, nt, (SPLIT ? ns : (ns + 3) / 4) * nf);
  const int tabf = nav <= kTabAngles ? nav * 192 : 0;
  const unsigned split = SPLIT ? 2 * 2 * 4 * NV * 64 + 128 + 8 : 0;
  const unsigned lds = (unsigned)(tabf + 4 * NV * rows * kWinStride + split) * 4u;
  if (tabf)
    hipLaunchKernelGGL((k_back_window<ZB, NV, true, WIN, SPLIT>), grid, dim3(256), lds, st, G, F, nf,
                       subset, nsub, dsub, tabf, rows);
  else
    hipLaunchKernelGGL((k_back_window<ZB, NV, false, WIN, SPLIT>), grid, dim3(256), lds, st, G, F, nf,
                       subset, nsub, dsub, tabf, rows);
  return hipGetLastError();
}

}  // namespace

// In bins: 7 sqrt(2) fxb, and 2 more as above.
bool back_window_fits(const DevGeom& G, int zb) {
  return 9.9f * G.fxb + 2.01f <= 15.f && window_rows(G, zb) <= kWinRows;
}

// Several views at a time: their windows take one load of 16 rows each.
static bool one_slice_fits(const DevGeom& G) {
  return back_window_fits(G, 1) && window_rows(G, 1) <= 16;
}

// Shape for a geometry that has not been measured. By the number of waves with
// 8 slices each, against 1024 SIMDs that hold 5 of them (us of one subset with
// 1 slice split / 1 / 4 / 8 slices: 108 waves 24 / 39 / 56 / 77, 256 waves 44 /
// 59 / 84 / 121, 576 waves 64 / 52 / 66 / 90, 864 waves 108 / 92 / 76 / 98, 1536
// waves 117 / 94 / 59 / 77, 3072 waves 442 / 388 / 139 / 150; 4 / 8 slices: 3840
// waves 249 / 310, 5120 waves 378 / 299).
// Where windows do not fit, as many slices as gathers from L1 favour; where one
// slice's window takes more than 16 rows, one slice gathers too (1 slice / 4 of
// the window kernel: 192 waves 92 / 104, 576 waves 97 / 108; 2 slices gathering
// 107 in both).
static Tune untuned_shape(const DevGeom& G) {
  const int nt = (G.res + 7) / 8, w8 = nt * nt * ((G.nzs + 7) / 8);
  Tune t;
  t.back_lds = 1;
  t.back_zb = w8 < 700 ? 1 : w8 < 4500 ? 4 : 8;
  t.back_ahead = w8 < 400 ? 2 : w8 < 700 ? 4 : 1;
  if (t.back_zb == 1 ? !one_slice_fits(G) : !back_window_fits(G, t.back_zb)) {
    t.back_lds = 0;
    t.back_zb = w8 < 700 ? 1 : w8 < 4500 ? 2 : 6;
    t.back_ahead = 1;
  }
  return t;
}

BackShape back_shape(const DevGeom& G, const Tune& asked) {
  const Tune t = asked.tuned ? asked : untuned_shape(G);
  const bool one = t.back_zb == 1 && t.back_ahead > 1 && one_slice_fits(G);
  BackShape b{};
  b.zb = t.back_zb;
  b.win = one || (t.back_zb >= 4 && t.back_lds && back_window_fits(G, t.back_zb));
  b.split = one && t.back_ahead == 2;
  b.nv = b.split ? 2 : one ? 4 : 1;
  b.rows = b.win ? max(16, window_rows(G, b.zb)) : 0;
  return b;
}

hipError_t launch_back_packed(const DevGeom& G, const BackFrames& F, int nf, int subset, int nsub,
                              const int* dsub, const Tune& tune, hipStream_t st) {
  if (nf < 1 || nf > kMaxGroup) return hipErrorInvalidValue;
  if (packed_bytes(G, dsub ? 0 : subset, nsub) >= 0xFFFFFFF0u) return hipErrorInvalidValue;
  const int nav = (G.nang - (dsub ? 0 : subset) + nsub - 1) / nsub;
  const BackShape b = back_shape(G, tune);
#define GFR_BS(ZB, NV, WIN, SPLIT) \
  return launch_zb<ZB, NV, WIN, SPLIT>(G, F, nf, subset, nsub, dsub, nav, b.rows, st)
#define GFR_BW(ZB, NV, WIN) GFR_BS(ZB, NV, WIN, false)
  if (b.split) GFR_BS(1, 2, true, true);
  if (b.nv == 4) GFR_BW(1, 4, true);
  if (b.win) {
    switch (b.zb) {
      case 4: GFR_BW(4, 1, true);
      case 5: GFR_BW(5, 1, true);
      case 6: GFR_BW(6, 1, true);
      case 8: GFR_BW(8, 1, true);
      case 16: GFR_BW(16, 1, true);
    }
    return hipErrorInvalidValue;
  }
  switch (b.zb) {
    case 1: GFR_BW(1, 1, false);
    case 2: GFR_BW(2, 1, false);
    case 4: GFR_BW(4, 1, false);
    case 5: GFR_BW(5, 1, false);
    case 6: GFR_BW(6, 1, false);
    case 8: GFR_BW(8, 1, false);
    case 16: GFR_BW(16, 1, false);
  }
  return hipErrorInvalidValue;
#undef GFR_BW
#undef GFR_BS
}

}  // namespace gfr
