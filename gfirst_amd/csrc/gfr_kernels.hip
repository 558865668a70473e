// gfr_kernels.hip — gfx950 kernels of the OSEM hot path.
//
// Rounding model (shared with the CPU oracle so results compare bit for bit):
// the file is compiled with -ffp-contract=off; the only fused multiply-adds
// are explicit fmaf() calls. Interpolation weights are exact FP32:
// lerp(a,b,t) = fma(t, b-a, a), x first, then y, then z.
#include <math.h>

#include "gfr_device.h"

namespace gfr {

namespace {

__device__ __forceinline__ Float4u load4(const float* p, int m) {
  if (m == 4) return *(const Float4u*)p;
  return Float4u{p[0], m > 1 ? p[1] : 0.f, m > 2 ? p[2] : 0.f, 0.f};
}

// Ratio alone (GFIRST.cu:415-430) over the subset's bins, 4 of a row a thread;
// the background is in storage format S. One subset of 16 at 128x160x4319 bins
// with packed rows: 29 -> 21 us (one bin a thread before).
template <int S>
__global__ __launch_bounds__(256) void k_ratio(DevGeom G, const float* __restrict__ proj,
                                               const float* __restrict__ y,
                                               const void* __restrict__ bg, float yscale,
                                               float* __restrict__ corr, PackedRows P,
                                               const uint8_t* __restrict__ mask, int subset,
                                               int nsub) {
  const int quads = (G.nrad + 3) / 4;
  const int i = blockIdx.x * 256 + threadIdx.x, s = i / quads, r = (i - s * quads) * 4;
  const int it = subset + (int)blockIdx.y * nsub;
  if (s >= G.nsinogs) return;
  const int m = min(4, G.nrad - r);
  const size_t bin = ((size_t)s * G.nang + it) * G.nrad + r;
  const Float4u pv = load4(proj + bin, m), yy = load4(y + bin, m);
  const float p[4] = {pv.x, pv.y, pv.z, pv.w}, yv[4] = {yy.x, yy.y, yy.z, yy.w};
  float c[4];
  bool valid[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    float bv = bg && k < m ? yscale * load_store<S>(bg, bin + k) : 0.f;
    if (bv < 0.f) bv = 0.f;
    const float den = p[k] + bv;
    c[k] = (den >= 0.01f) ? yscale * yv[k] / den : -1000.f;
    valid[k] = P.v && k < m ? mask[bin + k] != 0 : true;
    if (corr && k < m) corr[bin + k] = c[k];
  }
  if (P.v) store_packed(G, P, blockIdx.y, s, r, m, c, valid);
}

// ---------------------------------------------------------------------------
// XY blur (convolutionXY_GPU, GFIRST_GPU_Kernels.cu:332-358). SRC reads the
// input value (plain load, or the update ratio NUMER/DENOM).
// ---------------------------------------------------------------------------
struct SrcPlain {
  static constexpr bool kStage = false;
  const float* p;
  __device__ __forceinline__ float operator()(size_t i) const { return p[i]; }
};
struct SrcRatio {  // divVxVGPU (GFIRST_GPU_Kernels.cu:173-182)
  static constexpr bool kStage = true;  // a division per element: once, in LDS
  const float* num;
  const float* den;
  __device__ __forceinline__ float operator()(size_t i) const {
    const float b = den[i];
    return update_ratio(num[i], b);
  }
};

// One block per (plane, kBlurRows output rows). A thread loads the rows that
// kBlurCol outputs of one column need (zero outside the plane), y-filters them in registers and leaves them in LDS;
// then a thread x-filters four neighbouring columns from three 16-byte reads.
// What bounds it: the chain of loads, barrier and LDS reads, at about twice the
// time its bytes take. 128x128x159: 13 -> 8.7 us; with the ratio, whose divisions are
// done once in LDS, 18 -> 13 us (all through LDS by single words before).
constexpr int kBlurRows = 16, kBlurCol = 8;
__host__ __device__ inline int blur_stride(int res) { return (res + 3) / 4 * 4; }

template <class Src>
__global__ __launch_bounds__(256) void k_blur_xy(int res, int nzs, Taps9 t, Src src,
                                                 float* __restrict__ out) {
  extern __shared__ __align__(16) float yc[];  // kBlurRows rows of blur_stride(res)
  const int z = blockIdx.y, stride = blur_stride(res);
  const int y0 = blockIdx.x * kBlurRows;
  const int nrows = min(kBlurRows, res - y0);
  const size_t pb = (size_t)z * res * res;
  const int tid = threadIdx.x;
  float* const staged = yc + kBlurRows * stride;  // kBlurRows + 8 rows
  if constexpr (Src::kStage) {
    for (int i = tid; i < (nrows + 8) * res; i += 256) {
      const int y = y0 - 4 + i / res;
      staged[i] = (y >= 0 && y < res) ? src(pb + (size_t)(y0 * res) + i - 4 * res) : 0.f;
    }
    __syncthreads();
  }
  for (int i = tid; i < (kBlurRows / kBlurCol) * res; i += 256) {
    const int g = i / res, x = i - g * res, r0 = g * kBlurCol, ya = y0 + r0 - 4;
    if (r0 >= nrows) break;
    float in[kBlurCol + 8];
#pragma unroll
    for (int j = 0; j < kBlurCol + 8; j++) {
      const int y = ya + j;
      if constexpr (Src::kStage)
        in[j] = staged[(r0 + j) * res + x];
      else
        in[j] = (y >= 0 && y < res) ? src(pb + (size_t)y * res + x) : 0.f;
    }
    const bool border = x < 4 || x >= res - 4;  // raw input at the x borders
#pragma unroll
    for (int k = 0; k < kBlurCol; k++) {
      float acc = in[k] * t.g[0];
#pragma unroll
      for (int j = 1; j < 9; j++) acc = fmaf(in[k + j], t.g[j], acc);
      yc[(r0 + k) * stride + x] = acc;
      if (border && r0 + k < nrows) out[pb + (size_t)(y0 + r0 + k) * res + x] = in[k + 4];
    }
  }
  __syncthreads();
  const int quads = (res + 3) / 4;
  for (int i = tid; i < nrows * quads; i += 256) {
    const int row = i / quads, x = (i - row * quads) * 4;
    if (x < 4 || x >= res - 4) continue;
    const float* yr = yc + row * stride + x - 4;
    float v[12];
#pragma unroll
    for (int k = 0; k < 3; k++) *(float4*)(v + 4 * k) = ((const float4*)yr)[k];
    float o[4];
#pragma unroll
    for (int c = 0; c < 4; c++) {
      o[c] = v[c] * t.g[0];
#pragma unroll
      for (int k = 1; k < 9; k++) o[c] = fmaf(v[c + k], t.g[k], o[c]);
    }
    float* p = out + pb + (size_t)(y0 + row) * res + x;
    if (x + 4 <= res - 4) {
      *(Float4u*)p = Float4u{o[0], o[1], o[2], o[3]};
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++)
        if (x + c < res - 4) p[c] = o[c];
    }
  }
}

// Gz with the reference's index shift, multiply, slice copies
// (GFIRST_CPU_Kernels.cpp:174-186; GFIRST.cu:491-502), for slices 1..NZS-2, 4
// voxels a thread; slices 0 and NZS-1 receive copies of slices 1 and NZS-2, so
// each voxel is read and written by one thread only (in place). The reference
// takes the slice of voxel n as K = (n - 1) / RES^2: that is z, except for a
// slice's first voxel. 128x128x159: 10.7 -> 9.7 us (single voxels and a
// 64-bit division each before).
__global__ __launch_bounds__(256) void k_gz_mul(int res, int nzs, Taps5 t,
                                                const float* __restrict__ f1,
                                                float* __restrict__ x) {
  const int q = (blockIdx.x * 256 + threadIdx.x) * 4, r2 = res * res;
  const int z = blockIdx.y + 1, m = min(4, r2 - q);
  if (m <= 0) return;
  const size_t n = (size_t)z * r2 + q;
  // slices z - 2 .. z + 2 (zero outside the volume)
  float s[5][4];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int zz = z + k - 2;
    const Float4u v = zz >= 0 && zz < nzs ? load4(f1 + (size_t)zz * r2 + q, m)
                                          : Float4u{0.f, 0.f, 0.f, 0.f};
    s[k][0] = v.x, s[k][1] = v.y, s[k][2] = v.z, s[k][3] = v.w;
  }
  const Float4u xv = load4(x + n, m);
  const float xi[4] = {xv.x, xv.y, xv.z, xv.w};
  float o[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int K = q + c == 0 ? z - 1 : z;
    float v;
    if (K == 0)
      v = 0.5f * s[2][c] + 0.5f * s[3][c];
    else if (K == 1 || K == nzs - 2)
      v = 0.333f * s[1][c] + 0.333f * s[2][c] + 0.333f * s[3][c];
    else
      v = t.g[0] * s[0][c] + t.g[1] * s[1][c] + t.g[2] * s[2][c] + t.g[3] * s[3][c] +
          t.g[4] * s[4][c];
    o[c] = xi[c] * v;
  }
  auto put = [&](float* p) {
    if (m == 4) {
      *(Float4u*)p = Float4u{o[0], o[1], o[2], o[3]};
    } else {
#pragma unroll
      for (int c = 0; c < 3; c++)
        if (c < m) p[c] = o[c];
    }
  };
  put(x + n);
  if (z == 1) put(x + n - r2);
  if (z == nzs - 2) put(x + n + r2);
}

// ---------------------------------------------------------------------------
// Joint bilateral filter (jointbilateralfilter3D_K, GFIRST_GPU_Kernels.cu:
// 508-539). Spatial weights come from a host table of exp(-d2/(2 sigma)^2)
// (d2 is an integer); intensity weights exp() in double, stored as float.
// ---------------------------------------------------------------------------
struct GTab { float g[193]; };  // d2 = 0..3*8*8

__global__ __launch_bounds__(256) void k_jbf(int res, int nzs, const float* __restrict__ in,
                                             const float* __restrict__ guide,
                                             const float* __restrict__ d_max, float max_ref,
                                             int r, double kI, GTab gt,
                                             float* __restrict__ out) {
  const int ix = blockIdx.x * kWave + threadIdx.x;
  const int iy = blockIdx.y * 4 + threadIdx.y;
  const int iz = blockIdx.z;
  if (ix >= res || iy >= res) return;
  const size_t iV = ((size_t)iz * res + iy) * res + ix;
  if (ix < r || iy < r || iz < r) {
    out[iV] = 0.f;
    return;
  }
  const float mref = d_max ? __uint_as_float(*(const unsigned int*)d_max) : max_ref;
  const float rv = guide[iV];
  float norm = 0.f, sum = 0.f;
  const int z1 = min(iz + r, nzs - 1), y1 = min(iy + r, res - 1), x1 = min(ix + r, res - 1);
  for (int zz = iz - r; zz <= z1; zz++) {
    for (int yy = iy - r; yy <= y1; yy++) {
      const size_t rowb = ((size_t)zz * res + yy) * res;
      for (int xx = ix - r; xx <= x1; xx++) {
        const size_t iW = rowb + xx;
        const float tq = (guide[iW] - rv) / mref;
        const float di2 = tq * tq;
        const int d2 = (xx - ix) * (xx - ix) + (yy - iy) * (yy - iy) + (zz - iz) * (zz - iz);
        const float H = (float)exp(-(double)di2 / kI);
        const float hg = H * gt.g[d2];
        norm += hg;
        sum = fmaf(hg, in[iW], sum);
      }
    }
  }
  out[iV] = ((double)norm > 1e-8) ? sum / norm : 0.f;
}

// The reference's radius (4, GFIRST.cu:512). Lanes are consecutive voxels of
// the interior columns, so a wave is full whatever the image side; each walks
// its neighbours in the reference's order (z, then y, then x), skipping those
// past the volume's upper faces.
//
// Each intensity weight H = (float)exp(-(double)di2 / kI) is first computed in
// pairs of floats, with a result that is kept only if it is provably the same
// float:
//  - tq = (g - rv) / mref from y = RN(1/mref) and the rest yl of 1/mref:
//    q = RN(a y + a yl) is a faithful quotient, and its correction by the exact
//    remainder is the correctly rounded one (Markstein). It holds while
//    nothing underflows or overflows: for mref in [2^-20, 2^20) and |q| in
//    [2^-60, 2^90). Outside that range the weight is the same either way when
//    kI is in [2^-80, 2^40]: |q| < 2^-60 gives x < 2^-40 and H = 1; |q| >= 2^90
//    gives H = 0 or a NaN, which takes the reference expression. With mref or
//    kI outside those bounds every weight takes that expression.
//  - t = -di2 / kI * 8192 / ln2 is split as n + 1/2 + f, f in (-0.38, 0.63), by
//    a sum with 2^22 - 1/4, whose bits hold 4 n: f = di2 (nh + nl) - (n + 1/2)
//    in two FMAs, where nh + nl is the factor to 2^-48.
//  - H = 2^(n >> 13) |T + s|, s = RN(T p + Tl), with the table's T + Tl =
//    -2^((j + 1/2)/8192), j = n mod 8192, and p = exp(f ln2/8192) - 1 as a
//    quadratic. T + s is within 2^-35 of the exact value (0.82 of that at most
//    over all floats di2), so its rounding to 24 bits is that of the exact one
//    unless the rest e of that rounding lies within 2^-35 of half a unit.
//  - Rare rows of neighbours hold more: x >= 104.5 gives 0, a value below
//    2^-125 is rounded again to a multiple of 2^-149, and one that may lie at a
//    rounding midpoint (2e-4 of them) takes the reference expression.
//
// What bounds it: VALU issue, 29 full-rate instructions a weight with its sums
// (about 50 with the exponential in FP64, which issues at half the rate). One
// pass at 128x128x159: 1.37 -> 0.87 ms. A table of 8192 entries in 64 KB leaves
// 16 waves per CU, which is enough: the loop has no other long wait. Two rows
// per thread would share their loads but last twice as long: a few waves whose
// every row is rare end late, 1.00 ms.
namespace jbfx {
constexpr int kTab = 8192;
constexpr double kLn2 = 0x1.62e42fefa39efp-1;
constexpr float kS = 0x1p22f - 0.25f, kM = 0x1p22f - 0.5f;
constexpr float kC1 = (float)(kLn2 / kTab);
constexpr float kC2 = (float)(kLn2 / kTab * (kLn2 / kTab) / 2);
constexpr float kKeep = 0x1p-24f - 0x1p-35f;                        // largest |e| kept
constexpr float kFar = (float)(0x1p22 - 87.0 / kLn2 * kTab);        // H below 2^-125
constexpr float kUnder = (float)(0x1p22 - 104.5 / kLn2 * kTab);     // H = 0
struct Table { float v[2 * kTab]; };
// -2^((j + 1/2)/8192) as float + float, by the series of exp in double
constexpr Table table() {
  Table t{};
  for (int j = 0; j < kTab; j++) {
    const double u = kLn2 * (j + 0.5) / kTab;
    double e = 1.0;
    for (int i = 17; i > 0; i--) e = 1.0 + e * u / i;
    t.v[j] = (float)-e;
    t.v[kTab + j] = (float)((float)e - e);
  }
  return t;
}
__device__ const Table kT = table();
constexpr int kThreads = 512;

// The weight of a neighbour between 2^-151 and 2^-125, from the sum sh, the
// weight v = 2^k |h| as if exponents had no end, and the rest e of h: |h|
// rounded to a multiple of 2^-149. False if sh is not in that range or the
// value may lie at a rounding midpoint.
__device__ inline bool low_weight(float sh, float v, float e, float* w) {
  const unsigned n = (__float_as_uint(sh) & ~(4u * kTab - 1u)) << 8, x = n & 0x7f800000u;
  const float h = __uint_as_float(__float_as_uint(v) - n);
  *w = h * -0x1p-64f * __uint_as_float(x - (65u << 23));  // x: 256 + k, in place
  const float rest = h + *w * 0x1p64f * __uint_as_float((319u << 23) - x) + e;
  const float half = __uint_as_float((233u << 23) - x);
  return (sh < kFar) & (sh >= kUnder) & (fabsf(rest) <= fmaf(half, 1 - 0x1p-20f, -0x1p-35f));
}
}  // namespace jbfx

__global__ __launch_bounds__(jbfx::kThreads, 4) void k_jbf_r4(
    int res, int nzs, const float* __restrict__ in, const float* __restrict__ guide,
    const float* __restrict__ d_max, float max_ref, double kI, float nh_, float nl_, GTab gt,
    float* __restrict__ out) {
  using namespace jbfx;
  constexpr int R = 4, W = 2 * R + 1;
  __shared__ __align__(16) float tab[2 * kTab];
  const int r2 = res * res, iz = blockIdx.y, side = res - R;  // columns R..res-1
  const int i = blockIdx.x * kThreads + threadIdx.x, n = gridDim.x * kThreads;
  // the low borders are zero
  if (iz < R || side <= 0) {
    for (int j = i; j < r2; j += n) out[(size_t)iz * r2 + j] = 0.f;
    return;
  }
  for (int j = i; j < R * res + R * side; j += n) {
    const int k = j - R * res;
    out[(size_t)iz * r2 + (k < 0 ? j : (R + k / R) * res + k % R)] = 0.f;
  }
  for (int j = threadIdx.x; j < kTab / 2; j += kThreads)
    ((float4*)tab)[j] = ((const float4*)kT.v)[j];
  __syncthreads();
  const int iy = R + i / side, ix = R + i % side;
  if (iy >= res) return;
  const unsigned vbytes = (unsigned)(r2 * nzs) * 4u;
  const __amdgpu_buffer_rsrc_t rg = rsrc(guide, vbytes), ri = rsrc(in, vbytes);
  float mref = d_max ? __uint_as_float(*(const unsigned int*)d_max) : max_ref;
  const bool all = !(mref >= 0x1p-20f && mref < 0x1p20f && kI >= 0x1p-80 && kI <= 0x1p40);
  // constants in vector registers: an instruction with a scalar operand issues
  // at half the rate
  float yh = 1.0f / mref;
  float yl = fmaf(-mref, yh, 1.0f) * yh, nh = nh_, nl = nl_, S = kS, M = kM, C1 = kC1, C2 = kC2;
  asm volatile("" : "+v"(mref), "+v"(yh), "+v"(yl), "+v"(nh), "+v"(nl));
  asm volatile("" : "+v"(S), "+v"(M), "+v"(C1), "+v"(C2));
  const int iV = (iz * res + iy) * res + ix;
  const float rv = ld_f1(rg, 4u * iV, 0);
  float norm = 0.f, sum = 0.f;
  // bit k: neighbour ix + k - R lies inside the volume
  const unsigned vmask = 0x1ffu >> max(0, ix + R - (res - 1));
  for (int dz = -R; dz <= min(R, nzs - 1 - iz); dz++) {
    for (int dy = -R; dy <= R; dy++) {
      if (iy + dy > res - 1) continue;
      unsigned voff = (unsigned)(iV + dz * r2 + dy * res - R) * 4u;
      asm volatile("" : "+v"(voff));  // row start as the base: texel k at immediate 4k
      float gv[W], iv[W], H[W], e[W], sh[W];
#pragma unroll
      for (int k = 0; k < W; k++) {
        gv[k] = ld_f1(rg, voff + 4u * k, 0);
        iv[k] = ld_f1(ri, voff + 4u * k, 0);
      }
      float emax = 0.f, smin = 0x1p22f;
#pragma unroll
      for (int k = 0; k < W; k++) {
        const float a = gv[k] - rv;
        const float q = fmaf(a, yh, a * yl);
        const float tq = fmaf(fmaf(-q, mref, a), yh, q);
        const float di2 = tq * tq;
        sh[k] = fmaf(di2, nh, S);
        const unsigned b = __float_as_uint(sh[k]);
        const float* T = (const float*)((const char*)tab + (b & (4u * kTab - 4u)));
        float f = fmaf(di2, nh, M - __uint_as_float(b & ~3u));
        f = fmaf(di2, nl, f);
        const float p = f * fmaf(f, C2, C1);
        const float s = fmaf(T[0], p, T[kTab]);
        const float h = T[0] + s;
        e[k] = s - (h - T[0]);
        unsigned m = b & ~(4u * kTab - 1u);
        asm("" : "+v"(m));  // shift and add in one instruction
        H[k] = __uint_as_float((m << 8) + __float_as_uint(h));
        emax = fmaxf(emax, fabsf(e[k]));
        smin = __builtin_elementwise_minimum(smin, sh[k]);  // a NaN stays
      }
      if (emax > kKeep || !(smin >= kFar) || all) {
        unsigned left = 0;
        bool mid = false;
#pragma unroll
        for (int k = 0; k < W; k++) {
          const bool under = sh[k] < kUnder, low = !(sh[k] >= kFar) & !under;
          left |= (low | ((fabsf(e[k]) > kKeep) & !under)) ? 1u << k : 0u;
          mid |= low;
          H[k] = under ? 0.f : H[k];
        }
        if (__builtin_amdgcn_ballot_w64(mid)) {
#pragma unroll
          for (int k = 0; k < W; k++) {
            float w;
            const bool low = low_weight(sh[k], H[k], e[k], &w);
            H[k] = low ? w : H[k];
            left &= low ? ~(1u << k) : ~0u;
          }
        }
        // every lane takes its own next neighbour, and with it all that have
        // the same value (a flat background)
        left = (all ? 0x1ffu : left) & vmask;
        while (left) {
          const int k = __builtin_ctz(left);
          const float g = ld_f1(rg, voff + 4u * k, 0);
          const float tq = (g - rv) / mref;
          const float di2 = tq * tq;
          const float w = (float)exp(-(double)di2 / kI);
#pragma unroll
          for (int j = 0; j < W; j++) {
            const bool same = (j == k) | (gv[j] == g);
            H[j] = same ? w : H[j];
            left &= same ? ~(1u << j) : ~0u;
          }
        }
      }
      const int d2 = dz * dz + dy * dy;
      float gk[R + 1] = {gt.g[d2], gt.g[d2 + 1], gt.g[d2 + 4], gt.g[d2 + 9], gt.g[d2 + 16]};
      asm("" : "+v"(gk[0]), "+v"(gk[1]), "+v"(gk[2]), "+v"(gk[3]), "+v"(gk[4]));
#pragma unroll
      for (int k = 0; k < W; k++) {
        if (k <= R || (vmask >> k) & 1u) {
          const float hg = H[k] * gk[k < R ? R - k : k - R];
          norm += hg;
          sum = fmaf(hg, iv[k], sum);
        }
      }
    }
  }
  out[iV] = ((double)norm > 1e-8) ? sum / norm : 0.f;
}

__global__ void k_blend(long long nv, float coef, const float* __restrict__ filt,
                        float* __restrict__ x) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  x[i] = (float)((1.0 - (double)coef) * (double)x[i] + (double)(coef * filt[i]));
}

// max(0, max x): non-negative floats order like their bit patterns.
// 128x128x159: 17 -> 9 us (single words from 1024 blocks before).
__global__ __launch_bounds__(256) void k_max(long long nv, const float* __restrict__ x,
                                             unsigned int* bits) {
  __shared__ unsigned int red[256];
  float m4 = 0.f;
#pragma unroll 4
  for (long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4; i < nv;
       i += (long long)gridDim.x * 1024) {
    const Float4u v = load4(x + i, (int)min(4ll, nv - i));
    m4 = fmaxf(fmaxf(fmaxf(m4, v.x), v.y), fmaxf(v.z, v.w));  // a NaN is passed over
  }
  const unsigned int m = m4 > 0.f ? __float_as_uint(m4) : 0;
  red[threadIdx.x] = m;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] = max(red[threadIdx.x], red[threadIdx.x + w]);
    __syncthreads();
  }
  if (threadIdx.x == 0 && red[0]) atomicMax(bits, red[0]);
}

__global__ void k_fill_cylinder(int res, int nzs, float val, float* __restrict__ img) {
  const int x = blockIdx.x * kWave + threadIdx.x;
  const int y = blockIdx.y * 4 + threadIdx.y;
  const int z = blockIdx.z;
  if (x >= res || y >= res) return;
  const int h = res / 2;
  const long long d = (long long)(x - h) * (x - h) + (long long)(y - h) * (y - h);
  img[((size_t)z * res + y) * res + x] = (d <= (long long)h * h) ? val : 0.f;
}

__global__ void k_zero(uint32_t* __restrict__ p, size_t nwords) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nwords;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

__global__ void k_zero_bytes(uint8_t* __restrict__ p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Creation passes over whole sinograms: 4 bins an item, two items a thread, so
// that they run at the rate of memory (88M bins: the mask 270 -> 133 us, check and
// FP16 storage of the counts 273 -> 80 us).
constexpr int kItems = 512;  // items a block

// fn(first bin, bins) for this thread's items of n bins
template <class Fn>
__device__ __forceinline__ void each_item(long long n, Fn fn) {
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const long long i = ((long long)blockIdx.x * kItems + k * 256 + threadIdx.x) * 4;
    if (i < n) fn(i, (int)min(4ll, n - i));
  }
}
// Calibration mask (GFIRST.cu:453-458). The reference compares in double; a
// float is above 0.01 exactly where it is above the float nearest to it, which
// is smaller.
__global__ __launch_bounds__(256) void k_calib_mask(long long nd, const float* __restrict__ pb,
                                                    const float* __restrict__ norm,
                                                    uint8_t* __restrict__ mask) {
  each_item(nd, [&](long long i, int m) {
    const Float4u a = load4(pb + i, m), b = load4(norm + i, m);
    const uint8_t v[4] = {a.x > 0.01f && b.x > 0.01f, a.y > 0.01f && b.y > 0.01f,
                          a.z > 0.01f && b.z > 0.01f, a.w > 0.01f && b.w > 0.01f};
    if (m == 4 && ((uintptr_t)(mask + i) & 3) == 0) {
      *(uchar4*)(mask + i) = make_uchar4(v[0], v[1], v[2], v[3]);
    } else {
      for (int k = 0; k < m; k++) mask[i + k] = v[k];
    }
  });
}
// Counts into the storage format; *flag = 1 if one is NaN or infinite.
template <int S>
__global__ __launch_bounds__(256) void k_store_checked(const float* __restrict__ in,
                                                       void* __restrict__ out, long long n,
                                                       unsigned int* __restrict__ flag) {
  bool bad = false;
  each_item(n, [&](long long i, int m) {
    const Float4u v = load4(in + i, m);
    const float f[4] = {v.x, v.y, v.z, v.w};
    uint16_t h[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      uint32_t b = __float_as_uint(f[k]);
      const bool out_of_range = (b & 0x7f800000u) == 0x7f800000u;
      bad |= out_of_range;
      if constexpr (S == GFR_STORE_F16) {
        h[k] = __builtin_bit_cast(uint16_t, (_Float16)f[k]);
      } else if constexpr (S == GFR_STORE_BF16) {  // to nearest even; NaN kept quiet
        h[k] = (b & 0x7fffffffu) > 0x7f800000u
                   ? (uint16_t)((b >> 16) | 0x40u)
                   : (uint16_t)((b + 0x7fffu + ((b >> 16) & 1u)) >> 16);
      }
    }
    if constexpr (S == GFR_STORE_F32) {
      if (m == 4) *(Float4u*)((float*)out + i) = v;
      else for (int k = 0; k < m; k++) ((float*)out)[i + k] = f[k];
    } else {
      uint16_t* o = (uint16_t*)out + i;
      if (m == 4) *(uint2*)o = make_uint2(h[0] | (unsigned)h[1] << 16, h[2] | (unsigned)h[3] << 16);
      else for (int k = 0; k < m; k++) o[k] = h[k];
    }
  });
  if (bad) *flag = 1u;
}

// Deterministic final sum of per-block FP64 partials (fixed order).
__global__ void k_llh_final(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// ---------------------------------------------------------------------------
// VLOR (GFIRST.cu:229-247, 373-388).
// ---------------------------------------------------------------------------
// datos_v0 of the touched bins (GFIRST.cu:238-239): the length of a bin's list,
// which the reference counts in float.
__global__ void k_vlor_counts(DevGeom G, const unsigned* __restrict__ bins,
                              const int* __restrict__ start, long long nbins,
                              float* __restrict__ v0) {
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k < nbins) v0[vlor_bin(G, bins[k])] = (float)min(start[k + 1] - start[k], 1 << 24);
}

// The lists of a touched bin (angle-major, vlor_key): per event that names it
// the other bin and valor = BLANKT[i1] + BLANKT[i2] (GFIRST.cu:381), in record
// order, with BLANKT = T/(RES*v0) where v0 > 0.01 (GFIRST.cu:244-247) and T =
// yT * scale. A pass then reads its own angles' lists only, and nothing per event.
__global__ void k_vlor_entries(DevGeom G, const unsigned* __restrict__ bins,
                               const int* __restrict__ start, const int* __restrict__ ev,
                               const int* __restrict__ i1, const int* __restrict__ i2,
                               const float* __restrict__ yT, float scale, float res,
                               const float* __restrict__ v0, long long nbins,
                               int2* __restrict__ ent) {
  const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nbins) return;
  auto blankt = [&](int i) {
    const float val = v0[i];
    return ((double)val > 0.01) ? yT[i] * scale / (res * val) : 0.f;
  };
  const int b = vlor_bin(G, bins[k]);
  for (int j = start[k]; j < start[k + 1]; j++) {
    const int a = i1[ev[j]], c = i2[ev[j]];
    ent[j] = make_int2(a == b ? c : a, __float_as_int(blankt(a) + blankt(c)));
  }
}

// first[c]: the first touched bin of chunk c (angle-major, kVlorChunk bins of
// an angle) or after it; one more entry for the end.
__global__ void k_vlor_first(DevGeom G, const unsigned* __restrict__ bins, long long nbins,
                             int nch, int* __restrict__ first) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c > G.nang * nch) return;
  const unsigned per = (unsigned)(G.nsinogs * G.nrad);
  const unsigned long long key = (unsigned long long)(c / nch) * per + (unsigned)(c % nch) * kVlorChunk;
  long long lo = 0, hi = nbins;
  while (lo < hi) {
    const long long m = (lo + hi) >> 1;
    if (bins[m] < key) lo = m + 1; else hi = m;
  }
  first[c] = (int)lo;
}

// One chunk of one angle per block: the chunk is zeroed in LDS, the touched
// bins' contributions are summed in record order, one thread a bin
// (datos_v[i] += s_i * s_inv * valor with s_inv = 1/(s1+s2) in double, rounded
// to float, GFIRST.cu:384-387), and the whole chunk is written once.
// What bounds it: the chain first -> start -> entry -> projection of the other
// bin, four dependent reads of a block whose ten or so touched bins keep one
// wave busy; the writes (22 MB, 4 us) pass meanwhile. One pass of 860k events at
// 128x160x4319 bins, 16 subsets: 59 -> 12 us; before, every event's 1/(s1+s2)
// was computed in every pass.
__global__ __launch_bounds__(256) void k_vlor_assign(DevGeom G, const unsigned* __restrict__ bins,
                                                     const int* __restrict__ start,
                                                     const int2* __restrict__ ent,
                                                     const int* __restrict__ first, int nch,
                                                     const float* __restrict__ proj,
                                                     float* __restrict__ dv, int subset,
                                                     int nsub) {
  __shared__ float acc[kVlorChunk];
  const int it = subset + (int)blockIdx.y * nsub, c = blockIdx.x, t = threadIdx.x;
  const int per = G.nsinogs * G.nrad, q0 = c * kVlorChunk, n = min(kVlorChunk, per - q0);
  const int k0 = first[it * nch + c], k1 = first[it * nch + c + 1];
  for (int i = t; i < n; i += 256) acc[i] = 0.f;
  __syncthreads();
  for (int k = k0 + t; k < k1; k += 256) {
    const unsigned key = bins[k];
    const float sb = proj[vlor_bin(G, key)];
    float a = 0.f;
    const int j1 = start[k + 1];
    for (int j = start[k]; j < j1; j++) {
      const int2 x = ent[j];
      const float s = sb + proj[x.x];
      const float sinv = (s > 0.01f) ? (float)(1.0 / (double)s) : 0.f;
      a += sb * sinv * __int_as_float(x.y);
    }
    acc[key - (unsigned)(it * per + q0)] = a;
  }
  __syncthreads();
  for (int i = t; i < n; i += 256) {
    const int s = (q0 + i) / G.nrad, r = q0 + i - s * G.nrad;
    dv[((size_t)s * G.nang + it) * G.nrad + r] = acc[i];
  }
}

inline dim3 grid_img(const DevGeom& G, int nz) {
  return dim3((G.res + kWave - 1) / kWave, (G.res + 3) / 4, nz);
}

inline int nav_of(const DevGeom& G, int subset, int nsub) {
  return (G.nang - subset + nsub - 1) / nsub;
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
hipError_t launch_fill_cylinder(const DevGeom& G, float val, float* img, hipStream_t st) {
  hipLaunchKernelGGL(k_fill_cylinder, grid_img(G, G.nzs), dim3(kWave, 4), 0, st, G.res, G.nzs,
                     val, img);
  return hipGetLastError();
}

namespace {
// Advances the subset index of each listed slot: sub = (sub + 1) mod nsub, and
// clears the flag of its packed rows (PackedRows::bad), so that ratios out of
// range slow down the frame's one pass only.
__global__ void k_advance(int* __restrict__ sub, const int* __restrict__ nsub,
                          const int* __restrict__ slots, unsigned* __restrict__ bad, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int s = slots[i];
  const int v = sub[s] + 1;
  sub[s] = v >= nsub[s] ? 0 : v;
  bad[s] = 0u;
}
}  // namespace

namespace {
__global__ __launch_bounds__(256) void k_any_positive(const float* __restrict__ v, long long n,
                                                      unsigned int* __restrict__ flag) {
  bool any = false;
  each_item(n, [&](long long i, int m) {
    const Float4u f = load4(v + i, m);  // zeros past the end
    any |= !(f.x <= 0.f) | !(f.y <= 0.f) | !(f.z <= 0.f) | !(f.w <= 0.f);
  });
  if (any) *flag = 1u;
}
}  // namespace

static dim3 item_blocks(long long n) {
  return dim3((unsigned)((n + 4 * kItems - 1) / (4 * kItems)));
}

hipError_t launch_any_positive(const float* v, long long n, unsigned int* flag, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_any_positive, item_blocks(n), dim3(256), 0, st, v, n, flag);
  return hipGetLastError();
}

hipError_t launch_advance(int* sub, const int* nsub, const int* slots, unsigned* bad, int n,
                          hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_advance, dim3((n + 255) / 256), dim3(256), 0, st, sub, nsub, slots, bad, n);
  return hipGetLastError();
}

hipError_t launch_zero(void* p, size_t bytes, hipStream_t st) {
  if (bytes == 0) return hipSuccess;
  size_t nw = bytes / 4;
  if (nw) {
    size_t blocks = (nw + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, st, (uint32_t*)p, nw);
  }
  size_t rem = bytes - nw * 4;
  if (rem) {
    hipLaunchKernelGGL(k_zero_bytes, dim3(1), dim3(64), 0, st, (uint8_t*)p + nw * 4, rem);
  }
  return hipGetLastError();
}

template <class Src>
hipError_t blur_launch(const DevGeom& G, const Taps9& t, Src src, float* out, hipStream_t st) {
  const size_t lds = sizeof(float) * ((size_t)kBlurRows * blur_stride(G.res) +
                                     (Src::kStage ? (size_t)(kBlurRows + 8) * G.res : 0));
  if (sizeof(float) * (size_t)(2 * kBlurRows + 8) * G.res > 160 * 1024) return hipErrorInvalidValue;
  dim3 grid((G.res + kBlurRows - 1) / kBlurRows, G.nzs);
  hipLaunchKernelGGL(k_blur_xy<Src>, grid, dim3(256), lds, st, G.res, G.nzs, t, src, out);
  return hipGetLastError();
}

hipError_t launch_blur_xy(const DevGeom& G, const Taps9& t, const float* in, float* out,
                          hipStream_t st) {
  return blur_launch(G, t, SrcPlain{in}, out, st);
}

hipError_t launch_ratio(const DevGeom& G, const float* proj, const float* y, const void* bg,
                        int storage, float yscale, float* corr, const PackedRows& P,
                        const uint8_t* mask, int subset, int nsub, hipStream_t st) {
  const int nav = nav_of(G, subset, nsub);
  const dim3 grid((unsigned)((G.nsinogs * ((G.nrad + 3) / 4) + 255) / 256), nav);
  if (storage == GFR_STORE_F16)
    hipLaunchKernelGGL(k_ratio<GFR_STORE_F16>, grid, dim3(256), 0, st, G, proj, y, bg,
                       yscale, corr, P, mask, subset, nsub);
  else if (storage == GFR_STORE_BF16)
    hipLaunchKernelGGL(k_ratio<GFR_STORE_BF16>, grid, dim3(256), 0, st, G, proj, y, bg,
                       yscale, corr, P, mask, subset, nsub);
  else
    hipLaunchKernelGGL(k_ratio<GFR_STORE_F32>, grid, dim3(256), 0, st, G, proj, y, bg,
                       yscale, corr, P, mask, subset, nsub);
  return hipGetLastError();
}

hipError_t launch_calib_mask(const DevGeom& G, const float* pb, const float* norm,
                             uint8_t* mask, hipStream_t st) {
  const long long nd = G.ndata;
  hipLaunchKernelGGL(k_calib_mask, item_blocks(nd), dim3(256), 0, st, nd, pb, norm, mask);
  return hipGetLastError();
}

hipError_t launch_update(const DevGeom& G, const Taps9& t9, const Taps5& t5, const float* numer,
                         const float* denom, float* x, float* work, hipStream_t st) {
  hipError_t e = denom ? blur_launch(G, t9, SrcRatio{numer, denom}, work, st)
                       : blur_launch(G, t9, SrcPlain{numer}, work, st);
  if (e != hipSuccess) return e;
  if (G.nzs >= 3)
    hipLaunchKernelGGL(k_gz_mul, dim3((G.res * G.res + 1023) / 1024, G.nzs - 2), dim3(256), 0, st,
                       G.res, G.nzs, t5, work, x);
  return hipGetLastError();
}

hipError_t launch_jbf(const DevGeom& G, const float* in, const float* guide,
                      const float* d_max_ref, float max_ref, int r, float s3d, float sI,
                      float* out, hipStream_t st) {
  GTab gt;
  const double kS = (2.0 * (double)s3d) * (2.0 * (double)s3d);
  for (int d2 = 0; d2 < 193; d2++) gt.g[d2] = (float)exp(-(double)(float)d2 / kS);
  const double kI = (2.0 * (double)sI) * (2.0 * (double)sI);
  // the radius-4 kernel addresses the volume with 32-bit byte offsets
  if (r == 4 && G.nvox < (1ll << 29))
  {
    const long long items = (long long)(G.res - 4) * (G.res - 4);
    const unsigned gx = G.res > 4 ? (unsigned)((items + jbfx::kThreads - 1) / jbfx::kThreads) : 1u;
    const double nki = -jbfx::kTab / jbfx::kLn2 / kI;
    const float nh = (float)nki;
    hipLaunchKernelGGL(k_jbf_r4, dim3(gx, G.nzs), dim3(jbfx::kThreads), 0, st, G.res, G.nzs, in,
                       guide, d_max_ref, max_ref, kI, nh, (float)(nki - nh), gt, out);
  } else {
    hipLaunchKernelGGL(k_jbf, grid_img(G, G.nzs), dim3(kWave, 4), 0, st, G.res, G.nzs, in,
                       guide, d_max_ref, max_ref, r, kI, gt, out);
  }
  return hipGetLastError();
}

hipError_t launch_blend(const DevGeom& G, float coef, const float* filt, float* x,
                        hipStream_t st) {
  const long long nv = G.nvox;
  hipLaunchKernelGGL(k_blend, dim3((unsigned)((nv + 255) / 256)), dim3(256), 0, st, nv, coef,
                     filt, x);
  return hipGetLastError();
}

hipError_t launch_max(const DevGeom& G, const float* x, unsigned int* d_bits, hipStream_t st) {
  hipError_t e = launch_zero(d_bits, 4, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_max, dim3(512), dim3(256), 0, st, G.nvox, x, d_bits);
  return hipGetLastError();
}

hipError_t launch_store_checked(const float* in, void* out, int storage, long long n,
                                unsigned int* flag, hipStream_t st) {
  const dim3 grid = item_blocks(n);
  if (storage == GFR_STORE_F32)
    hipLaunchKernelGGL(k_store_checked<GFR_STORE_F32>, grid, dim3(256), 0, st, in, out, n, flag);
  else if (storage == GFR_STORE_F16)
    hipLaunchKernelGGL(k_store_checked<GFR_STORE_F16>, grid, dim3(256), 0, st, in, out, n, flag);
  else
    hipLaunchKernelGGL(k_store_checked<GFR_STORE_BF16>, grid, dim3(256), 0, st, in, out, n, flag);
  return hipGetLastError();
}

hipError_t launch_llh_final(const double* part, int n, double* out, hipStream_t st) {
  hipLaunchKernelGGL(k_llh_final, dim3(1), dim3(256), 0, st, part, n, out);
  return hipGetLastError();
}

hipError_t launch_vlor_lists(const DevGeom& G, const unsigned* bins, const int* start,
                             const int* ev, const int* i1, const int* i2, const float* yT,
                             float scale, float res, float* v0, long long nbins, int2* ent,
                             int* first, hipStream_t st) {
  if (nbins) {
    const dim3 grid((unsigned)((nbins + 255) / 256));
    hipLaunchKernelGGL(k_vlor_counts, grid, dim3(256), 0, st, G, bins, start, nbins, v0);
    hipLaunchKernelGGL(k_vlor_entries, grid, dim3(256), 0, st, G, bins, start, ev, i1, i2, yT,
                       scale, res, v0, nbins, ent);
  }
  const int nch = vlor_chunks(G);
  hipLaunchKernelGGL(k_vlor_first, dim3((G.nang * nch + 256) / 256), dim3(256), 0, st, G, bins,
                     nbins, nch, first);
  return hipGetLastError();
}

hipError_t launch_vlor_assign(const DevGeom& G, const unsigned* bins, const int* start,
                              const int2* ent, const int* first, const float* proj, float* dv,
                              int subset, int nsub, hipStream_t st) {
  const int nch = vlor_chunks(G);
  hipLaunchKernelGGL(k_vlor_assign, dim3(nch, nav_of(G, subset, nsub)), dim3(256), 0, st, G, bins,
                     start, ent, first, nch, proj, dv, subset, nsub);
  return hipGetLastError();
}

}  // namespace gfr
