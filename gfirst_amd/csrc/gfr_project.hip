// gfr_project.hip — the forward projector of the OSEM path on gfx950, the packed
// rows that the backprojector (gfr_back_window.hip) reads, the FP64 sensitivity
// and the autotuner of both projectors.
//
// Forward projection (FORWPROJ_K, GFIRST_GPU_Kernels.cu:40-102): a LOR of view
// (segment, angle theta), plane p, radial bin r sums RES+1 trilinear samples of
// the blurred image at (xc + l dx, yc + l dy, p + 0.5 + l dz). The x/y sample
// positions depend only on (theta, r, l); only z depends on the segment and
// plane. Trilinear = lerp_z(bilinear_xy(plane z0), bilinear_xy(plane z1)), so
// the kernel pair below computes every bilinear value once per angle:
//   k_rotate_tile: R[a][l][z][r] = bilinear_xy(image plane z, x(theta,r,l), y(theta,r,l))
//   k_zsum_*     : P(s, r) = sum_l lerp(R[a][l][z0][r], R[a][l][z1][r], alpha_z)
// which is the same arithmetic, operation for operation, as sampling the
// volume directly (bit-identical results). The z interpolation of sinogram s
// at sample l, (z0, z1, alpha_z), is a per-geometry table.
#include <algorithm>

#include "gfr_device.h"

namespace gfr {

namespace {

// ---------------------------------------------------------------------------
// k_rotate_tile: R[a][l][z][r], the bilinear sample of image plane z at the
// position of (bin r, sample l) of angle a. A block takes one angle, a tile
// of 32 bins x up to 40 samples and ZC planes (autotuned). The tile's sample
// points fall in a rotated rectangle of the image; since x and y (and then
// the clamped texel indices) are monotone in r and l, the texels the tile
// touches lie in the bounding box of its four corner samples. Per pair of
// planes the block copies that box into LDS with coalesced row loads, the two
// planes side by side (the next pair's rows are in flight while the current
// one is used), and every output reads its four texels of both planes from
// LDS. A box larger than the LDS tile (coarse geometries) falls back to
// gathers from global memory.
// What bounds it: the loads and barriers of a plane, not bytes or arithmetic;
// two planes a turn halve them, and tiles of equal height (129 samples in four
// tiles of 33 instead of 32 + 32 + 32 + 32 + 1) save a fifth of the blocks:
// 10 angles at 128x128x159 59 -> 35 us, 16 at 147x147x239 84 -> 55 us (write
// floors at the rate of a large copy, 16 and 32 us).
// ---------------------------------------------------------------------------
constexpr int kRotTile = 64;  // largest LDS box: texels per row and rows
constexpr int kRotOut = 5;    // samples per thread: tiles of up to 40

// Samples per tile: as few tiles as tiles of up to 40 give, of equal height.
__host__ __device__ inline int rot_tile_samples(int nl) {
  const int n = (nl + 8 * kRotOut - 1) / (8 * kRotOut);
  return (nl + n - 1) / n;
}

template <int ZC>
__global__ __launch_bounds__(256) void k_rotate_tile(DevGeom G, const float* __restrict__ img,
                                                     float* __restrict__ R, int subset, int nsub,
                                                     const int* __restrict__ dsub, int a0,
                                                     int nl, int zouter, int side) {
  extern __shared__ float2 box[];  // side rows of side | 1 texels (odd: rows on different banks)
  const int stride = side | 1;
  if (dsub) subset = *dsub;
  // Logical order: bin tile, sample tile, then angle and plane chunk; every
  // XCD walks one contiguous range of logical blocks. With zouter the plane
  // chunk is outermost: an XCD rotates a few plane chunks for every angle
  // and reads each image plane once into its L2 (rotation outputs larger than
  // an L2). Otherwise the angle is: an XCD writes the angles whose z-sum blocks
  // it reads next, while they are still in its L2.
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int tl = rot_tile_samples(nl);
  const unsigned nrt = (G.nrad + 31) / 32, nlt = (nl + tl - 1) / tl;
  const unsigned nzc = (G.nzs + ZC - 1) / ZC;
  const unsigned na = gridDim.x / (nrt * nlt * nzc);
  const unsigned rt = b % nrt;
  unsigned q = b / nrt;
  const unsigned lt = q % nlt;
  q /= nlt;
  const int a = (int)(zouter ? q % na : q / nzc);
  const int zc = (int)(zouter ? q / na : q % nzc) * ZC;
  if (a0 + a >= (G.nang - subset + nsub - 1) / nsub) return;  // whole block
  const int it = subset + (a0 + a) * nsub;
  const float st = G.sin_t[it], ct = G.cos_t[it];
  const int tid = threadIdx.x;
  // texels and weights of sample (r, li)
  auto texels = [&](int r, int li, int& x0i, int& x1i, float& ax, int& y0i, int& y1i,
                    float& ay) {
    const float x0 = G.fxf * ((float)r - G.RADM);
    const float xc = fmaf(x0, ct, G.RESM) + 0.5f;
    const float yc = fmaf(x0, st, G.RESM) + 0.5f;
    const float fl = (float)(G.l0 + li);
    axis(fmaf(fl, st, xc), G.res, x0i, x1i, ax);   // dx = sin(theta) (GFIRST_GPU_Kernels.cu:81)
    axis(fmaf(fl, -ct, yc), G.res, y0i, y1i, ay);  // dy = -cos(theta) (:82)
  };
  const int rlo = (int)rt * 32, rhi = min(rlo + 31, G.nrad - 1);
  const int llo = (int)lt * tl, lhi = min(llo + tl, nl) - 1;
  int bx0 = G.res, bx1 = -1, by0 = G.res, by1 = -1;
#pragma unroll
  for (int c = 0; c < 4; c++) {
    int x0i, x1i, y0i, y1i;
    float ax, ay;
    texels(c & 1 ? rhi : rlo, c & 2 ? lhi : llo, x0i, x1i, ax, y0i, y1i, ay);
    bx0 = min(bx0, x0i);
    bx1 = max(bx1, x1i);
    by0 = min(by0, y0i);
    by1 = max(by1, y1i);
  }
  const int bw = bx1 - bx0 + 1, bh = by1 - by0 + 1;
  const bool staged = bw <= side && bh <= side;
  // this thread's outputs: bin rlo + (tid & 31), samples llo + (tid >> 5) + 8k
  const int r = rlo + (tid & 31);
  int o00[kRotOut], dx[kRotOut], dy[kRotOut];
  float ax[kRotOut], ay[kRotOut];
  bool ok[kRotOut];
#pragma unroll
  for (int k = 0; k < kRotOut; k++) {
    const int li = llo + (tid >> 5) + 8 * k;
    ok[k] = r < G.nrad && li <= lhi;
    int x0i, x1i, y0i, y1i;
    texels(r, min(li, lhi), x0i, x1i, ax[k], y0i, y1i, ay[k]);
    const int w = staged ? stride : G.res;
    o00[k] = staged ? (y0i - by0) * w + (x0i - bx0) : y0i * w + x0i;
    dx[k] = x1i - x0i;
    dy[k] = (y1i - y0i) * w;
  }
  const size_t plane = (size_t)G.res * G.res;
  const int nz = min(ZC, G.nzs - zc);
  float* out = R + (((size_t)a * nl + llo + (tid >> 5)) * G.nzs + zc) * G.nrad + r;
  const size_t lstep = (size_t)8 * G.nzs * G.nrad;  // 8 samples further
  if (!staged) {
    for (int zi = 0; zi < nz; zi++) {
      const float* pk = img + (size_t)(zc + zi) * plane;
#pragma unroll
      for (int k = 0; k < kRotOut; k++) {
        if (ok[k]) {
          const float* p = pk + o00[k];
          out[k * lstep + (size_t)zi * G.nrad] =
              lerp1(lerp1(p[0], p[dx[k]], ax[k]), lerp1(p[dy[k]], p[dy[k] + dx[k]], ax[k]), ay[k]);
        }
      }
    }
    return;
  }
  // box loader: thread copies column tid & 63 of rows tid / 64 + 4 j
  const int lc = tid & 63, lr = tid >> 6;
  const int nj = (bh + 3) >> 2;
  const float* src = img + (size_t)(by0 + lr) * G.res + bx0 + lc;
  float2 pre[kRotTile / 4];
  auto fetch = [&](int z) {  // planes z and z + 1 (the last one again past the end)
    const float* p0 = src + (size_t)z * plane;
    const float* p1 = src + (size_t)min(z + 1, G.nzs - 1) * plane;
#pragma unroll
    for (int j = 0; j < kRotTile / 4; j++)
      if (j < nj && lc < bw && lr + 4 * j < bh) {
        const size_t o = (size_t)(4 * j) * G.res;
        pre[j] = make_float2(p0[o], p1[o]);
      }
  };
  fetch(zc);
  for (int zi = 0; zi < nz; zi += 2) {
    __syncthreads();  // the previous planes' reads are done
#pragma unroll
    for (int j = 0; j < kRotTile / 4; j++)
      if (j < nj && lc < bw && lr + 4 * j < bh) box[(lr + 4 * j) * stride + lc] = pre[j];
    __syncthreads();
    if (zi + 2 < nz) fetch(zc + zi + 2);
    const bool two = zi + 1 < nz;
#pragma unroll
    for (int k = 0; k < kRotOut; k++) {
      if (ok[k]) {
        const float2* p = box + o00[k];
        const float2 v00 = p[0], v01 = p[dx[k]], v10 = p[dy[k]], v11 = p[dy[k] + dx[k]];
        float* w = out + k * lstep + (size_t)zi * G.nrad;
        w[0] = lerp1(lerp1(v00.x, v01.x, ax[k]), lerp1(v10.x, v11.x, ax[k]), ay[k]);
        if (two)
          w[G.nrad] = lerp1(lerp1(v00.y, v01.y, ax[k]), lerp1(v10.y, v11.y, ax[k]), ay[k]);
      }
    }
  }
}

// Where the forward kernel writes.
struct FwdArgs {
  float* proj;           // full sinogram layout, or NULL
  float* corr;           // full layout ratio, or NULL
  PackedRows rows;       // packed rows of the subset (v NULL: not written)
  const uint8_t* mask;   // calibration mask (full layout) for rows
  const void* y;         // measured prompts (storage format), unscaled
  const void* bg;        // background or NULL
  float yscale;          // RES (GFIRST.cu:224-260)
  double* llh_part;      // per-block FP64 partial log-likelihoods, or NULL
};

// ---------------------------------------------------------------------------
// z-sums: every LOR of sinogram s, angle a, bin r sums its samples in l order,
// each the lerp of two rows of R with the sample's weight.
// Epilogue per LOR: projection, ratio (GFIRST.cu:415-430), packed row, and the
// FP64 Poisson log-likelihood partial of the block (bins with valid calibration
// and den >= 0.01: sum of (y/RES) ln(den/RES) - den/RES; the reference computes
// no likelihood).
// ---------------------------------------------------------------------------
// N <= 4 consecutive bins r .. of sinogram s, angle it (ag of the subset).
template <int S, bool RATIO, bool LLH>
__device__ __forceinline__ void emit(const DevGeom& G, const FwdArgs& o, int s, int ag, int it,
                                     int r, int N, const float (&p)[4], double& ll) {
  const size_t bin0 = ((size_t)s * G.nang + it) * G.nrad + r;
  float c[4];
  bool valid[4];
#pragma unroll
  for (int h = 0; h < 4; h++) {
    c[h] = 0.f;
    valid[h] = true;
    if (h >= N) continue;
    const size_t bin = bin0 + h;
    if (o.proj) o.proj[bin] = p[h];
    if constexpr (RATIO) {
      const float yv = o.yscale * load_store<S>(o.y, bin);
      float bv = o.bg ? o.yscale * load_store<S>(o.bg, bin) : 0.f;
      if (bv < 0.f) bv = 0.f;
      const float den = p[h] + bv;
      c[h] = (den >= 0.01f) ? yv / den : -1000.f;
      if (o.mask) valid[h] = o.mask[bin] != 0;
      if (o.corr) o.corr[bin] = c[h];
      if constexpr (LLH) {
        // Poisson log-likelihood in count units over the bins whose ratio
        // enters the backprojection: model mean den/RES, counts yv/RES (yv
        // and den as the ratio sees them).
        if (den >= 0.01f && valid[h]) {
          const double m = (double)den / (double)o.yscale;
          ll += ((double)yv / (double)o.yscale) * log(m) - m;
        }
      }
    }
  }
  if constexpr (RATIO) {
    if (o.rows.v && N > 0) store_packed(G, o.rows, ag, s, r, N, c, valid);
  }
}

template <bool LLH>
__device__ __forceinline__ void block_llh(double ll, double* part) {
  if constexpr (LLH) {
    __shared__ double red[256];
    const int t = threadIdx.x;
    red[t] = ll;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if (t < w) red[t] += red[t + w];
      __syncthreads();
    }
    if (t == 0) *part = red[0];
  }
}

// Wide waves: one wave per (64 quads of bins, group of SG planes of a segment).
// Its lanes are consecutive (angle, 4 bins) items, so a row load is one 16-byte
// access per lane and a wave is full whatever the bin count; the SG LORs of a
// lane share SG + 1 rows. Row and weights of a sample are wave-uniform (scalar
// loads, one sample ahead). The four waves of a block take the same planes of
// four neighbouring segments, which blend nearly the same rows, so L1 serves
// three of them. Groups whose LORs do not blend consecutive rows in every
// sample (at the volume's ends) load each LOR's two rows.
// What bounds it: the vector-memory path (16 cycles a row load) and the L2
// misses of the rotation. 10 angles of 4319 x 128 LORs with ratio: 190 -> 145 us,
// 16 angles of 1293 x 147: 150 -> 130 us (waves of two angles, half empty at 147
// bins, with scalar table reads per LOR before).
template <int S, bool RATIO, bool LLH, int SG>
__global__ __launch_bounds__(256) void k_zsum_wide(DevGeom G, const float* __restrict__ R,
                                                   unsigned r_bytes, FwdArgs o, int subset,
                                                   int nsub, const int* __restrict__ dsub, int a0,
                                                   int na, int nl, unsigned llh_off) {
  if (dsub) subset = *dsub;
  const ZGroups zg = G.zg[zg_index(SG)];
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int nq = (G.nrad + 3) / 4, ngb = (zg.n + 3) / 4;
  const int ib = (int)(b / (unsigned)ngb), gb = (int)(b % (unsigned)ngb);
  const int nav = (G.nang - subset + nsub - 1) / nsub;
  if (a0 + ib * 64 / nq >= nav) return;  // whole block: no angle of the subset
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int item = ib * 64 + (int)(threadIdx.x & 63);
  const int a = item / nq, r = 4 * (item - a * nq);
  const int ag = a0 + a, it = subset + ag * nsub;
  const int gi = gb * 4 + wv;
  double ll = 0.0;
  const int2 grp = zg.s[gi];  // zg.n is a multiple of 4
  const int ng = grp.y < 0 ? -grp.y : grp.y;
  if (ng > 0) {
    const __amdgpu_buffer_rsrc_t rr = rsrc(R, r_bytes);
    const unsigned rowb = (unsigned)G.nrad * 4u;
    const unsigned planeb = rowb * (unsigned)G.nzs;
    // Lanes past the chunk's angles read past r_bytes: zeros, unused.
    const unsigned voff = (unsigned)a * (unsigned)nl * planeb + (unsigned)r * 4u;
    float4 acc[SG];
#pragma unroll
    for (int i = 0; i < SG; i++) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [&](float4& c, const float4& v0, const float4& v1, float al) {
      c.x += lerp1(v0.x, v1.x, al);
      c.y += lerp1(v0.y, v1.y, al);
      c.z += lerp1(v0.z, v1.z, al);
      c.w += lerp1(v0.w, v1.w, al);
    };
    const uint32_t* rows = zg.row + gi;
    const float* wts = G.za + grp.x;
    unsigned soff = 0;
    if (grp.y > 0) {
      float e[SG];
      unsigned roff[SG + 1];
#pragma unroll
      for (int k = 0; k <= SG; k++) {
        roff[k] = (unsigned)zg_row(k, ng) * rowb;
        asm("" : "+s"(roff[k]));  // one addition a row, not a product
      }
      uint32_t z = rows[0];
#pragma unroll
      for (int i = 0; i < SG; i++) e[i] = wts[i];
      for (int li = 0; li < nl; li++, soff += planeb) {
        const unsigned base = soff + z * rowb;
        float4 row[SG + 1];
#pragma unroll
        for (int k = 0; k <= SG; k++) row[k] = ld_f4(rr, voff, base + roff[k]);
        float en[SG];
        if (li + 1 < nl) {  // the next sample's, while the rows come
          rows += zg.n;
          wts += G.nsinogs;
        }
        z = rows[0];
#pragma unroll
        for (int i = 0; i < SG; i++) en[i] = wts[i];
#pragma unroll
        for (int i = 0; i < SG; i++) add(acc[i], row[i], row[i + 1], e[i]);
#pragma unroll
        for (int i = 0; i < SG; i++) e[i] = en[i];
      }
    } else {
      for (int li = 0; li < nl; li++, soff += planeb) {
        const uint2* t = G.ztab + (size_t)li * G.nsinogs + grp.x;
#pragma unroll
        for (int i = 0; i < SG; i++) {
          const uint2 q = t[i < ng ? i : 0];
          add(acc[i], ld_f4(rr, voff, soff + (q.x & 0xffffu) * rowb),
              ld_f4(rr, voff, soff + (q.x >> 16) * rowb), __uint_as_float(q.y));
        }
      }
    }
    if (a < na && ag < nav) {
      const int N = min(4, G.nrad - r);
#pragma unroll
      for (int i = 0; i < SG; i++) {
        if (i >= ng) break;
        const float p[4] = {acc[i].x, acc[i].y, acc[i].z, acc[i].w};
        emit<S, RATIO, LLH>(G, o, grp.x + i, ag, it, r, N, p, ll);
      }
    }
  }
  block_llh<LLH>(ll, o.llh_part + llh_off + b);
}

// Narrow waves for small sinograms, where a few hundred wide waves would each
// walk the samples one memory round trip at a time: one wave per (64 bins of
// consecutive angles, 2 sinograms), the rows of 4 samples requested together.
template <int S, bool RATIO, bool LLH>
__global__ __launch_bounds__(256) void k_zsum_narrow(DevGeom G, const float* __restrict__ R,
                                                     unsigned r_bytes, FwdArgs o, int subset,
                                                     int nsub, const int* __restrict__ dsub,
                                                     int a0, int na, int nl, unsigned llh_off) {
  constexpr int LA = 4;
  if (dsub) subset = *dsub;
  const unsigned b = xcd_remap(blockIdx.x, gridDim.x);
  const int ngb = (G.nsinogs + 7) / 8;
  const int ib = (int)(b / (unsigned)ngb), gb = (int)(b % (unsigned)ngb);
  const int nav = (G.nang - subset + nsub - 1) / nsub;
  if (a0 + ib * 64 / G.nrad >= nav) return;  // whole block: no angle of the subset
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int item = ib * 64 + (int)(threadIdx.x & 63);
  const int a = item / G.nrad, r = item - a * G.nrad;
  const int ag = a0 + a, it = subset + ag * nsub;
  const int s0 = 2 * (gb * 4 + wv);
  double ll = 0.0;
  if (s0 < G.nsinogs) {
    const int s1 = min(s0 + 1, G.nsinogs - 1);
    const __amdgpu_buffer_rsrc_t rr = rsrc(R, r_bytes);
    const unsigned rowb = (unsigned)G.nrad * 4u;
    const unsigned planeb = rowb * (unsigned)G.nzs;
    const unsigned voff = (unsigned)a * (unsigned)nl * planeb + (unsigned)r * 4u;
    float p0 = 0.f, p1 = 0.f;
    uint2 e0[LA], e1[LA];
    auto entries = [&](int l0) {
#pragma unroll
      for (int u = 0; u < LA; u++) {
        const uint2* t = G.ztab + (size_t)min(l0 + u, nl - 1) * G.nsinogs;
        e0[u] = t[s0];
        e1[u] = t[s1];
      }
    };
    float v[LA][4];
    auto load = [&](int l0) {
#pragma unroll
      for (int u = 0; u < LA; u++) {
        const unsigned so = (unsigned)min(l0 + u, nl - 1) * planeb;
        v[u][0] = ld_f1(rr, voff, so + (e0[u].x & 0xffffu) * rowb);
        v[u][1] = ld_f1(rr, voff, so + (e0[u].x >> 16) * rowb);
        v[u][2] = ld_f1(rr, voff, so + (e1[u].x & 0xffffu) * rowb);
        v[u][3] = ld_f1(rr, voff, so + (e1[u].x >> 16) * rowb);
      }
    };
    entries(0);
    for (int l0 = 0; l0 < nl; l0 += LA) {
      load(l0);
      float w0[LA], w1[LA];
#pragma unroll
      for (int u = 0; u < LA; u++) {
        w0[u] = __uint_as_float(e0[u].y);
        w1[u] = __uint_as_float(e1[u].y);
      }
      if (l0 + LA < nl) entries(l0 + LA);
#pragma unroll
      for (int u = 0; u < LA; u++) {
        if (l0 + u < nl) {
          p0 += lerp1(v[u][0], v[u][1], w0[u]);
          p1 += lerp1(v[u][2], v[u][3], w1[u]);
        }
      }
    }
    if (a < na && ag < nav) {
      const float q0[4] = {p0, 0.f, 0.f, 0.f}, q1[4] = {p1, 0.f, 0.f, 0.f};
      emit<S, RATIO, LLH>(G, o, s0, ag, it, r, 1, q0, ll);
      if (s0 + 1 < G.nsinogs) emit<S, RATIO, LLH>(G, o, s0 + 1, ag, it, r, 1, q1, ll);
    }
  }
  block_llh<LLH>(ll, o.llh_part + llh_off + b);
}

// The z-sum's weights and rows by themselves, from the table of samples, and the
// groups' marks: a wave then reads 4 bytes a LOR and 4 a group in a sample, not 8
// a LOR. On the device, since the host took a third as long again for them as
// for the table itself (128x128x159 voxels, 4319 sinograms: 2.5 -> 3.5 ms).
struct GroupTables {
  int2* s[3];
  uint32_t* row[3];
};
__global__ __launch_bounds__(256) void k_zsum_tables(DevGeom G, float* __restrict__ za,
                                                     GroupTables o) {
  const int i = blockIdx.x * 256 + threadIdx.x, li = blockIdx.y;
  const uint2* t = G.ztab + (size_t)li * G.nsinogs;
  if (i < G.nsinogs) za[(size_t)li * G.nsinogs + i] = __uint_as_float(t[i].y);
  if (li == 0 && i < kZPad) za[(size_t)gridDim.y * G.nsinogs + i] = 0.f;
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const int n = G.zg[j].n;
    if (i >= n) continue;
    int2* const e = o.s[j] + i;
    const int first = e->x, len = abs(e->y);  // marked or not meanwhile
    o.row[j][(size_t)li * n + i] = t[first].x & 0xffffu;
    if (!zg_regular(t + first, len)) e->y = -len;
  }
}

// Full-layout ratio + byte mask -> packed rows of a subset.
__global__ void k_pack(DevGeom G, const float* __restrict__ corr, const uint8_t* __restrict__ mask,
                       PackedRows P, int subset, int nsub) {
  const int r = blockIdx.x * kWave + threadIdx.x;
  const int s = blockIdx.y * 4 + threadIdx.y;
  const int a = blockIdx.z;
  if (r >= G.nrad || s >= G.nsinogs) return;
  const size_t bin = ((size_t)s * G.nang + subset + a * nsub) * G.nrad + r;
  const float c[4] = {corr[bin], 0.f, 0.f, 0.f};
  const bool valid[4] = {mask[bin] != 0, true, true, true};
  store_packed(G, P, a, s, r, 1, c, valid);
}

// Byte mask -> {1, calib} pairs of a subset.
__global__ void k_pack_calib(DevGeom G, const uint8_t* __restrict__ mask, float2* __restrict__ c2,
                             int subset, int nsub) {
  const int r = blockIdx.x * kWave + threadIdx.x;
  const int s = blockIdx.y * 4 + threadIdx.y;
  const int a = blockIdx.z;
  if (r >= G.nrad || s >= G.nsinogs) return;
  const size_t bin = ((size_t)s * G.nang + subset + a * nsub) * G.nrad + r;
  store_calib(G, c2, a, s, r, make_float2(1.f, mask[bin] ? 1.f : -1000.f));
}

// ---------------------------------------------------------------------------
// FP64 sensitivity: the denominator half of the backprojector (BACKWPROJ_K,
// GFIRST_GPU_Kernels.cu:112-160; gfr_back_window.hip has the pair of sums): per
// voxel and view, bilinear (radial bin, plane) interpolation of {1, calib}
// pairs, the -1000 gap rule, sums over views in the reference's order (segments
// outer, angles inner, GFIRST.cu:439-467).
// ---------------------------------------------------------------------------
// Per-lane state of one view.
struct LaneView {
  float yr, w0, wl, s0, au;
  int iq;      // clamp(floor(u - 0.5), -1, NRAD-1): packed entry pair at iq + 1
  bool any;
};

__device__ __forceinline__ LaneView lane_view(const DevGeom& G, float xv, float yv, float st,
                                              float ct, float fzb, float fz0, float fzl,
                                              float fzm, float fzhi, bool act) {
  LaneView v;
  v.yr = fmaf(yv, ct, -(xv * st));
  v.s0 = fmaf(v.yr, fzb, fz0);
  const float sl = fmaf(v.yr, fzb, fzl);
  v.w0 = v.s0 + 0.5f;
  v.wl = sl + 0.5f;
  v.any = act && v.wl >= fzm && v.w0 < fzhi;
  const float xr = fmaf(yv, st, xv * ct);
  const float u = fmaf(xr, G.fxb, G.RADM) + 0.5f;
  const float t = u - 0.5f;
  const float f = floorf(t);
  const int i = (int)f;
  v.au = t - f;
  v.iq = min(max(i, -1), G.nrad - 1);
  return v;
}

// Accumulates one view into n[], d[]. The fetcher returns the {ratio, calib}
// entries of this lane's two bins (r0, r1) of a plane: rows(i0) selects
// planes i0 .. i0 + ZB, pair(k, a0, a1) reads plane i0 + k, get2(ii, a0, a1)
// any plane.
template <int ZB, class F, class T>
__device__ __forceinline__ void accumulate_view(const LaneView& v, float fzb, float yr, int zb,
                                                int nzs, float fzm, float fzhi, F& fetch, T* n,
                                                T* d) {
  // Shared z axis. Slice j samples plane position w_j = fl(fl(P + zb + j) + 0.5)
  // with P = yr * fzb exact inside the fma. When s0 = fl(P + zb) >= 1 and
  // w_{ZB-1} lie in one binade [2^E, 2^(E+1)), every exact sum P + zb + j
  // (j >= 1) lies in that binade too and rounds on its grid (ulp <= 2^-16, so
  // integer shifts keep the nearest point and the tie parity): fl(P + zb + j) =
  // s0 + j, w_j = s0 + j + 0.5 and t_j = w_j - 0.5 = s0 + j exactly. Then all
  // slices share alpha = s0 - floor(s0) and take planes floor(s0) + j, j + 1.
  const bool slow = v.any && !(v.s0 >= 1.f && (__float_as_uint(v.s0) >> 23) ==
                                                   (__float_as_uint(v.wl) >> 23));
  if (__builtin_amdgcn_ballot_w64(slow) == 0) {
    const float f0 = floorf(v.s0);
    const float al = v.s0 - f0;
    const int i0 = (int)f0;
    float c[ZB + 1], q[ZB + 1];
    fetch.rows(i0);
#pragma unroll
    for (int k = 0; k <= ZB; k++) {
      float2 a0, a1;
      fetch.pair(k, a0, a1);
      c[k] = lerp1(a0.x, a1.x, v.au);
      q[k] = lerp1(a0.y, a1.y, v.au);
    }
#pragma unroll
    for (int j = 0; j < ZB; j++) {
      const float wj = v.w0 + (float)j;  // exact, see above
      const float A = lerp1(c[j], c[j + 1], al);
      const float B = lerp1(q[j], q[j + 1], al);
      // in range and not a gap (GFIRST_GPU_Kernels.cu:157)
      const bool ok =
          v.any && (zb + j < nzs) && wj >= fzm && wj < fzhi && !(B < 0.f) && !(A < 0.f);
      n[j] += ok ? (T)A : (T)0;
      d[j] += ok ? (T)B : (T)0;
    }
    return;
  }
  // General case: one plane position per slice, as the reference computes it.
  float al[ZB];
  int ii[ZB];
  bool inr[ZB];
#pragma unroll
  for (int j = 0; j < ZB; j++) {
    const float w = (j == 0) ? v.w0 : (j == ZB - 1) ? v.wl : fmaf(yr, fzb, (float)(zb + j)) + 0.5f;
    inr[j] = v.any && (zb + j < nzs) && w >= fzm && w < fzhi;
    const float t = w - 0.5f;
    const float f = floorf(t);
    al[j] = t - f;
    ii[j] = (int)f;
  }
  bool reg = true;
#pragma unroll
  for (int j = 1; j < ZB; j++) reg = reg && (!inr[j] || ii[j] == ii[0] + j);
  float av[ZB], bv[ZB];
  if (reg) {
    float c[ZB + 1], q[ZB + 1];
    fetch.rows(ii[0]);
#pragma unroll
    for (int k = 0; k <= ZB; k++) {
      float2 a0, a1;
      fetch.pair(k, a0, a1);
      c[k] = lerp1(a0.x, a1.x, v.au);
      q[k] = lerp1(a0.y, a1.y, v.au);
    }
#pragma unroll
    for (int j = 0; j < ZB; j++) {
      av[j] = inr[j] ? lerp1(c[j], c[j + 1], al[j]) : 0.f;
      bv[j] = inr[j] ? lerp1(q[j], q[j + 1], al[j]) : 0.f;
    }
  } else {
#pragma unroll
    for (int j = 0; j < ZB; j++) {
      av[j] = 0.f;
      bv[j] = 0.f;
      if (inr[j]) {
        float2 w00, w01, w10, w11;
        fetch.get2(ii[j], w00, w01);
        fetch.get2(ii[j] + 1, w10, w11);
        av[j] = lerp1(lerp1(w00.x, w01.x, v.au), lerp1(w10.x, w11.x, v.au), al[j]);
        bv[j] = lerp1(lerp1(w00.y, w01.y, v.au), lerp1(w10.y, w11.y, v.au), al[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < ZB; j++) {
    float A = av[j], B = bv[j];
    if (B < 0.f || A < 0.f) {  // gaps (GFIRST_GPU_Kernels.cu:157)
      A = 0.f;
      B = 0.f;
    }
    n[j] += (T)A;
    d[j] += (T)B;
  }
}

// {ratio, calib} pairs: one 16-byte buffer load per plane gives both bins
// (32-bit offsets).
struct FetchPairs {
  __amdgpu_buffer_rsrc_t rc;
  unsigned vrow, rowb, oq, rb0 = 0;
  __device__ __forceinline__ void rows(int i0) { rb0 = (vrow + (unsigned)i0) * rowb; }
  __device__ __forceinline__ void pair(int k, float2& a0, float2& a1) const {
    const float4 q = ld_f4(rc, rb0 + oq, (unsigned)k * rowb);
    a0 = make_float2(q.x, q.y);
    a1 = make_float2(q.z, q.w);
  }
  __device__ __forceinline__ void get2(int ii, float2& a0, float2& a1) const {
    const float4 q = ld_f4(rc, (vrow + (unsigned)ii) * rowb + oq, 0);
    a0 = make_float2(q.x, q.y);
    a1 = make_float2(q.z, q.w);
  }
};

template <int ZB>
__global__ __launch_bounds__(256) void k_sensitivity(DevGeom G, const float2* __restrict__ c2,
                                                     unsigned c2_bytes,
                                                     double* __restrict__ sens, int subset,
                                                     int nsub) {
  const int nav = (G.nang - subset + nsub - 1) / nsub;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int bx, by, bz;
  xcd_region(bx, by, bz);
  const int ix = bx * 16 + (wv & 1) * 8 + (lane & 7);
  const int iy = by * 16 + (wv >> 1) * 8 + (lane >> 3);
  const int zb = bz * ZB;
  const bool act = ix < G.res && iy < G.res;
  FetchPairs f;
  f.rc = rsrc(c2, c2_bytes);
  f.rowb = (unsigned)packed_row_len(G.nrad) * 8u;
  const float xv = (float)ix - G.RESM, yv = (float)iy - G.RESM;
  const unsigned nr = (unsigned)(G.nsinogs + 2 * G.nseg);
  const float fz0 = (float)zb, fzl = (float)(zb + ZB - 1);
  double n[ZB], d[ZB];
#pragma unroll
  for (int j = 0; j < ZB; j++) n[j] = d[j] = 0.0;
  for (int si = 0; si < G.nseg; si++) {
    const SegEntry se = G.seg[si];
    const float fzm = (float)se.zmin, fzhi = (float)(G.nzs - se.zmin);
    const unsigned segrow = (unsigned)(se.nza + 2 * si + 1 - se.zmin);
    for (int a = 0; a < nav; a++) {
      const int it = subset + a * nsub;
      const LaneView v = lane_view(G, xv, yv, G.sin_t[it], G.cos_t[it], se.fzb, fz0, fzl, fzm,
                                   fzhi, act);
      if (__builtin_amdgcn_ballot_w64(v.any) == 0) continue;
      f.vrow = (unsigned)a * nr + segrow;
      f.oq = (unsigned)(v.iq + 1) * 8u;
      accumulate_view<ZB>(v, se.fzb, v.yr, zb, G.nzs, fzm, fzhi, f, n, d);
    }
  }
  if (!act) return;
#pragma unroll
  for (int j = 0; j < ZB; j++) {
    const int iz = zb + j;
    if (iz < G.nzs) sens[((size_t)iz * G.res + iy) * G.res + ix] = d[j];
  }
}

inline int nav_of(const DevGeom& G, int subset, int nsub) {
  return (G.nang - subset + nsub - 1) / nsub;
}

}  // namespace

size_t rotate_floats_per_angle(const DevGeom& G) {
  return (size_t)(G.l1 - G.l0 + 1) * G.nzs * G.nrad;
}

namespace {

// z-sum blocks (= log-likelihood partials): along the sinograms, and for na
// angles of a chunk.
__host__ __device__ inline int zsum_ngb(bool wide, int ngroups, int nsinogs) {
  return wide ? (ngroups + 3) / 4 : (nsinogs + 7) / 8;  // 4 waves a block
}
__host__ __device__ inline int zsum_nib(bool wide, int nrad, int na) {
  return (na * (wide ? (nrad + 3) / 4 : nrad) + 63) / 64;
}

// Blocks of a pass over nav angles in chunks.
inline int zsum_blocks(bool wide, int ngb, int nrad, int nav, int chunk) {
  return ngb * (nav / chunk * zsum_nib(wide, nrad, chunk) + zsum_nib(wide, nrad, nav % chunk));
}
// The narrow kernel serves passes up to this many of its blocks (measured,
// narrow / best wide, us of a whole projection: 368 blocks 26 / 60, 750 40 / 79,
// 1472 53 / 66, 2016 89 / 98, 2466 104 / 107, 2745 94 / 85, 4575 141 / 98).
constexpr int kNarrowBlocks = 2400;

}  // namespace

bool zsum_narrow_serves(const ZsumDims& d, int nsub) {
  const int nav = (d.nang + nsub - 1) / nsub;
  return zsum_blocks(false, zsum_ngb(false, 0, d.nsinogs), d.nrad, nav, kRotChunk) <= kNarrowBlocks;
}

// Sinograms per wave for the passes of a subset count. The longest subset
// decides for all of them. Where no measurement says: narrow waves where they
// serve, 4 sinograms where 6 leave too few waves (3.3M LORs a pass 150 us with 4,
// 163 with 6; 4.8M 202 and 170).
static int zsum_kind(const ZsumDims& d, const Tune& tune, int nsub) {
  if (tune.tuned) return tune.zsum_sg;
  if (zsum_narrow_serves(d, nsub)) return kZsumNarrow;
  const int nav = (d.nang + nsub - 1) / nsub;
  return (long long)d.nsinogs * nav * d.nrad < 3800000 ? 4 : 6;
}

ZsumDims zsum_dims(const GeomHost& h) {
  return {h.info.nsinogs, h.g.nrad, h.g.nang,
          {(int)h.zgrp[0].size(), (int)h.zgrp[1].size(), (int)h.zgrp[2].size()},
          (size_t)(h.info.lambda1 - h.info.lambda0 + 1) * h.g.nzs * h.g.nrad};
}

ZsumPlan zsum_plan(const ZsumDims& d, const Tune& tune, int subset, int nsub,
                   size_t r_cap_floats) {
  const int nav = (d.nang - subset + nsub - 1) / nsub;
  ZsumPlan p{};
  p.kind = zsum_kind(d, tune, nsub);
  const bool wide = p.kind != kZsumNarrow;
  size_t chunk = std::min(r_cap_floats / d.per, (size_t)nav);
  if (chunk * d.per * sizeof(float) >= 0xFFFFFFF0u) chunk = 0xFFFFFFF0u / (d.per * sizeof(float));
  p.chunk = (int)chunk;
  p.ngb = zsum_ngb(wide, d.ngroups[zg_index(p.kind)], d.nsinogs);
  if (p.chunk > 0) p.blocks = zsum_blocks(wide, p.ngb, d.nrad, nav, p.chunk);
  return p;
}

namespace {

ZsumDims zsum_dims(const DevGeom& G) {
  return {G.nsinogs, G.nrad, G.nang, {G.zg[0].n, G.zg[1].n, G.zg[2].n}, rotate_floats_per_angle(G)};
}

hipError_t zsum_launch(const DevGeom& G, const ZsumPlan& zp, const float* R, unsigned rbytes,
                       const FwdArgs& o, bool ratio, int storage, int subset, int nsub,
                       const int* dsub, int a0, int na, int nl, unsigned llh_off, hipStream_t st) {
  const unsigned blocks = (unsigned)zp.ngb * (unsigned)zsum_nib(zp.kind != kZsumNarrow, G.nrad, na);
#define GFR_ZK(K)                                                                             \
  hipLaunchKernelGGL(K, dim3(blocks), dim3(256), 0, st, G, R, rbytes, o, subset, nsub, dsub, \
                     a0, na, nl, llh_off)
#define GFR_ZL(S, RT, LL)                                      \
  switch (zp.kind) {                                           \
    case kZsumNarrow: GFR_ZK((k_zsum_narrow<S, RT, LL>)); break; \
    case 4: GFR_ZK((k_zsum_wide<S, RT, LL, 4>)); break;        \
    case 6: GFR_ZK((k_zsum_wide<S, RT, LL, 6>)); break;        \
    default: GFR_ZK((k_zsum_wide<S, RT, LL, 8>)); break;       \
  }
#define GFR_ZS(S)              \
  if (o.llh_part) {            \
    GFR_ZL(S, true, true)      \
  } else {                     \
    GFR_ZL(S, true, false)     \
  }
  if (!ratio) {
    GFR_ZL(GFR_STORE_F32, false, false)
  } else if (storage == GFR_STORE_F16) {
    GFR_ZS(GFR_STORE_F16)
  } else if (storage == GFR_STORE_BF16) {
    GFR_ZS(GFR_STORE_BF16)
  } else {
    GFR_ZS(GFR_STORE_F32)
  }
#undef GFR_ZS
#undef GFR_ZL
#undef GFR_ZK
  return hipGetLastError();
}

// Deterministic sum of the partials of the subset's angles (full chunks of
// `full` partials each, then the last one's); with dsub the count follows the
// device-side subset index.
__global__ void k_llh_sum(const double* __restrict__ part, int wide, int ngb, int nrad, int chunk,
                          int nang, int subset, int nsub, const int* __restrict__ dsub,
                          double* __restrict__ out) {
  if (dsub) subset = *dsub;
  const int nav = (nang - subset + nsub - 1) / nsub;
  const int n = ngb * (nav / chunk * zsum_nib(wide, nrad, chunk) + zsum_nib(wide, nrad, nav % chunk));
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

}  // namespace

// Planes per rotation block: 16, or 4 where that alone makes enough blocks (16
// angles at 64x64x32: the rotation 14 us with 16, 8 with 4; 64 angles: no
// difference)
static int untuned_rot_z(int kind) { return kind == kZsumNarrow ? 4 : 16; }

Tune untuned_tune(const DevGeom& G, int nsub) {
  const BackShape b = back_shape(G, Tune());
  Tune t;
  t.zsum_sg = zsum_kind(zsum_dims(G), t, nsub);
  t.rot_z = untuned_rot_z(t.zsum_sg);
  t.back_zb = b.zb;
  t.back_lds = b.win && b.zb > 1;  // one slice: back_ahead says how it reads
  t.back_ahead = b.split ? 2 : b.nv;
  return t;
}

hipError_t launch_forward(const DevGeom& G, const float* img, float* R, size_t r_cap_floats,
                          const FwdOut& out, int subset, int nsub, const int* dsub,
                          const Tune& tune, hipStream_t st) {
  // with a device-side subset index the launch covers the largest subset
  const int nav = dsub ? nav_of(G, 0, nsub) : nav_of(G, subset, nsub);
  const int nl = G.l1 - G.l0 + 1;
  const size_t per = rotate_floats_per_angle(G);
  const ZsumPlan zp = zsum_plan(zsum_dims(G), tune, dsub ? 0 : subset, nsub, r_cap_floats);
  const int chunk = zp.chunk;
  if (chunk < 1 || (out.llh_part && zp.blocks > out.llh_cap)) return hipErrorInvalidValue;
  const unsigned llh_per_chunk =
      (unsigned)zp.ngb * (unsigned)zsum_nib(zp.kind != kZsumNarrow, G.nrad, chunk);
  FwdArgs o{out.proj, out.corr,  out.rows,   out.mask,
            out.y,    out.bg,    out.yscale, out.llh_part};
  const bool ratio = out.corr || out.rows.v;
  for (int a0 = 0; a0 < nav; a0 += chunk) {
    const int na = min(chunk, nav - a0);
    const unsigned rbytes = (unsigned)((size_t)na * per * sizeof(float));
    const int tl = rot_tile_samples(nl);
    const unsigned gxy = ((G.nrad + 31) / 32) * ((nl + tl - 1) / tl) * na;
    // plane chunks outermost when an angle pair's rotation exceeds an XCD's
    // 4 MiB L2 (the z-sum cannot find it there anyway)
    const int zouter = 2 * per * sizeof(float) > ((size_t)4 << 20);
    // texels a tile can touch: its diagonal's span, the interpolation partner and rounding
    const float diag = sqrtf(31.f * G.fxf * 31.f * G.fxf + (float)((tl - 1) * (tl - 1)));
    const int side = min(kRotTile, min((int)diag + 4, G.res));
    const unsigned lds = (unsigned)(side * (side | 1) * sizeof(float2));
    const int rz = tune.tuned ? tune.rot_z : untuned_rot_z(zp.kind);
#define GFR_RT(ZC)                                                                                \
  hipLaunchKernelGGL(k_rotate_tile<ZC>, dim3(gxy * ((G.nzs + ZC - 1) / ZC)), dim3(256), lds, st, G, \
                     img, R, subset, nsub, dsub, a0, nl, zouter, side)
    if (rz == 4) GFR_RT(4);
    else if (rz == 32) GFR_RT(32);
    else GFR_RT(16);
#undef GFR_RT
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = zsum_launch(G, zp, R, rbytes, o, ratio, out.storage, subset, nsub, dsub, a0, na, nl,
                    llh_per_chunk * (unsigned)(a0 / chunk), st);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_llh_sum(const DevGeom& G, const double* part, int subset, int nsub,
                          const int* dsub, size_t r_cap_floats, const Tune& tune, double* out,
                          hipStream_t st) {
  const ZsumPlan zp = zsum_plan(zsum_dims(G), tune, dsub ? 0 : subset, nsub, r_cap_floats);
  if (zp.chunk < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_llh_sum, dim3(1), dim3(256), 0, st, part, zp.kind != kZsumNarrow, zp.ngb, G.nrad,
                     zp.chunk, G.nang, subset, nsub, dsub, out);
  return hipGetLastError();
}

hipError_t launch_zsum_tables(const DevGeom& G, float* za, int2* const s[3],
                              uint32_t* const row[3], hipStream_t st) {
  const int n = std::max({G.nsinogs, G.zg[0].n, G.zg[1].n, G.zg[2].n, kZPad});
  hipLaunchKernelGGL(k_zsum_tables, dim3((n + 255) / 256, G.l1 - G.l0 + 1), dim3(256), 0, st, G, za,
                     GroupTables{{s[0], s[1], s[2]}, {row[0], row[1], row[2]}});
  return hipGetLastError();
}

size_t packed_bytes(const DevGeom& G, int subset, int nsub) {
  return sizeof(float2) * (size_t)nav_of(G, subset, nsub) * (G.nsinogs + 2 * (size_t)G.nseg) *
         packed_row_len(G.nrad);
}

PackedRows packed_rows(const DevGeom& G, void* buf, int subset, int nsub, unsigned* bad,
                       unsigned epoch) {
  const size_t entries = packed_bytes(G, subset, nsub) / 8;
  return PackedRows{(float*)buf, (float*)buf + entries, (unsigned)(entries * 4), epoch, bad};
}

hipError_t launch_pack(const DevGeom& G, const float* corr, const uint8_t* mask,
                       const PackedRows& P, int subset, int nsub, hipStream_t st) {
  dim3 grid((G.nrad + kWave - 1) / kWave, (G.nsinogs + 3) / 4, nav_of(G, subset, nsub));
  hipLaunchKernelGGL(k_pack, grid, dim3(kWave, 4), 0, st, G, corr, mask, P, subset, nsub);
  return hipGetLastError();
}

hipError_t launch_sensitivity(const DevGeom& G, const uint8_t* mask, float2* c2, double* sens,
                              int subset, int nsub, hipStream_t st) {
  const size_t bytes = packed_bytes(G, subset, nsub);
  dim3 grid((G.nrad + kWave - 1) / kWave, (G.nsinogs + 3) / 4, nav_of(G, subset, nsub));
  hipLaunchKernelGGL(k_pack_calib, grid, dim3(kWave, 4), 0, st, G, mask, c2, subset, nsub);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (bytes >= 0xFFFFFFF0u) return hipErrorInvalidValue;
  const unsigned nbx = (G.res + 15) / 16;
  hipLaunchKernelGGL(k_sensitivity<4>, dim3(nbx, nbx, (G.nzs + 3) / 4), dim3(256), 0, st, G, c2,
                     (unsigned)bytes, sens, subset, nsub);
  return hipGetLastError();
}

int llh_capacity(const GeomHost& h, int nsub) {
  const ZsumDims d = zsum_dims(h);
  const size_t r_cap = d.per * std::min((d.nang + nsub - 1) / nsub, kRotChunk);
  int most = 0, last = 0;
  for (int n = nsub; n <= d.nang; n++) {
    const int nav = (d.nang + n - 1) / n;
    if (nav == last) continue;  // the same passes
    last = nav;
    for (int sg : {kZsumNarrow, 4, 6, 8}) {
      if (sg == kZsumNarrow && !zsum_narrow_serves(d, n)) continue;
      Tune t;
      t.tuned = true;
      t.zsum_sg = sg;
      most = std::max(most, zsum_plan(d, t, 0, n, r_cap).blocks);
    }
  }
  return most;
}

hipError_t tune_shapes(const DevGeom& G, int nsub, const FwdOut& fo, const float* img, float* R,
                       size_t r_floats, float* num, hipStream_t st, Tune* out) {
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return hipErrorUnknown;
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return hipErrorUnknown;
  }
  hipError_t e = hipSuccess;
  // best of two timed runs after one warm-up; short passes four times in a run,
  // so that the gaps of the host's launches do not hide the kernels
  auto time_it = [&](auto&& launch) -> float {
    float best = 1e30f;
    int n = 1;
    for (int rep = 0; rep < 3 && e == hipSuccess; rep++) {
      e = hipEventRecord(e0, st);
      for (int i = 0; i < n && e == hipSuccess; i++) e = launch();
      if (e == hipSuccess) e = hipEventRecord(e1, st);
      if (e == hipSuccess) e = hipEventSynchronize(e1);
      float ms = 0.f;
      if (e == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess && rep > 0)
        best = ms < best ? ms : best;
      if (rep == 0 && ms < 0.2f) n = 4;
    }
    return best / (float)n;
  };
  Tune t;
  t.tuned = true;
  const int cand[4] = {4, 6, 8, kZsumNarrow};
  float bz = 1e30f, bb = 1e30f;
  for (int c : cand) {
    if (c == kZsumNarrow && !zsum_narrow_serves(zsum_dims(G), nsub)) continue;
    Tune tt = t;
    tt.zsum_sg = c;
    const float ms = time_it([&] {
      return launch_forward(G, img, R, r_floats, fo, 0, nsub, nullptr, tt, st);
    });
    if (ms < bz) {
      bz = ms;
      t.zsum_sg = tt.zsum_sg;
    }
  }
  const int rcand[3] = {4, 16, 32};  // planes per rotation block
  for (int c : rcand) {
    Tune tt = t;
    tt.rot_z = c;
    const float ms = time_it([&] {
      return launch_forward(G, img, R, r_floats, fo, 0, nsub, nullptr, tt, st);
    });
    if (ms < bz) {
      bz = ms;
      t.rot_z = c;
    }
  }
  // backprojector: (LDS window, slices, views loaded ahead). One slice and
  // several views ahead: small images, where each wave's walk over the views,
  // not the device's throughput, sets the time.
  const int bcand[10][3] = {{1, 8, 1}, {1, 4, 1}, {1, 5, 1}, {1, 6, 1}, {1, 16, 1},
                            {0, 1, 4}, {0, 1, 2}, {0, 2, 1}, {0, 4, 1}, {0, 6, 1}};
  const int w8 = ((G.res + 7) / 8) * ((G.res + 7) / 8) * ((G.nzs + 7) / 8);
  for (const auto& c : bcand) {
    Tune tt = t;
    // one slice only where it can win (3072 waves of 8 slices: 388 us against 139)
    if (c[2] > 1 && w8 > 2000) continue;
    // the gathering shapes serve what the windows cannot hold
    if (c[2] == 1 && c[0] != (int)back_window_fits(G, c[1])) continue;
    tt.back_lds = c[0];
    tt.back_zb = c[1];
    tt.back_ahead = c[2];
    tt.tuned = true;
    const float ms = time_it([&] {
      return launch_back_packed(G, {{fo.rows}, {num}}, 1, 0, nsub, nullptr, tt, st);
    });
    if (ms < bb) {
      bb = ms;
      t.back_lds = tt.back_lds;
      t.back_zb = tt.back_zb;
      t.back_ahead = tt.back_ahead;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (e != hipSuccess) return e;
  t.tuned = true;
  t.ms_zsum = bz;
  t.ms_back = bb;
  *out = t;
  return hipSuccess;
}

}  // namespace gfr
