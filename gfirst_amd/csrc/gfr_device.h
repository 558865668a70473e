// gfr_device.h — device helpers shared by the gfx950 kernels.
//
// Rounding model (shared with the CPU oracle so results compare bit for bit):
// every kernel file is compiled with -ffp-contract=off; the only fused
// multiply-adds are explicit fmaf() calls. Interpolation weights are exact
// FP32: lerp(a,b,t) = fma(t, b-a, a), x first, then y, then z.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gfr_internal.h"

namespace gfr {

constexpr int kWave = 64;

__device__ __forceinline__ float lerp1(float a, float b, float t) { return fmaf(t, b - a, a); }

// Raw buffer resource over [p, p + bytes): 32-bit offsets, loads past the end
// return 0 without touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes,
                                           0x00020000);
}
__device__ __forceinline__ float ld_f1(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ float2 ld_f2(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ float4 ld_f4(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// Unnormalized coordinate -> (i0, i1, alpha) with clamp-to-edge addressing:
// texel i covers [i, i+1), so the filter blends floor(c-0.5) and the next one
// (the reference's textures use linear filtering + clamp,
// GFIRST_GPU_Kernels.cu:260-263, 270-279).
__device__ __forceinline__ void axis(float c, int n, int& i0, int& i1, float& a) {
  const float t = c - 0.5f;
  const float f = floorf(t);
  const int i = (int)f;
  a = t - f;
  i0 = min(max(i, 0), n - 1);
  i1 = min(max(i + 1, 0), n - 1);
}

template <int S>
__device__ __forceinline__ float load_store(const void* p, size_t i) {
  if constexpr (S == GFR_STORE_F32) {
    return ((const float*)p)[i];
  } else if constexpr (S == GFR_STORE_F16) {
    return (float)((const _Float16*)p)[i];
  } else {
    const uint32_t b = (uint32_t)((const uint16_t*)p)[i] << 16;
    return __uint_as_float(b);
  }
}

// Work-groups of a 1-D grid are dispatched round-robin over the 8 XCDs (each
// with its own L2). This maps the hardware block id to a logical id so that
// every XCD walks one contiguous range of logical blocks (bijective for any
// grid size).
__device__ __forceinline__ unsigned xcd_remap(unsigned b, unsigned n) {
  const unsigned nx = n >> 3, rem = n & 7u, x = b & 7u, k = b >> 3;
  return x < rem ? x * (nx + 1) + k : rem * (nx + 1) + (x - rem) * nx + k;
}

// The same round-robin for a 3-D grid of (x tile, y tile, z slab) blocks,
// linearised x fastest. With an even x count and a y count divisible by 4,
// XCD k takes every z slab of the tiles of one (nx/2) x (ny/4) region
// (x half k & 1, y quarter k >> 1), so its L2 holds only the rows that
// region projects to; other grids keep the hardware order. Bijective.
__device__ __forceinline__ void xcd_region(int& bx, int& by, int& bz) {
  bx = blockIdx.x;
  by = blockIdx.y;
  bz = blockIdx.z;
  if ((gridDim.x & 1u) == 0 && (gridDim.y & 3u) == 0) {
    const unsigned b = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const unsigned k = b & 7u, j = b >> 3;
    const unsigned hx = gridDim.x >> 1, hy = gridDim.y >> 2, t = j % (hx * hy);
    bz = (int)(j / (hx * hy));
    bx = (int)((k & 1u) * hx + t % hx);
    by = (int)((k >> 1) * hy + t / hx);
  }
}

// divVxVGPU (GFIRST_GPU_Kernels.cu:173-182)
__device__ __forceinline__ float update_ratio(float num, float den) {
  return (den < 0.001f) ? 1.0f : num / den;
}

// Lanes of one wave exchange values through LDS: orders what the wave wrote
// before what it reads, without a barrier (DS operations of a wave are in
// order).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Packed rows of a subset for the backprojector (PackedRows): one ratio per
// bin. Per angle of the subset and per segment, the segment's planes
// zmin..NZS-zmin-1 are preceded and followed by one extra row, so that every
// plane a voxel can blend (zmin-1 .. NZS-zmin) is addressable without a test:
//  - segments with zmin > 0: the extra rows hold -1000, the value the
//    reference stores outside the segment's planes (GFIRST.cu:447);
//  - the direct segment (zmin = 0): the extra rows repeat planes 0 and NZS-1,
//    which is what the clamp-to-edge filter reads for planes -1 and NZS.
// Each row holds NRAD + 2 entries: bin r at r + 1, and copies of bins 0 and
// NRAD-1 at both ends, so the pair of bins a radial position blends under
// clamp-to-edge, (clamp(i), clamp(i + 1)), is the two adjacent entries at
// clamp(i, -1, NRAD-1) + 1.
// The calibration (1, or -1000 in gaps and in the extra rows of oblique
// segments) has no storage of its own: a bin with calibration -1000 reads
// kInvalid in `v` and its ratio is in `side`, which holds nothing else. A
// ratio whose bits are kInvalid's (far below zero: it drops every sample that
// weighs it) is in `side` as well.
// *bad == epoch says that some ratio of the pass lies outside the range for
// which the fast summation is exact (regular_ratio).
constexpr float kInvalid = -0x1.5a5a5ap126f;
__host__ __device__ __forceinline__ size_t packed_row_len(int nrad) { return (size_t)nrad + 2; }
__device__ __forceinline__ size_t packed_rows_per_angle(const DevGeom& G) {
  return (size_t)G.nsinogs + 2 * (size_t)G.nseg;
}
// 0 <= c <= 2^60 or -2^60 <= c <= -2^-32 (gaps are -1000): interpolated
// values stay below 2^61 in magnitude, and negative ones above 2^-127 (every
// weight is a multiple of 2^-24).
__device__ __forceinline__ bool regular_ratio(float c) {
  return (c >= 0.f && c <= 0x1p60f) || (c <= -0x1p-32f && c >= -0x1p60f);
}
// Writes the N <= 4 consecutive bins r .. r + N - 1 (N wave-uniform or not) of
// one sinogram and angle.
struct __align__(4) Float4u { float x, y, z, w; };
__device__ __forceinline__ void store_packed(const DevGeom& G, const PackedRows& P, int ag, int s,
                                             int r, int N, const float (&c)[4],
                                             const bool (&valid)[4]) {
  const int2 sp = G.sino[s];
  const SegEntry se = G.seg[sp.x];
  const size_t row0 = (size_t)ag * packed_rows_per_angle(G) + se.nza + 2 * (size_t)sp.x;
  const int k = sp.y - se.zmin;
  const int nz = G.nzs - 2 * se.zmin;
  const size_t L = packed_row_len(G.nrad);
  bool out = false, inv = false;
  float f[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    f[i] = valid[i] ? c[i] : kInvalid;
    if (i < N) {
      out |= !regular_ratio(c[i]);
      inv |= f[i] == kInvalid;
    }
  }
  if (out) *P.bad = P.epoch;
  auto put = [&](size_t row, const float (&val)[4], const float (&sd)[4], bool side) {
    const size_t o = row * L + r + 1;
    if (N == 4) {
      *(Float4u*)(P.v + o) = Float4u{val[0], val[1], val[2], val[3]};
    } else {
#pragma unroll
      for (int i = 0; i < 3; i++)
        if (i < N) P.v[o + i] = val[i];
    }
    if (r == 0) P.v[o - 1] = val[0];
    if (r + N == G.nrad) P.v[o + N] = val[N - 1 > 2 ? 3 : N - 1 > 1 ? 2 : N - 1 > 0 ? 1 : 0];
    if (side) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i < N && val[i] == kInvalid) {
          P.side[o + i] = sd[i];
          if (r + i == 0) P.side[o - 1] = sd[i];
          if (r + i == G.nrad - 1) P.side[o + i + 1] = sd[i];
        }
    }
  };
  put(row0 + 1 + k, f, c, inv);
  if (k == 0 || k == nz - 1) {
    const float gap[4] = {kInvalid, kInvalid, kInvalid, kInvalid};
    const float out4[4] = {-1000.f, -1000.f, -1000.f, -1000.f};
    if (se.zmin == 0) {
      if (k == 0) put(row0, f, c, inv);
      if (k == nz - 1) put(row0 + nz + 1, f, c, inv);
    } else {
      if (k == 0) put(row0, gap, out4, true);
      if (k == nz - 1) put(row0 + nz + 1, gap, out4, true);
    }
  }
}

// The same rows as {ratio 1, calib} pairs, for the FP64 sensitivity.
__device__ __forceinline__ void store_calib(const DevGeom& G, float2* c2, int ag, int s, int r,
                                            float2 v) {
  const int2 sp = G.sino[s];
  const SegEntry se = G.seg[sp.x];
  const size_t row0 = (size_t)ag * packed_rows_per_angle(G) + se.nza + 2 * (size_t)sp.x;
  const int k = sp.y - se.zmin;
  const int nz = G.nzs - 2 * se.zmin;
  const float2 edge = se.zmin == 0 ? v : make_float2(-1000.f, -1000.f);
  const size_t L = packed_row_len(G.nrad);
  auto put = [&](size_t row, float2 val) {
    float2* p = c2 + row * L + r + 1;
    p[0] = val;
    if (r == 0) p[-1] = val;
    if (r == G.nrad - 1) p[1] = val;
  };
  put(row0 + 1 + k, v);
  if (k == 0) put(row0, edge);
  if (k == nz - 1) put(row0 + nz + 1, edge);
}

// Sinogram bin b in angle-major order, and back.
__device__ __forceinline__ unsigned vlor_key(const DevGeom& G, int b) {
  const int row = b / G.nrad, s = row / G.nang;
  return (unsigned)(((row - s * G.nang) * G.nsinogs + s) * G.nrad + b - row * G.nrad);
}
__device__ __forceinline__ int vlor_bin(const DevGeom& G, unsigned key) {
  const int row = (int)key / G.nrad, it = row / G.nsinogs;
  return ((row - it * G.nsinogs) * G.nang + it) * G.nrad + (int)key - row * G.nrad;
}

}  // namespace gfr
