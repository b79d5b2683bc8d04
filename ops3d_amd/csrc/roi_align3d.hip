// 3-D RoI Align on gfx950 (replaces the reference's roi_align_3d_{forward,backward}_cuda_kernel,
// csrc/cuda/roi_align_3d_cuda_kernel.cuh:27-220, with the interpolation helpers of
// csrc/cuda/interpolation_helpers_3d.h:25-260; bound as _C.roi_align_3d_forward/backward by
// csrc/roi_align_3d.h:97-136).
//
// features [N, C, D, H, W]; rois [R, 7] (batch index, x1, y1, z1, x2, y2, z2) in the features'
// dtype; output [R, C, PD, PH, PW].  Per output bin: the roi scaled by spatial_scale (no
// rounding), extents clamped to >= 1, the bin cut into a grid of samples (sampling_ratio per
// axis, or ceil(extent / pooled) when it is <= 0), each sample interpolated (order 1: trilinear
// with the reference's edge handling -- a sample beyond [-1, size] reads 0, coordinates below 0
// clamp to 0, a base corner at size-1 collapses both corners onto it; order 0: the nearest
// corner), and the samples averaged.  All arithmetic is fp32 (16-bit types are widened on load;
// the reference computes in the element type), rounded step by step (no contraction).
//
// Forward: a gather, one thread per (roi, CPT = 4 channels, bin), or on channels-last features
// one lane per (bin, 8 channels) (the same bits).  It is separable: the bin's average is the sum
// over its distinct z, y and x taps of the per-axis weight sums times the value, taken along x, then
// y, then z in fused multiply-adds, fewer loads than 8 corners per sample; bins of more than 8 taps
// on an axis take the reference's per-sample loop.  Backward: the adjoint, as a gather when the
// output has at most 64 bins per axis and 384 in all (each voxel sums, in registers, the rois
// that reach it, in an order that they alone decide: no atomics, the same bits on every run; the
// workspace holds the rois' axis weight tables and a channels-last copy of grad_output), otherwise
// (or with more than 2^20 channels) by fp32 atomics into a channels-last workspace (64 lanes = 64
// contiguous channels per atomic instruction) transposed into grad_input afterwards.  A roi whose batch index is
// outside [0, N) reads and writes nothing (its output is 0; the reference indexes out of
// bounds).
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/ops3d_roi_align3d.h"

namespace ops3d_roi {

template <typename T> __device__ __forceinline__ float to_f(T v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f(float v) { return (T)v; }

struct Roi {
  int b;
  float sw, sh, sd;      // roi start (x, y, z) in feature voxels
  float bw, bh, bd;      // bin sizes
  int gw, gh, gd;        // samples per bin and axis
  float count;
};

template <typename T>
__device__ __forceinline__ Roi roi_setup(const T *rois, int r, float scale, int sr, int PD, int PH, int PW) {
#pragma clang fp contract(off)
  const T *p = rois + (int64_t)r * 7;
  Roi o;
  o.b = (int)to_f(p[0]);
  o.sw = to_f(p[1]) * scale;
  o.sh = to_f(p[2]) * scale;
  o.sd = to_f(p[3]) * scale;
  const float ew = to_f(p[4]) * scale, eh = to_f(p[5]) * scale, ed = to_f(p[6]) * scale;
  const float rw = fmaxf(ew - o.sw, 1.f), rh = fmaxf(eh - o.sh, 1.f), rd = fmaxf(ed - o.sd, 1.f);
  o.bd = rd / (float)PD;
  o.bh = rh / (float)PH;
  o.bw = rw / (float)PW;
  o.gd = sr > 0 ? sr : (int)ceilf(rd / (float)PD);
  o.gh = sr > 0 ? sr : (int)ceilf(rh / (float)PH);
  o.gw = sr > 0 ? sr : (int)ceilf(rw / (float)PW);
  o.count = (float)max(o.gd * o.gh * o.gw, 1);
  return o;
}

// Sample coordinate along one axis: start + p * bin + (i + 0.5) * bin / grid.
__device__ __forceinline__ float sample_coord(float start, int p, float bin, int i, int grid) {
#pragma clang fp contract(off)
  return start + (float)p * bin + ((float)i + 0.5f) * bin / (float)grid;
}

// The 8 corner offsets (voxel index inside one (batch, channel) volume) and weights of a
// sample; false when the sample lies beyond [-1, size] on some axis (it contributes nothing).
// Corner order: (z0|z1) x (y0|y1) x (x0|x1), x fastest.
__device__ __forceinline__ bool corners(float z, float y, float x, int D, int H, int W, int order, int64_t off[8],
                                        float w[8]) {
#pragma clang fp contract(off)
  if (y < -1.f || y > (float)H || x < -1.f || x > (float)W || z < -1.f || z > (float)D) return false;
  if (z <= 0.f) z = 0.f;
  if (y <= 0.f) y = 0.f;
  if (x <= 0.f) x = 0.f;
  int z0 = (int)z, y0 = (int)y, x0 = (int)x, z1, y1, x1;
  if (z0 >= D - 1) { z1 = z0 = D - 1; z = (float)z0; } else { z1 = z0 + 1; }
  if (y0 >= H - 1) { y1 = y0 = H - 1; y = (float)y0; } else { y1 = y0 + 1; }
  if (x0 >= W - 1) { x1 = x0 = W - 1; x = (float)x0; } else { x1 = x0 + 1; }
  const float lz = z - (float)z0, ly = y - (float)y0, lx = x - (float)x0;
  const float hz = 1.f - lz, hy = 1.f - ly, hx = 1.f - lx;
  const int64_t zz[2] = {(int64_t)z0 * H * W, (int64_t)z1 * H * W}, yy[2] = {(int64_t)y0 * W, (int64_t)y1 * W};
  const int xx[2] = {x0, x1};
#pragma unroll
  for (int c = 0; c < 8; ++c) off[c] = zz[c >> 2] + yy[(c >> 1) & 1] + xx[c & 1];
  if (order == 0) {   // the first corner (in this order) whose three weights are all >= 0.5
    const bool zl = hz >= 0.5f, zh = lz >= 0.5f, yl = hy >= 0.5f, yh = ly >= 0.5f, xl = hx >= 0.5f, xh = lx >= 0.5f;
    const bool hit[8] = {zl && yl && xl, zl && yl && xh, zl && yh && xl, zl && yh && xh,
                         zh && yl && xl, zh && yl && xh, zh && yh && xl, zh && yh && xh};
    bool done = false;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      w[c] = (!done && hit[c]) ? 1.f : 0.f;
      done = done || hit[c];
    }
  } else {
    const float wz[2] = {hz, lz}, wy[2] = {hy, ly}, wx[2] = {hx, lx};
#pragma unroll
    for (int c = 0; c < 8; ++c) w[c] = wz[c >> 2] * wy[(c >> 1) & 1] * wx[c & 1];
  }
  return true;
}

// The taps of one axis of a bin: up to NT distinct positions with their summed weights, in the
// order the samples first reach them (increasing position; weights of invalid samples and
// collapsed taps are left out); `over` when the samples reach more than NT positions.  Static
// register indices only (predicated), so nothing spills to scratch.
template <int NT>
struct AxisTaps {
  int n;
  bool over;
  int pos[NT];
  float w[NT];
  __device__ __forceinline__ void add(int p, float wt) {
    if (wt == 0.f) return;
    bool done = false;
#pragma unroll
    for (int k = 0; k < NT; ++k)
      if (!done && k < n && pos[k] == p) {
        w[k] += wt;
        done = true;
      }
    if (!done) {
      if (n == NT) {
        over = true;
        return;
      }
#pragma unroll
      for (int k = 0; k < NT; ++k)
        if (k == n) {
          pos[k] = p;
          w[k] = wt;
        }
      ++n;
    }
  }
  // drop the first tap (register moves, so a loop over the taps needs no dynamic index)
  __device__ __forceinline__ void shift() {
#pragma unroll
    for (int k = 0; k + 1 < NT; ++k) {
      pos[k] = pos[k + 1];
      w[k] = w[k + 1];
    }
    --n;
  }
};
using AxisTaps4 = AxisTaps<4>;
using AxisTaps8 = AxisTaps<8>;
// Grids of more than 2 samples per axis take the separable sum when every axis of the bin has
// at most kSepTaps distinct taps, the per-sample loop otherwise.
constexpr int kSepTaps = 8;

__device__ __forceinline__ AxisTaps4 bin_taps(float start, int p, float bin, int grid, int size, int order);
template <int NT>
__device__ __forceinline__ AxisTaps<NT> bin_taps_n(float start, int p, float bin, int grid, int size, int order);

// One step of a sum over taps: the first product, then fused multiply-adds.
__device__ __forceinline__ float tap_add(int k, float w, float v, float sum) {
#pragma clang fp contract(off)
  return k == 0 ? w * v : fmaf(w, v, sum);
}

template <typename T, int CPT>
__global__ __launch_bounds__(256) void roi_align3d_forward_kernel(const T *feat, const T *rois, T *out, int N, int C, int D,
                                                                  int H, int W, int R, int PD, int PH, int PW,
                                                                  float scale, int sr, int order) {
#pragma clang fp contract(off)
  const int CG = C / CPT;
  const int64_t total = (int64_t)R * CG * PD * PH * PW;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int pw = (int)(idx % PW), ph = (int)((idx / PW) % PH), pd = (int)((idx / ((int64_t)PW * PH)) % PD);
  const int cg = (int)((idx / ((int64_t)PW * PH * PD)) % CG);
  const int r = (int)(idx / ((int64_t)PW * PH * PD * CG));
  const Roi q = roi_setup(rois, r, scale, sr, PD, PH, PW);
  const int64_t vol = (int64_t)D * H * W;
  const bool inb = q.b >= 0 && q.b < N;   // a roi of a batch item that does not exist reads nothing
  const T *base = feat + ((int64_t)(inb ? q.b : 0) * C + (int64_t)cg * CPT) * vol;
  float acc[CPT];
#pragma unroll
  for (int c = 0; c < CPT; ++c) acc[c] = 0.f;
  if (inb && q.gd <= 2 && q.gh <= 2 && q.gw <= 2) {
    // separable: the bin's average is sum over its distinct z, y, x taps of WZ * WY * WX * value
    // (the samples form a full grid and the corner weights are products, so the per-axis weight
    // sums factor), at most 4 taps per axis instead of 8 corners per sample; summed along x, then
    // y, then z (tap_add), as in the channels-last kernel
    const AxisTaps4 tz = bin_taps(q.sd, pd, q.bd, q.gd, D, order);
    const AxisTaps4 ty = bin_taps(q.sh, ph, q.bh, q.gh, H, order);
    const AxisTaps4 tx = bin_taps(q.sw, pw, q.bw, q.gw, W, order);
    if (tx.n > 0 && ty.n > 0) {
#pragma unroll
      for (int kz = 0; kz < 4; ++kz) {
        if (kz >= tz.n) break;
        float u[CPT];
#pragma unroll
        for (int ky = 0; ky < 4; ++ky) {
          if (ky >= ty.n) break;
          const int64_t rowo = ((int64_t)tz.pos[kz] * H + ty.pos[ky]) * W;
          float t[CPT];
#pragma unroll
          for (int kx = 0; kx < 4; ++kx) {
            if (kx >= tx.n) break;
#pragma unroll
            for (int c = 0; c < CPT; ++c) t[c] = tap_add(kx, tx.w[kx], to_f(base[(int64_t)c * vol + rowo + tx.pos[kx]]), t[c]);
          }
#pragma unroll
          for (int c = 0; c < CPT; ++c) u[c] = tap_add(ky, ty.w[ky], t[c], u[c]);
        }
#pragma unroll
        for (int c = 0; c < CPT; ++c) acc[c] = tap_add(kz, tz.w[kz], u[c], acc[c]);
      }
    }
  }
  bool wide = inb && (q.gd > 2 || q.gh > 2 || q.gw > 2);
  if (wide) {
    // larger grids: separable too when every axis has at most kSepTaps distinct taps (the same
    // loop over taps, z and y taps consumed by shifting the lists)
    AxisTaps8 tz = bin_taps_n<kSepTaps>(q.sd, pd, q.bd, q.gd, D, order);
    AxisTaps8 ty = bin_taps_n<kSepTaps>(q.sh, ph, q.bh, q.gh, H, order);
    const AxisTaps8 tx = bin_taps_n<kSepTaps>(q.sw, pw, q.bw, q.gw, W, order);
    if (!tz.over && !ty.over && !tx.over) {
      wide = false;
      if (tx.n > 0 && ty.n > 0)
        for (int kz = 0; tz.n > 0; tz.shift(), ++kz) {
          AxisTaps8 tyc = ty;
          float u[CPT];
#pragma unroll
          for (int c = 0; c < CPT; ++c) u[c] = 0.f;
          for (int ky = 0; tyc.n > 0; tyc.shift(), ++ky) {
            const int64_t rowo = ((int64_t)tz.pos[0] * H + tyc.pos[0]) * W;
            float t[CPT];
#pragma unroll
            for (int kx = 0; kx < kSepTaps; ++kx) {
              if (kx >= tx.n) break;
#pragma unroll
              for (int c = 0; c < CPT; ++c)
                t[c] = tap_add(kx, tx.w[kx], to_f(base[(int64_t)c * vol + rowo + tx.pos[kx]]), t[c]);
            }
#pragma unroll
            for (int c = 0; c < CPT; ++c) u[c] = tap_add(ky, tyc.w[0], t[c], u[c]);
          }
#pragma unroll
          for (int c = 0; c < CPT; ++c) acc[c] = tap_add(kz, tz.w[0], u[c], acc[c]);
        }
    }
  }
  for (int iz = 0; wide && iz < q.gd; ++iz) {
    const float z = sample_coord(q.sd, pd, q.bd, iz, q.gd);
    for (int iy = 0; iy < q.gh; ++iy) {
      const float y = sample_coord(q.sh, ph, q.bh, iy, q.gh);
      for (int ix = 0; ix < q.gw; ++ix) {
        const float x = sample_coord(q.sw, pw, q.bw, ix, q.gw);
        int64_t off[8];
        float w[8];
        if (!corners(z, y, x, D, H, W, order, off, w)) continue;
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
          const T *v = base + (int64_t)c * vol;
          float s = w[0] * to_f(v[off[0]]);   // w1 v1 + w2 v2 + ... in order (the reference's sum)
#pragma unroll
          for (int k = 1; k < 8; ++k) s = s + w[k] * to_f(v[off[k]]);
          acc[c] = acc[c] + s;
        }
      }
    }
  }
  const int64_t o = ((((int64_t)r * C + (int64_t)cg * CPT) * PD + pd) * PH + ph) * PW + pw;
  const int64_t cs = (int64_t)PD * PH * PW;
#pragma unroll
  for (int c = 0; c < CPT; ++c) out[o + c * cs] = from_f<T>(acc[c] / q.count);
}

__global__ __launch_bounds__(256) void fill_zero_kernel(float *p, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = 0.f;
}

// Channels-last fp32 [N, V, C] -> [N, C, V] in T, through a 64 x 64 LDS tile (padded rows: the
// column reads are conflict-free).  grid (ceil(V/64), ceil(C/64), N), 256 threads.
template <typename T>
__global__ __launch_bounds__(256) void channels_last_to_ncdhw_kernel(const float *src, T *dst, int C, int64_t V) {
  __shared__ float t[64][65];
  const int tid = threadIdx.x, lane = tid & 63, row = tid >> 6;
  const int64_t v0 = (int64_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  const int64_t n = blockIdx.z;
  const float *s = src + n * V * C;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int vv = i * 4 + row;
    if (v0 + vv < V && c0 + lane < C) t[vv][lane] = s[(v0 + vv) * C + c0 + lane];
  }
  __syncthreads();
  T *d = dst + n * C * V;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int cc = i * 4 + row;
    if (c0 + cc < C && v0 + lane < V) d[(int64_t)(c0 + cc) * V + v0 + lane] = from_f<T>(t[lane][cc]);
  }
}

// One axis of a sample's interpolation, with the edge rules of corners(): valid unless beyond
// [-1, size]; below 0 clamps to 0; a base at size - 1 collapses both taps onto it (weights 1, 0).
// Order 0 keeps the nearest tap (the low one when its weight is >= 0.5), weight 1.  corners()'s
// eight weights are the products of the three axes' (its nearest-corner rule picks, axis by
// axis, the low tap whenever allowed, so it is this per-axis choice too).
struct AxisTap {
  bool ok;
  int i0, i1;
  float w0, w1;
};
__device__ __forceinline__ AxisTap axis_tap(float c, int size, int order) {
#pragma clang fp contract(off)
  AxisTap t;
  t.ok = !(c < -1.f || c > (float)size);
  if (c <= 0.f) c = 0.f;
  t.i0 = (int)c;
  if (t.i0 >= size - 1) {
    t.i1 = t.i0 = size - 1;
    c = (float)t.i0;
  } else {
    t.i1 = t.i0 + 1;
  }
  const float l = c - (float)t.i0, h = 1.f - l;
  if (order == 0) {
    t.w0 = h >= 0.5f ? 1.f : 0.f;
    t.w1 = h >= 0.5f ? 0.f : 1.f;
  } else {
    t.w0 = h;
    t.w1 = l;
  }
  return t;
}

// The taps of bin p on one axis (grid <= 2 samples), merged by position.
__device__ __forceinline__ AxisTaps4 bin_taps(float start, int p, float bin, int grid, int size, int order) {
  AxisTaps4 t;
  t.n = 0;
  t.over = false;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    t.pos[k] = 0;
    t.w[k] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (i >= grid) break;
    const AxisTap a = axis_tap(sample_coord(start, p, bin, i, grid), size, order);
    if (!a.ok) continue;
    t.add(a.i0, a.w0);
    if (a.i1 != a.i0) t.add(a.i1, a.w1);
  }
  return t;
}

// The taps of bin p on one axis for any grid, up to NT of them (t.over beyond that).
template <int NT>
__device__ __forceinline__ AxisTaps<NT> bin_taps_n(float start, int p, float bin, int grid, int size, int order) {
  AxisTaps<NT> t;
  t.n = 0;
  t.over = false;
#pragma unroll
  for (int k = 0; k < NT; ++k) {
    t.pos[k] = 0;
    t.w[k] = 0.f;
  }
  for (int i = 0; i < grid && !t.over; ++i) {
    const AxisTap a = axis_tap(sample_coord(start, p, bin, i, grid), size, order);
    if (!a.ok) continue;
    t.add(a.i0, a.w0);
    if (a.i1 != a.i0) t.add(a.i1, a.w1);
  }
  return t;
}

// Sum of the valid samples' weights on tap position `pos` of one axis (sample i at
// sample_coord(start, p, bin, i, grid)).
__device__ __forceinline__ float axis_weight_at(int pos, float start, int p, float bin, int grid, int size, int order) {
  float s = 0.f;
  for (int i = 0; i < grid; ++i) {
    const AxisTap t = axis_tap(sample_coord(start, p, bin, i, grid), size, order);
    if (!t.ok) continue;
    if (t.i0 == pos) s += t.w0;
    if (t.i1 == pos && t.i1 != t.i0) s += t.w1;
  }
  return s;
}

// Backward: one wave per (roi, 64 channels, output row (pd, ph)); lane = channel.  The weights
// are separable, so the row's contribution to voxel (z, y, x) is WZ[z] * WY[y] * X[x], with WZ
// and WY the row's summed z and y tap weights and X[x] = sum over the row's x samples of
// top[bin] * wx / count.  The wave walks the x samples in increasing x (they are sorted), keeps
// the running X of the two newest tap positions per lane and, once the walk has passed a
// position, adds WZ * WY * X to every (z, y) tap of it with one atomic instruction each: 64
// contiguous channels of the channels-last workspace.  Every voxel a row touches thus gets one
// atomic per (row, 64 channels) instead of one per sample corner.  WZ / WY sit in lanes
// (lane t: tap position min + t); rows with more than 64 tap positions on an axis (adaptive
// grids of huge bins) take the per-sample path.
constexpr int kBwdWaves = 4;
template <typename T>
__global__ __launch_bounds__(64 * kBwdWaves) void roi_align3d_backward_kernel(const T *top, const T *rois, float *acc,
                                                                            int N, int C, int D, int H, int W, int R,
                                                                            int PD, int PH, int PW, float scale, int sr,
                                                                            int order) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int CG = (C + 63) / 64;
  const int64_t wid = (int64_t)blockIdx.x * kBwdWaves + (threadIdx.x >> 6);
  if (wid >= (int64_t)R * CG * PD * PH) return;   // whole waves
  const int ph = (int)(wid % PH), pd = (int)((wid / PH) % PD);
  const int cg = (int)((wid / ((int64_t)PH * PD)) % CG);
  const int r = (int)(wid / ((int64_t)PH * PD * CG));
  const int c = cg * 64 + lane;
  const bool active = c < C;
  const Roi q = roi_setup(rois, r, scale, sr, PD, PH, PW);
  if (q.b < 0 || q.b >= N) return;   // a roi of a batch item that does not exist
  const int64_t vol = (int64_t)D * H * W;
  float *base = acc + (int64_t)q.b * vol * C + c;
  const T *tg = top + (((int64_t)r * C + (active ? c : 0)) * PD + pd) * PH * PW + (int64_t)ph * PW;
  // tap ranges of the row's z and y samples (coordinates increase with the sample index)
  int z_lo = 1 << 30, z_hi = -1, y_lo = 1 << 30, y_hi = -1;
  for (int i = 0; i < q.gd; ++i) {
    const AxisTap t = axis_tap(sample_coord(q.sd, pd, q.bd, i, q.gd), D, order);
    if (t.ok) { z_lo = min(z_lo, t.i0); z_hi = max(z_hi, t.i1); }
  }
  for (int i = 0; i < q.gh; ++i) {
    const AxisTap t = axis_tap(sample_coord(q.sh, ph, q.bh, i, q.gh), H, order);
    if (t.ok) { y_lo = min(y_lo, t.i0); y_hi = max(y_hi, t.i1); }
  }
  if (z_hi < 0 || y_hi < 0) return;   // no valid sample in z or y: the row adds nothing
  const int nz = z_hi - z_lo + 1, ny = y_hi - y_lo + 1;
  if (nz <= 64 && ny <= 64) {
    const float wz_l = lane < nz ? axis_weight_at(z_lo + lane, q.sd, pd, q.bd, q.gd, D, order) : 0.f;
    const float wy_l = lane < ny ? axis_weight_at(y_lo + lane, q.sh, ph, q.bh, q.gh, H, order) : 0.f;
    // X of the tap position px (a0) and px + 1 (a1); `open`: px holds a position
    int px = 0;
    bool open = false, used1 = false;
    float a0 = 0.f, a1 = 0.f;
    const auto flush = [&](int x, float v) {
      const float vc = v / q.count;
      for (int tz = 0; tz < nz; ++tz) {
        const float wz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wz_l), tz));
        if (wz == 0.f) continue;
        for (int ty = 0; ty < ny; ++ty) {
          const float wy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wy_l), ty));
          if (wy == 0.f) continue;
          if (active) atomicAdd(base + (((int64_t)(z_lo + tz) * H + (y_lo + ty)) * W + x) * C, (wz * wy) * vc);
        }
      }
    };
    for (int pw = 0; pw < PW; ++pw) {
      const float g = active ? to_f(tg[pw]) : 0.f;
      for (int ix = 0; ix < q.gw; ++ix) {
        const AxisTap t = axis_tap(sample_coord(q.sw, pw, q.bw, ix, q.gw), W, order);
        if (!t.ok) continue;
        if (!open) {
          px = t.i0;
          open = true;
        } else if (t.i0 == px + 1) {
          flush(px, a0);
          px = t.i0;
          a0 = a1;
          a1 = 0.f;
          used1 = false;
        } else if (t.i0 > px + 1) {
          flush(px, a0);
          if (used1) flush(px + 1, a1);
          px = t.i0;
          a0 = a1 = 0.f;
          used1 = false;
        }
        a0 += g * t.w0;
        if (t.i1 != t.i0) {
          a1 += g * t.w1;
          used1 = true;
        }
      }
    }
    if (open) {
      flush(px, a0);
      if (used1) flush(px + 1, a1);
    }
    return;
  }
  // per-sample path: the 8 corners of each sample, top * w / count each
  for (int pw = 0; pw < PW; ++pw) {
    const float g = active ? to_f(tg[pw]) : 0.f;
    for (int iz = 0; iz < q.gd; ++iz) {
      const float z = sample_coord(q.sd, pd, q.bd, iz, q.gd);
      for (int iy = 0; iy < q.gh; ++iy) {
        const float y = sample_coord(q.sh, ph, q.bh, iy, q.gh);
        for (int ix = 0; ix < q.gw; ++ix) {
          const float x = sample_coord(q.sw, pw, q.bw, ix, q.gw);
          int64_t off[8];
          float w[8];
          if (!corners(z, y, x, D, H, W, order, off, w)) continue;
#pragma unroll
          for (int k = 0; k < 8; ++k)
            if (w[k] != 0.f && active) atomicAdd(base + off[k] * C, g * w[k] / q.count);
        }
      }
    }
  }
}

// Backward as a gather (no atomics).  From roi r voxel (z, y, x) gets the sum over bins
// (pd, ph, pw) of WZ[pd][z] * WY[ph][y] * WX[pw][x] * top[r, c, pd, ph, pw] / count, where
// WZ[pd][z] is the sum of bin pd's z-sample tap weights on z (and so on) -- the sum over the bin's
// samples of their corner weights, separable because the samples form a full grid.  A wave owns a
// tile of 4 x 4 x 4 voxels and 64 channels, a lane per channel, its 64 sums in registers, and adds
// up the rois whose footprint reaches the tile in a fixed order (index order, except that of every
// 192 the few with small bins come last), so the result is the same on every run.  With channels
// on the lanes everything but top is uniform over the wave: weights, bin ranges and loop bounds sit
// in scalar registers, no lane diverges, and the sum is taken axis by axis -- over pw into 4 x positions, over ph into 4 x 4, over pd into
// the 64 voxels -- about 5 multiply-adds per voxel and roi instead of one per bin combination.
// A lane's top values of a bin row (one 128-byte line per bin from the channels-last copy) are
// loaded one row ahead.
// Two passes fill the workspace first: roi_axis_table_kernel and grad_channels_last_kernel.  Needs at most 64 bins per axis and 384 in all (else the atomic path).
// What it measured, and what bounds it: at backward().
constexpr int kGT = 4;                           // tile edge
constexpr int kGRun = 128;                       // consecutive tiles of one XCD when not ordered, at most
constexpr int kGMaxAxisBins = 64, kGMaxBins = 384;

constexpr int kGMaxChannels = 1 << 20;           // a roi's bins within 32-bit byte offsets

__host__ __device__ inline bool gather_fits(int C, int PD, int PH, int PW) {
  return C <= kGMaxChannels && PD <= kGMaxAxisBins && PH <= kGMaxAxisBins && PW <= kGMaxAxisBins && PD * PH * PW <= kGMaxBins;
}
__host__ __device__ inline int tiles_of(int n) { return (n + kGT - 1) / kGT; }

// A tile's bins on one axis: first, last (first > last: none); bit 31 of the z words: the roi's top
// holds an infinity or NaN.
constexpr uint32_t kNoBins = 1u;                 // first 1, last 0
constexpr uint32_t kNonFinite = 0x80000000u;
__device__ __forceinline__ int first_bin(uint32_t w) { return (int)(w & 0xffu); }
__device__ __forceinline__ int last_bin(uint32_t w) { return (int)((w >> 8) & 0xffu); }

// Per-roi axis tables, made once per call: for roi r and axis a (size S, P bins) the weights
// wt[r][a][p][x] of every bin at every position (z's divided by the sample count), and for every
// tile of 4 positions the first and last bin with a nonzero weight in it, tr[tile][r] (tiles of z,
// then y, then x: consecutive rois together, as the gather tests them).
template <typename T>
__global__ __launch_bounds__(256) void roi_axis_table_kernel(const T *rois, float *wt, uint32_t *tr, int D, int H,
                                                             int W, int PD, int PH, int PW, int R, float scale,
                                                             int sr, int order) {
  const int r = blockIdx.x, ax = blockIdx.y;
  const Roi q = roi_setup(rois, r, scale, sr, PD, PH, PW);
  const int S = ax == 0 ? D : (ax == 1 ? H : W), P = ax == 0 ? PD : (ax == 1 ? PH : PW);
  const float st = ax == 0 ? q.sd : (ax == 1 ? q.sh : q.sw), bn = ax == 0 ? q.bd : (ax == 1 ? q.bh : q.bw);
  const int gr = ax == 0 ? q.gd : (ax == 1 ? q.gh : q.gw);
  float *w = wt + (size_t)r * ((size_t)D * PD + (size_t)H * PH + (size_t)W * PW) +
             (ax == 0 ? 0 : (ax == 1 ? (size_t)D * PD : (size_t)D * PD + (size_t)H * PH));
  uint32_t *t = tr + (size_t)(ax == 0 ? 0 : (ax == 1 ? tiles_of(D) : tiles_of(D) + tiles_of(H))) * R + r;
  const float norm = ax == 0 ? 1.f / q.count : 1.f;
  for (int x0 = 0; x0 < S; x0 += 256) {
    const int x = x0 + threadIdx.x;
    int first = 0xff, last = 0;
    if (x < S)
      for (int p = 0; p < P; ++p) {
        const float v = axis_weight_at(x, st, p, bn, gr, S, order);
        w[(size_t)p * S + x] = v * norm;
        if (v != 0.f) {
          first = min(first, p);
          last = p;
        }
      }
    // over the tile's 4 positions (4 consecutive lanes)
#pragma unroll
    for (int d = 1; d < kGT; d <<= 1) {
      first = min(first, __shfl_xor(first, d));
      last = max(last, __shfl_xor(last, d));
    }
    if (x < S && x % kGT == 0) t[(size_t)(x / kGT) * R] = first == 0xff ? kNoBins : (uint32_t)(first | (last << 8));
  }
}

// top [R, C, bins] -> [R, bins, C].  A block copies kCopyChannels channels of one roi, which are one
// contiguous run: read in 16-byte pieces into LDS as they lie (at the run's alignment), written a
// bin at a time, a lane per channel.  Also marks rois that hold an infinity or NaN.
template <typename T> constexpr int kCopyChannels = sizeof(T) == 4 ? 32 : 64;   // at most 48 KB of LDS
// Fewer channels where the call would have fewer blocks than the chip CUs: 2 to 6 us of a call of 9 to
// 35 rois over 64 to 256 channels.
constexpr int kCopyFewChannels = 16, kCopyFewBlocks = 256;
template <typename T, int CB>
__global__ __launch_bounds__(256) void grad_channels_last_kernel(const T *top, T *top_cl, uint32_t *tr, int C, int bins,
                                                                 int ntz, int R) {
  extern __shared__ __align__(16) unsigned char copy_lds[];
  constexpr int E = 16 / (int)sizeof(T);
  T *l = reinterpret_cast<T *>(copy_lds);
  const int t = threadIdx.x, r = blockIdx.x, c0 = blockIdx.y * CB, nc = min(CB, C - c0);
  const T *src = top + ((int64_t)r * C + c0) * bins;
  const int n = nc * bins, shift = (int)((reinterpret_cast<uintptr_t>(src) & 15u) / sizeof(T));
  const int lead = min(n, (E - shift) % E);   // elements before the first 16-byte boundary
  bool bad = false;
  const auto check = [&](T v) { bad |= !(fabsf(to_f(v)) < INFINITY); };
  if (t < lead) {
    l[shift + t] = src[t];
    check(src[t]);
  }
  const int pieces = (n - lead) / E;
  for (int p = t; p < pieces; p += 256) {
    const uint4 u = *reinterpret_cast<const uint4 *>(src + lead + p * E);
    *reinterpret_cast<uint4 *>(l + shift + lead + p * E) = u;
    const T *e = reinterpret_cast<const T *>(&u);
#pragma unroll
    for (int k = 0; k < E; ++k) check(e[k]);
  }
  for (int e = lead + pieces * E + t; e < n; e += 256) {
    l[shift + e] = src[e];
    check(src[e]);
  }
  const bool any = __syncthreads_or(bad) != 0;
  if (any)
    for (int z = t; z < ntz; z += 256) atomicOr(&tr[(size_t)z * R + r], kNonFinite);
  const int ch = t % CB;
  T *dst = top_cl + (int64_t)r * bins * C + c0 + ch;
  if (ch < nc)
    for (int b = t / CB; b < bins; b += 256 / CB) dst[(int64_t)b * C] = l[shift + ch * bins + b];
}

// How many rois reach each tile (at most 255 counted): a wave per tile of one batch item.
template <typename T>
__global__ __launch_bounds__(256) void roi_tile_count_kernel(const T *__restrict__ rois, const uint32_t *__restrict__ tr,
                                                             uint8_t *__restrict__ counts, int ntz, int nty, int ntx,
                                                             int R, int tiles) {
  const int lane = threadIdx.x & 63, tile = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile >= tiles) return;
  const int tx = tile % ntx, ty = tile / ntx % nty, tz = tile / (ntx * nty) % ntz, n = tile / (ntx * nty * ntz);
  int c = 0;
#pragma unroll 4
  for (int r = lane; r < R; r += 64) {
    const uint32_t z = tr[(size_t)tz * R + r], y = tr[(size_t)(ntz + ty) * R + r], x = tr[(size_t)(ntz + nty + tx) * R + r];
    const int item = (int)to_f(rois[(int64_t)r * 7]);
    c += item == n && first_bin(z) <= last_bin(z) && first_bin(y) <= last_bin(y) && first_bin(x) <= last_bin(x) ? 1 : 0;
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d);
  if (lane == 0) counts[tile] = (uint8_t)min(c, 255);
}

// Tiles by decreasing count (a counting sort in one block): order[rank] = tile.
__global__ __launch_bounds__(1024) void roi_tile_order_kernel(const uint8_t *counts, unsigned short *order, int tiles) {
  __shared__ uint32_t at_l[256];
  const int t = threadIdx.x;
  if (t < 256) at_l[t] = 0;
  __syncthreads();
  for (int i = t; i < tiles; i += 1024) atomicAdd(&at_l[255 - counts[i]], 1u);
  __syncthreads();
  if (t < 64) {   // exclusive scan, 4 levels a lane
    uint32_t v[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = at_l[4 * t + k];
      sum += v[k];
    }
    uint32_t inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t u = __shfl_up(inc, d);
      if (t >= d) inc += u;
    }
    uint32_t at = inc - sum;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      at_l[4 * t + k] = at;
      at += v[k];
    }
  }
  __syncthreads();
  for (int i = t; i < tiles; i += 1024) order[atomicAdd(&at_l[255 - counts[i]], 1u)] = (unsigned short)i;
}
// How a gather is launched, by its blocks (a wave per tile and 64 channels), the rois R and the tiles
// (figures: at backward()).
constexpr int kGSplitBlocks = 4096, kGSplitRois = 16;   // up to so many blocks, from so many rois: SPLIT
constexpr int kGClearRois = 27;                  // R * 27 <= tiles: many tiles are empty, clear_tiles()
constexpr int kGClearMiddle = 12288;             // up to so many blocks, not SPLIT: in the tiles' middle
constexpr int kGUnordered = 8192, kGOrderRois = 12;     // more blocks, R * 12 > tiles: crowded tiles first
constexpr int kGOrdered = 65535;                 // tiles that are ordered (16-bit numbers)
constexpr int kGList = 192;                      // rois listed at a time

// One element by a raw buffer load at voffset + soffset.
template <typename T> using RawOf = std::conditional_t<sizeof(T) == 4, uint32_t, unsigned short>;
template <typename T>
__device__ __forceinline__ RawOf<T> load_raw(__amdgpu_buffer_rsrc_t rs, uint32_t voff, uint32_t soff) {
  if constexpr (sizeof(T) == 4)
    return __builtin_amdgcn_raw_buffer_load_b32(rs, (int)voff, (int)soff, 0);
  else
    return __builtin_amdgcn_raw_buffer_load_b16(rs, (int)voff, (int)soff, 0);
}

// Zeros for the tiles that no roi reaches (the waves of those tiles then store nothing): a block per
// row of tiles along x and kGClearChannels channels, 4 voxels per thread with the lanes along x.
constexpr int kGClearWords = 8, kGClearChannels = 8;   // 256 tiles at a time
template <typename T, int NT>
__device__ __forceinline__ void clear_tiles(int blk, uint32_t *lds_l, const T *__restrict__ rois,
                                            const uint32_t *__restrict__ tr, T *__restrict__ grad, int C, int D, int H,
                                            int W, int R) {
  const int t = threadIdx.x, ntz = tiles_of(D), nty = tiles_of(H), ntx = tiles_of(W);
  const int parts = (C + kGClearChannels - 1) / kGClearChannels, c0 = blk % parts * kGClearChannels;
  const int ty = blk / parts % nty, tz = blk / parts / nty % ntz, n = blk / parts / nty / ntz;
  const int nc = min(kGClearChannels, C - c0);
  uint32_t *const reached_l = lds_l, *const count_l = lds_l + kGClearWords, *const row_l = count_l + 1;
  for (int tx0 = 0; tx0 < ntx; tx0 += 32 * kGClearWords) {
    const int nt = min(32 * kGClearWords, ntx - tx0);
    if (t <= kGClearWords) lds_l[t] = 0;
    __syncthreads();
    // the rois of this row of tiles, NT at a time, and then every pair of one of them and a tile
    for (int r0 = 0; r0 < R; r0 += NT) {
      const int r = min(r0 + t, R - 1);
      const uint32_t z = tr[(size_t)tz * R + r], y = tr[(size_t)(ntz + ty) * R + r];
      if (r0 + t < R && (int)to_f(rois[(int64_t)r * 7]) == n && first_bin(z) <= last_bin(z) && first_bin(y) <= last_bin(y))
        row_l[atomicAdd(count_l, 1u)] = (uint32_t)r;
      __syncthreads();
      const int pairs = (int)*count_l * nt;
#pragma unroll 4
      for (int i = t; i < pairs; i += NT) {
        const int q = i / nt, k = i - q * nt;
        const uint32_t x = tr[(size_t)(ntz + nty + tx0 + k) * R + row_l[q]];
        if (first_bin(x) <= last_bin(x)) atomicOr(&reached_l[k >> 5], 1u << (k & 31));
      }
      __syncthreads();
      if (t == 0) *count_l = 0;
      __syncthreads();
    }
    for (int k0 = 0; k0 < nt; k0 += NT) {
      // threads in rows of the next power of two above the tiles
      const int m = min(NT, nt - k0), shift = m > 1 ? 32 - __clz(m - 1) : 0, kk = t & ((1 << shift) - 1), k = k0 + kk;
      if (kk >= m || ((reached_l[k >> 5] >> (k & 31)) & 1u)) continue;
      const int x0 = (tx0 + k) * kGT;
      for (int row = t >> shift; row < nc * kGT * kGT; row += NT >> shift) {
        const int c = c0 + row / (kGT * kGT), z = tz * kGT + row / kGT % kGT, y = ty * kGT + row % kGT;
        if (z >= D || y >= H) continue;
        T *o = grad + ((((int64_t)n * C + c) * D + z) * H + y) * W + x0;
        if (x0 + kGT <= W) {   // at any alignment
          const uint32_t zero[kGT * sizeof(T) / 4] = {};
          __builtin_memcpy(o, zero, sizeof(zero));
        } else {
          for (int x = 0; x < W - x0; ++x) o[x] = from_f<T>(0.f);
        }
      }
    }
    __syncthreads();
  }
}

// SPLIT: a block of kGSplit waves per tile and channel group, each taking every kGSplit-th roi; their
// sums are added in LDS, two planes at a time, wave w those of plane w (launched where a tile's chain
// of rois is the time: few tiles, which run at once or nearly).  `clears` blocks from clear_at on are
// clear_tiles()'s (multiples of 8: the tiles keep their XCDs).
constexpr int kGSplit = 4;
template <typename T, bool SPLIT>
__global__ __launch_bounds__(SPLIT ? 64 * kGSplit : 64, 4) void roi_align3d_backward_gather_kernel(
    const T *__restrict__ top_cl, const T *__restrict__ rois, T *__restrict__ grad, const float *__restrict__ wt,
    const uint32_t *__restrict__ tr, const unsigned short *__restrict__ order, int N, int C, int D, int H,
    int W, int R, int PD, int PH, int PW, int blocks, int run, int clear_at, int clears) {
  constexpr int NW = SPLIT ? kGSplit : 1;
  static_assert(!SPLIT || kGSplit == kGT, "a wave per plane of the tile");
  // the rois' lists; with SPLIT then the waves' sums of two planes (32 KB: four blocks per CU)
  constexpr int kSums = 2 * kGT * kGT;
  __shared__ uint4 lds_l[SPLIT ? NW * kSums * 64 / 4 : kGList];
  static_assert(!SPLIT || NW * kGList <= NW * kSums * 64 / 4, "the lists fit");
  const int lane = threadIdx.x & 63, wave = SPLIT ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  uint4 *const list_l = lds_l + wave * kGList;
  const int ntz = tiles_of(D), nty = tiles_of(H), ntx = tiles_of(W);
  const int ncg = (C + 63) / 64;
  // Tiles differ several times over in the rois that they meet, so a block is one wave (a larger one
  // would hold its slots until its last wave is done), and with `order` the crowded tiles come first.
  // Without it block i runs on XCD i % 8: an XCD takes runs of `run` neighbouring tiles, which read
  // the same rois' bins, and which run of a round of eight it takes moves on, so that no XCD gets
  // only the crowded middle of the volume.
  int bid = blockIdx.x, cg;
  if (bid >= clear_at) {
    bid -= clears;
    if (bid < clear_at) {
      const int blk = bid + clears - clear_at;
      if (blk < N * ntz * nty * ((C + kGClearChannels - 1) / kGClearChannels))
        clear_tiles<T, 64 * NW>(blk, reinterpret_cast<uint32_t *>(lds_l), rois, tr, grad, C, D, H, W, R);
      return;
    }
  }
  if (order) {
    if (bid >= blocks) return;
    cg = bid % ncg;
    bid = order[bid / ncg];
  } else {
    const int seq = bid >> 3, round = seq / run, xcd = (bid + round + round / 4 + round / 16) & 7;
    bid = (round * 8 + xcd) * run + seq % run;
    if (bid >= blocks) return;
    const int tiles = ntx * nty * ntz, ng = bid / tiles;
    cg = ng % ncg;
    bid = ng / ncg * tiles + bid % tiles;
  }
  const int tx = bid % ntx;
  bid /= ntx;
  const int ty = bid % nty;
  bid /= nty;
  const int tz = bid % ntz, n = bid / ntz;
  const int c = cg * 64 + lane;
  const uint32_t cl_bytes = (uint32_t)min(c, C - 1) * (uint32_t)sizeof(T);
  const int z0 = tz * kGT, y0 = ty * kGT, x0 = tx * kGT;
  const size_t wroi = (size_t)D * PD + (size_t)H * PH + (size_t)W * PW;

  // the weight of a roi that a lane fetches: axis (z, y, x; 16 lanes each), bin, position
  const int wax = min(lane >> 4, 2), wbin = (lane >> 2) & 3, wsize = wax == 0 ? D : (wax == 1 ? H : W);
  const uint32_t wfirst = (uint32_t)((wax == 0 ? z0 : (wax == 1 ? D * PD + y0 : D * PD + H * PH + x0)) + (lane & 3));
  const auto lane_of = [](float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
  };
  const auto nonzero = [](float w) { return (__float_as_int(w) << 1) != 0; };

  float acc[kGT][kGT * kGT];
#pragma unroll
  for (int z = 0; z < kGT; ++z)
#pragma unroll
    for (int i = 0; i < kGT * kGT; ++i) acc[z][i] = 0.f;

  // top of one plane of bins, a row of 4 per register quad: a row is reloaded with the next plane's
  // as soon as it is used, so four rows are in flight
  using Raw = RawOf<T>;
  Raw v[4][4];
  const uint32_t row_bytes = (uint32_t)(PW * C) * (uint32_t)sizeof(T), plane_bytes = (uint32_t)PH * row_bytes;
  const auto load_row = [&](Raw(&row)[4], const char *plane, int h, const uint32_t(&off)[4]) {
    // (buffer loads: the row's offset is a scalar operand; bounded by the roi's bins)
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(plane), (short)0, (int)((uint32_t)PD * plane_bytes), 0x00020000);
#pragma unroll
    for (int k = 0; k < 4; ++k) row[k] = load_raw<T>(rs, off[k], (uint32_t)h * row_bytes);
  };
  // x sums of a row of up to 4 bins
  const auto x_sum = [&](float(&t)[kGT], const float(&wx)[4][kGT], const float(&g)[4], int nx) {
#pragma unroll
    for (int x = 0; x < kGT; ++x) t[x] = wx[0][x] * g[0];
#pragma unroll
    for (int k = 1; k < 4; ++k)
      if (k < nx)
#pragma unroll
        for (int x = 0; x < kGT; ++x) t[x] += wx[k][x] * g[k];
  };

  int roi = 0;
  uint32_t b_zy = 0, b_x = 0;   // bins of the roi to come: z | y << 16, x | flag << 16
  const auto take = [&](int i) {
    const uint4 e = list_l[i];
    roi = __builtin_amdgcn_readfirstlane((int)e.x);
    b_zy = (uint32_t)__builtin_amdgcn_readfirstlane((int)e.y);
    b_x = (uint32_t)__builtin_amdgcn_readfirstlane((int)e.z);
  };
  const auto count = [](uint32_t w) { return last_bin(w) - first_bin(w) + 1; };
  const auto weights = [&]() {
    const uint32_t zy = wax == 0 ? b_zy : b_zy >> 16, word = wax == 2 ? b_x : zy;
    const int p = first_bin(word) + wbin, last = last_bin(word);
    // positions past the volume's end read the next row: their sums are not stored
    const float w = (wt + (size_t)roi * wroi)[wfirst + (uint32_t)(min(p, last) * wsize)];
    return p <= last ? w : 0.f;
  };
  const uint32_t bin_bytes = (uint32_t)C * (uint32_t)sizeof(T), roi_bytes = (uint32_t)(PD * PH * PW) * bin_bytes;
  const auto first_plane = [&]() {
    const uint32_t bin = (uint32_t)((first_bin(b_zy) * PH + first_bin(b_zy >> 16)) * PW + first_bin(b_x));
    return reinterpret_cast<const char *>(top_cl) + ((uint64_t)(uint32_t)roi * roi_bytes + bin * bin_bytes);
  };
  const auto offsets = [&](uint32_t(&off)[4], int nx) {   // bytes: a bin's channel, at most 384 bins away
#pragma unroll
    for (int k = 0; k < 4; ++k) off[k] = (uint32_t)min(k, nx - 1) * bin_bytes + cl_bytes;
  };

  bool reached = false;
  for (int r0 = 0; r0 * NW + wave < R;) {
    // the next rois of batch item n that reach the tile, in index order: from the front those with
    // at most 4 bins on every axis of it and only finite values (nearly all), from the back the
    // others
    int narrow = 0, wide = 0;
    for (; r0 * NW + wave < R && narrow + wide <= kGList - 64; r0 += 64) {
      const int r = (r0 + lane) * NW + wave, q = min(r, R - 1);
      const uint32_t z = tr[(size_t)tz * R + q], y = tr[(size_t)(ntz + ty) * R + q], x = tr[(size_t)(ntz + nty + tx) * R + q];
      const int item = (int)to_f(rois[(int64_t)q * 7]);
      const int cz = last_bin(z) - first_bin(z), cy = last_bin(y) - first_bin(y), cx = last_bin(x) - first_bin(x);
      const bool hit = r < R && item == n && min(cz, min(cy, cx)) >= 0, big = max(cz, max(cy, cx)) > 3 || (z & kNonFinite) != 0;
      const uint64_t mn = __ballot(hit && !big), mw = __ballot(hit && big), below = (1ull << lane) - 1ull;
      const uint4 e = make_uint4((uint32_t)r, (z & 0xffffu) | (y << 16), (x & 0xffffu) | ((z & kNonFinite) >> 15), 0u);
      if (hit) list_l[big ? kGList - 1 - (wide + __popcll(mw & below)) : narrow + __popcll(mn & below)] = e;
      narrow += __popcll(mn);
      wide += __popcll(mw);
    }
    __builtin_amdgcn_wave_barrier();
    reached = reached || narrow + wide > 0;

    if (narrow > 0) {
      take(0);
      uint32_t off[4];
      const char *plane = first_plane();
      float w_ahead = weights();
      int ahead_ny = count(b_zy >> 16), ahead_nx = count(b_x);
      offsets(off, ahead_nx);
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        load_row(v[h], plane, min(h, ahead_ny - 1), off);
        __builtin_amdgcn_sched_barrier(0);   // in the order of their use
      }
      for (int i = 1; i <= narrow; ++i) {
        const float w = w_ahead;
        uint64_t set = __ballot(w != 0.f);   // which weights are not 0, by lane
        int nx = ahead_nx, ny = ahead_ny;
        const int nz = count(b_zy);
        if (i < narrow) {
          take(i);
          w_ahead = weights();
        }
        float wx[4][kGT];
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int x = 0; x < kGT; ++x) wx[b][x] = lane_of(w, 32 + b * 4 + x);
        for (int d = 0; d < nz; ++d) {
          // the plane to load: this roi's next, then the next roi's first (at the end: this one again)
          if (d + 1 < nz) {
            plane += plane_bytes;
          } else if (i < narrow) {
            plane = first_plane();
            ahead_ny = count(b_zy >> 16);
            ahead_nx = count(b_x);
            offsets(off, ahead_nx);
          }
          // (opaque: the compiler would keep every test below in scalar registers over the loop)
          asm volatile("" : "+s"(set), "+s"(nx), "+s"(ny));
          float u[kGT * kGT];
#pragma unroll
          for (int j = 0; j < kGT * kGT; ++j) u[j] = 0.f;
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            float g[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              g[k] = to_f(__builtin_bit_cast(T, v[h][k]));
              asm volatile("" : "+v"(g[k]));   // here: v[h][k] is free for the load
            }
            __builtin_amdgcn_sched_barrier(0);   // or the loads move up and need registers of their own
            load_row(v[h], plane, min(h, ahead_ny - 1), off);
            __builtin_amdgcn_sched_barrier(0);
            if (h < ny) {
              float t[kGT];
              x_sum(t, wx, g, nx);
#pragma unroll
              for (int y = 0; y < kGT; ++y)
                if ((set >> (16 + h * 4 + y)) & 1) {
                  const float wy = lane_of(w, 16 + h * 4 + y);
#pragma unroll
                  for (int x = 0; x < kGT; ++x) u[y * kGT + x] += wy * t[x];
                }
            }
          }
#pragma unroll
          for (int z = 0; z < kGT; ++z)
            if ((set >> (d * 4 + z)) & 1) {
              const float wz = lane_of(w, d * 4 + z);
#pragma unroll
              for (int j = 0; j < kGT * kGT; ++j) acc[z][j] += wz * u[j];
            }
        }
      }
    }

    // bins smaller than the voxels, or values that are not finite: the bins along x four at a time,
    // row by row
    for (int i = 0; i < wide; ++i) {
      take(kGList - 1 - i);
      const bool clean = (b_x >> 16) == 0;
      const float *wz = wt + (size_t)roi * wroi + z0, *wy = wt + (size_t)roi * wroi + (size_t)D * PD + y0,
                  *wx = wt + (size_t)roi * wroi + (size_t)D * PD + (size_t)H * PH + x0;
      for (int px = first_bin(b_x); px <= last_bin(b_x & 0xffffu); px += 4) {
        const int nx = min(4, last_bin(b_x) - px + 1);
        float wxr[4][kGT];
        uint32_t off[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
          for (int x = 0; x < kGT; ++x) wxr[k][x] = k < nx ? wx[(px + k) * W + x] : 0.f;
        offsets(off, nx);
        for (int pd = first_bin(b_zy); pd <= last_bin(b_zy); ++pd) {
          float u[kGT * kGT];
#pragma unroll
          for (int j = 0; j < kGT * kGT; ++j) u[j] = 0.f;
          const char *plane = reinterpret_cast<const char *>(top_cl) +
                              ((uint64_t)(uint32_t)roi * roi_bytes + ((uint32_t)pd * plane_bytes + (uint32_t)px * bin_bytes));
          const int last_ph = last_bin(b_zy >> 16);
          for (int ph0 = first_bin(b_zy >> 16); ph0 <= last_ph; ph0 += 4) {   // four rows in flight
#pragma unroll
            for (int h = 0; h < 4; ++h) load_row(v[h], plane, min(ph0 + h, last_ph), off);
#pragma unroll
            for (int h = 0; h < 4; ++h) {
              const int ph = ph0 + h;
              if (ph > last_ph) break;
              float g[4], t[kGT];
#pragma unroll
              for (int k = 0; k < 4; ++k) g[k] = to_f(__builtin_bit_cast(T, v[h][k]));
              if (clean) {
                x_sum(t, wxr, g, nx);
              } else {   // 0 * infinity must not reach a voxel outside the bin
#pragma unroll
                for (int x = 0; x < kGT; ++x) t[x] = 0.f;
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                  for (int x = 0; x < kGT; ++x)
                    if (nonzero(wxr[k][x])) t[x] += wxr[k][x] * g[k];
              }
#pragma unroll
              for (int y = 0; y < kGT; ++y) {
                const float w = wy[ph * H + y];
                if (nonzero(w))
#pragma unroll
                  for (int x = 0; x < kGT; ++x) u[y * kGT + x] += w * t[x];
              }
            }
          }
#pragma unroll
          for (int z = 0; z < kGT; ++z) {
            const float w = wz[pd * D + z];
            if (nonzero(w))
#pragma unroll
              for (int j = 0; j < kGT * kGT; ++j) acc[z][j] += w * u[j];
          }
        }
      }
    }
    __builtin_amdgcn_wave_barrier();   // the list is read before the next rois are written to it
  }
  // nothing to store where the zeros come from clear_tiles(), no sums to add where there are none
  const bool any = (SPLIT ? __syncthreads_or(reached) != 0 : reached) || clears == 0;
  if constexpr (SPLIT) {   // wave w: the sums of plane w, in acc[0]
    if (any) {
      float(*sums_l)[kSums][64] = reinterpret_cast<float(*)[kSums][64]>(lds_l);
      float sum[kGT * kGT];
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kSums; ++j) sums_l[wave][j][lane] = acc[2 * half + j / (kGT * kGT)][j % (kGT * kGT)];
        __syncthreads();
        if (wave >> 1 == half)
#pragma unroll
          for (int j = 0; j < kGT * kGT; ++j) {
            sum[j] = sums_l[0][(wave & 1) * kGT * kGT + j][lane];
#pragma unroll
            for (int k = 1; k < NW; ++k) sum[j] += sums_l[k][(wave & 1) * kGT * kGT + j][lane];
          }
      }
#pragma unroll
      for (int j = 0; j < kGT * kGT; ++j) acc[0][j] = sum[j];
    }
  }
  if (c >= C || !any) return;
  T *o = grad + ((int64_t)n * C + c) * D * H * W;
#pragma unroll
  for (int z = 0; z < (SPLIT ? 1 : kGT); ++z)
#pragma unroll
    for (int y = 0; y < kGT; ++y) {
      const int zz = z0 + (SPLIT ? wave : z);
      if (zz >= D || y0 + y >= H) continue;
      T *row = o + ((int64_t)zz * H + (y0 + y)) * W + x0;
      T e[kGT];
#pragma unroll
      for (int x = 0; x < kGT; ++x) e[x] = from_f<T>(acc[z][y * kGT + x]);
      if (x0 + kGT <= W) {   // one 8- or 16-byte store, at any alignment
        if constexpr (sizeof(T) == 4) {
          __builtin_memcpy(row, e, sizeof(e));
        } else {
          uint32_t h[2];
#pragma unroll
          for (int k = 0; k < 2; ++k)
            h[k] = (uint32_t)__builtin_bit_cast(unsigned short, e[2 * k]) |
                   ((uint32_t)__builtin_bit_cast(unsigned short, e[2 * k + 1]) << 16);
          __builtin_memcpy(row, h, sizeof(h));
        }
      } else {
#pragma unroll
        for (int x = 0; x < kGT; ++x)
          if (x0 + x < W) row[x] = e[x];
      }
    }
}

// ---------------------------------------------------------------------------------------------
// Channels-last forward.  With features [N, D, H, W, C] a voxel's C channels are one contiguous
// row, so a sample's corner is one 16-byte (8-channel) load per lane and the 32 lanes of a
// 256-channel bin read whole 128-byte lines; from [N, C, D, H, W] every corner of every channel
// is a separate 2- or 4-byte access.  A block owns bpb consecutive bins of the (ph, pw) plane
// of one (roi, pd): lane group cg takes channels 8 cg .. 8 cg + 7 of one bin, the rounded
// results are staged in LDS and written out as [R, C, PD, PH, PW] runs of bpb elements per
// channel.  The blocks of a roi run on one XCD, whose L2 then serves the overlap of their taps.
// The arithmetic is the NCDHW kernel's, term by term, so both give the same bits.
// Measured (bf16 [2, 256, 32, 64, 64], 512 rois of 4-32 voxels, 7^3 bins, 2 samples per axis): 430 us
// with every lane's own tap lists, one weight product, multiplication and addition per tap and
// channel; 305 us with the lists made once per bin in LDS and the sum taken along x, y, z in fused
// multiply-adds, four loads at a time (fp32 [1, 120, 21, 45, 77], 150 rois, adaptive samples: 130 ->
// 72 us).  Bound by the lines that the rois' overlapping regions fetch past L2, about 2 GB; loading
// only the taps that a bin has, or two rows at a time, measured the same (306, 307 us).
constexpr int kClChannels = 8;                  // channels per lane

template <typename T>
__device__ __forceinline__ void load8(const T *p, float f[8]) {
  if constexpr (sizeof(T) == 4) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
    f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
  } else {
    const uint4 u = *reinterpret_cast<const uint4 *>(p);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const unsigned short s = (unsigned short)((k & 1) ? (w[k >> 1] >> 16) : (w[k >> 1] & 0xffffu));
      f[k] = to_f(__builtin_bit_cast(T, s));
    }
  }
}

// Bins per block: one per lane group (256 / (C / 8) groups), the (ph, pw) plane of a (roi, pd)
// cut into equal parts (one bin per thread: more blocks in flight).
inline void cl_split(int C, int PHW, int &bpb, int &parts) {
  const int slots = 256 / (C / kClChannels);
  parts = (PHW + slots - 1) / slots;
  bpb = (PHW + parts - 1) / parts;
}

inline bool cl_supported(int C) { return C > 0 && C % kClChannels == 0 && C / kClChannels <= 256; }

// The taps of one axis of one bin, in LDS.
template <int NT>
struct TapList {
  int n, over, pos[NT];
  float w[NT];
};

// WIDE: lists of 8 taps, for grids of more than 2 samples per axis (launched when sampling_ratio is
// adaptive or above 2; without it the kernel needs fewer registers).  The tap lists of the block's
// bins (one per axis and bin, z's once) are made by a thread each and read from LDS: the C / 8 lanes
// of a bin each made all three before, 40 % of the kernel's instructions.
template <typename T, bool WIDE>
__global__ __launch_bounds__(256) void roi_align3d_forward_cl_kernel(const T *__restrict__ feat, const T *__restrict__ rois,
                                                                     T *__restrict__ out, int N, int C, int D, int H,
                                                                     int W, int PD, int PH, int PW, float scale, int sr,
                                                                     int order, int bpb, int parts, int nblk) {
#pragma clang fp contract(off)
  constexpr int NT = WIDE ? kSepTaps : 4;
  using Taps = TapList<NT>;
  extern __shared__ __align__(16) unsigned char cl_lds[];
  Taps *list_l = reinterpret_cast<Taps *>(cl_lds);          // y of every bin, x of every bin, z
  T *res = reinterpret_cast<T *>(list_l + 2 * bpb + 1);     // [C][bpb]
  __shared__ float count_l;
  __shared__ int item_l;
  // block i runs on XCD i % 8: XCD x takes the x-th eighth of the (roi, pd, part) blocks, so a
  // roi's blocks share one L2 (gridDim.x is a multiple of 8; nblk blocks are real)
  const unsigned blk = (blockIdx.x & 7u) * (gridDim.x / 8u) + (blockIdx.x >> 3);
  if (blk >= (unsigned)nblk) return;
  const int r = (int)(blk / (unsigned)(PD * parts));
  const int rem = (int)(blk % (unsigned)(PD * parts));
  const int pd = rem / parts, b0 = (rem - pd * parts) * bpb;
  const int nbin = min(bpb, PH * PW - b0);
  const int CG = C / kClChannels;
  const int tid = threadIdx.x, cg = tid % CG, bin = tid / CG;   // bpb * CG <= 256: one bin per lane group
  for (int i = tid; i < 2 * nbin + 1; i += 256) {
    const Roi q = roi_setup(rois, r, scale, sr, PD, PH, PW);
    const int ax = i == 2 * nbin ? 0 : (i < nbin ? 1 : 2), b = b0 + (i < nbin ? i : i - nbin);
    const int p = ax == 0 ? pd : (ax == 1 ? b / PW : b % PW);
    const AxisTaps<NT> t = bin_taps_n<NT>(ax == 0 ? q.sd : (ax == 1 ? q.sh : q.sw), p, ax == 0 ? q.bd : (ax == 1 ? q.bh : q.bw),
                                          ax == 0 ? q.gd : (ax == 1 ? q.gh : q.gw), ax == 0 ? D : (ax == 1 ? H : W), order);
    Taps &l = list_l[i < nbin ? i : (i < 2 * nbin ? bpb + i - nbin : 2 * bpb)];
    l.n = t.n;
    l.over = t.over;
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      l.pos[k] = t.pos[k];
      l.w[k] = t.w[k];
    }
    if (ax == 0) {
      count_l = q.count;
      item_l = q.b;
    }
  }
  __syncthreads();
  const bool inb = item_l >= 0 && item_l < N;
  const int64_t vol = (int64_t)D * H * W;
  const T *base = feat + (int64_t)(inb ? item_l : 0) * vol * C + cg * kClChannels;
  if (bin < nbin) {
    float acc[kClChannels];
#pragma unroll
    for (int c = 0; c < kClChannels; ++c) acc[c] = 0.f;
    const Taps &ty = list_l[bin], &tz = list_l[2 * bpb];
    const Taps tx = list_l[bpb + bin];
    if (inb && !tz.over && !ty.over && !tx.over) {
      // along x, then y, then z (the NCDHW kernel's sums)
      const int nz = tx.n > 0 && ty.n > 0 ? tz.n : 0, ny = ty.n;
      for (int kz = 0; kz < nz; ++kz) {
        const uint32_t plane = (uint32_t)tz.pos[kz] * (uint32_t)H;
        float u[kClChannels];
#pragma unroll
        for (int c = 0; c < kClChannels; ++c) u[c] = 0.f;
        for (int ky = 0; ky < ny; ++ky) {
          const uint32_t rowo = (plane + (uint32_t)ty.pos[ky]) * (uint32_t)W;
          const float wy = ty.w[ky];
          float t[kClChannels];
          // four loads in flight; past the last tap its row again, left out of the sum
#pragma unroll
          for (int x0 = 0; x0 < NT; x0 += 4) {
            if (x0 > 0 && x0 >= tx.n) break;
            float v[4][kClChannels];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const int pos = x0 + k < tx.n ? tx.pos[x0 + k] : tx.pos[x0];
              load8(base + (rowo + (uint32_t)pos) * (uint32_t)C, v[k]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (x0 + k < tx.n)
#pragma unroll
                for (int c = 0; c < kClChannels; ++c) t[c] = tap_add(x0 + k, tx.w[x0 + k], v[k][c], t[c]);
          }
#pragma unroll
          for (int c = 0; c < kClChannels; ++c) u[c] = tap_add(ky, wy, t[c], u[c]);
        }
#pragma unroll
        for (int c = 0; c < kClChannels; ++c) acc[c] = tap_add(kz, tz.w[kz], u[c], acc[c]);
      }
    } else if (WIDE && inb) {   // too many taps on some axis: sample by sample
      const Roi q = roi_setup(rois, r, scale, sr, PD, PH, PW);
      const int ph = (b0 + bin) / PW, pw = (b0 + bin) % PW;
      for (int iz = 0; iz < q.gd; ++iz) {
        const float z = sample_coord(q.sd, pd, q.bd, iz, q.gd);
        for (int iy = 0; iy < q.gh; ++iy) {
          const float y = sample_coord(q.sh, ph, q.bh, iy, q.gh);
          for (int ix = 0; ix < q.gw; ++ix) {
            const float x = sample_coord(q.sw, pw, q.bw, ix, q.gw);
            int64_t off[8];
            float w[8];
            if (!corners(z, y, x, D, H, W, order, off, w)) continue;
            float s[kClChannels];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              float v[kClChannels];
              load8(base + (uint32_t)off[k] * (uint32_t)C, v);
#pragma unroll
              for (int c = 0; c < kClChannels; ++c) s[c] = k == 0 ? w[0] * v[c] : s[c] + w[k] * v[c];
            }
#pragma unroll
            for (int c = 0; c < kClChannels; ++c) acc[c] = acc[c] + s[c];
          }
        }
      }
    }
#pragma unroll
    for (int c = 0; c < kClChannels; ++c) res[(cg * kClChannels + c) * nbin + bin] = from_f<T>(acc[c] / count_l);
  }
  __syncthreads();
  // channel c's bins b0 .. b0 + nbin - 1 of plane pd are nbin consecutive output elements
  T *o = out + ((int64_t)r * C * PD + pd) * PH * PW + b0;
  const int64_t cs = (int64_t)PD * PH * PW;
  for (int e = tid; e < C * nbin; e += 256) {
    const int c = e / nbin, k = e - c * nbin;
    o[c * cs + k] = res[e];
  }
}

// [N, C, V] -> [N, V, C] in T, through 64 x 64 LDS tiles.  Global accesses are 16-byte pieces
// (E = 16 / sizeof(T) elements: E voxels of a channel on the way in, E channels of a voxel on
// the way out, 8 lanes per 128-byte line) when `vec` (C and V multiples of E, both buffers
// 16-byte aligned); element by element otherwise.
template <typename T>
__global__ __launch_bounds__(256) void ncdhw_to_channels_last_kernel(const T *src, T *dst, int C, int64_t V, bool vec) {
  constexpr int E = 16 / (int)sizeof(T);
  __shared__ T t[64][64 + 2];   // [voxel][channel]; rows 4 bytes apart from a multiple of 128
  const int tid = threadIdx.x;
  const int64_t v0 = (int64_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  const int64_t n = blockIdx.z;
  const T *s = src + n * C * V;
  T *d = dst + n * V * C;
  if (vec) {
    constexpr int PPL = 64 / E;   // pieces per 64-element line
#pragma unroll
    for (int i = 0; i < 64 * PPL / 256; ++i) {
      const int p = i * 256 + tid, cc = p / PPL, vv = (p % PPL) * E;
      if (c0 + cc < C && v0 + vv < V) {
        const uint4 u = *reinterpret_cast<const uint4 *>(s + (int64_t)(c0 + cc) * V + v0 + vv);
        const T *e = reinterpret_cast<const T *>(&u);
#pragma unroll
        for (int k = 0; k < E; ++k) t[vv + k][cc] = e[k];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * PPL / 256; ++i) {
      const int p = i * 256 + tid, vv = p / PPL, cc = (p % PPL) * E;
      if (v0 + vv < V && c0 + cc < C) {
        uint4 u;
        T *e = reinterpret_cast<T *>(&u);
#pragma unroll
        for (int k = 0; k < E; ++k) e[k] = t[vv][cc + k];
        *reinterpret_cast<uint4 *>(d + (v0 + vv) * C + c0 + cc) = u;
      }
    }
    return;
  }
  const int lane = tid & 63, row = tid >> 6;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int cc = i * 4 + row;
    if (c0 + cc < C && v0 + lane < V) t[lane][cc] = s[(int64_t)(c0 + cc) * V + v0 + lane];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int vv = i * 4 + row;
    if (v0 + vv < V && c0 + lane < C) d[(v0 + vv) * C + c0 + lane] = t[vv][lane];
  }
}

template <typename T>
int forward(const void *features, const void *rois, void *output, int N, int C, int D, int H, int W, int R, int PD,
            int PH, int PW, float scale, int sr, int order, hipStream_t st) {
  const T *f = static_cast<const T *>(features);
  const T *ro = static_cast<const T *>(rois);
  T *o = static_cast<T *>(output);
  // channels per thread: 4 (1 when C % 4 != 0); more channels per thread share each bin's
  // set-up but leave fewer threads to hide the gathers' latency (bench workload, separable
  // path: 1 / 2 / 4 / 8 / 16 channels 1.90 / 1.46 / 1.37 / 1.52 / 2.32 ms)
  constexpr int kC = 4;
  const int cpt = C % kC == 0 ? kC : 1;
  const int64_t total = (int64_t)R * (C / cpt) * PD * PH * PW;
  const unsigned grid = (unsigned)((total + 255) / 256);
  if (cpt == kC)
    hipLaunchKernelGGL((roi_align3d_forward_kernel<T, kC>), dim3(grid), dim3(256), 0, st, f, ro, o, N, C, D, H, W, R, PD,
                       PH, PW, scale, sr, order);
  else
    hipLaunchKernelGGL((roi_align3d_forward_kernel<T, 1>), dim3(grid), dim3(256), 0, st, f, ro, o, N, C, D, H, W, R, PD,
                       PH, PW, scale, sr, order);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

template <typename T>
int forward_cl(const void *features_cl, const void *rois, void *output, int N, int C, int D, int H, int W, int R, int PD,
               int PH, int PW, float scale, int sr, int order, hipStream_t st) {
  int bpb = 0, parts = 0;
  cl_split(C, PH * PW, bpb, parts);
  const int64_t blocks = (int64_t)R * PD * parts;
  const int64_t grid = (blocks + 7) / 8 * 8;   // a multiple of 8: the kernel maps blocks to XCDs
  if (grid >= ((int64_t)1 << 31)) return OPS3D_FDA_EINVAL;
  const bool narrow = sr > 0 && sr <= 2;
  const size_t lds = (size_t)C * bpb * sizeof(T) + (size_t)(2 * bpb + 1) * (narrow ? sizeof(TapList<4>) : sizeof(TapList<kSepTaps>));
  if (narrow)   // every roi's grid is separable with 4 taps per axis
    hipLaunchKernelGGL((roi_align3d_forward_cl_kernel<T, false>), dim3((unsigned)grid), dim3(256), lds, st,
                       static_cast<const T *>(features_cl), static_cast<const T *>(rois), static_cast<T *>(output), N,
                       C, D, H, W, PD, PH, PW, scale, sr, order, bpb, parts, (int)blocks);
  else
    hipLaunchKernelGGL((roi_align3d_forward_cl_kernel<T, true>), dim3((unsigned)grid), dim3(256), lds, st,
                       static_cast<const T *>(features_cl), static_cast<const T *>(rois), static_cast<T *>(output), N,
                       C, D, H, W, PD, PH, PW, scale, sr, order, bpb, parts, (int)blocks);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

template <typename T>
int to_channels_last(const void *features, void *features_cl, int N, int C, int64_t V, hipStream_t st) {
  hipLaunchKernelGGL((ncdhw_to_channels_last_kernel<T>), dim3((unsigned)((V + 63) / 64), (unsigned)((C + 63) / 64), N),
                     dim3(256), 0, st, static_cast<const T *>(features), static_cast<T *>(features_cl), C, V,
                     C % (16 / (int)sizeof(T)) == 0 && V % (16 / (int)sizeof(T)) == 0 &&
                         ((reinterpret_cast<uintptr_t>(features) | reinterpret_cast<uintptr_t>(features_cl)) & 15u) == 0);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

// Bytes of the gather backward's per-roi axis tables, rounded up to 16 (the channels-last copy of
// grad_output follows them).
inline size_t gather_tables_bytes(int R, int D, int H, int W, int PD, int PH, int PW) {
  const size_t b = (size_t)R * ((size_t)D * PD + (size_t)H * PH + (size_t)W * PW + (size_t)D + H + W) * 4;
  return (b + 15) & ~(size_t)15;
}

// Backward.  Measured on bf16 [2, 256, 32, 64, 64], 512 rois of 4-32 voxels, 7^3 bins, one MI355X:
// tables 7, copy 47, tile counts and order 14, gather 445 us (0.86 ms forward and backward); before,
// with a block per 4 x 8 x 8 voxels and 16 channels that staged its rois' bins in LDS, a thread per
// voxel: tables 6, copy 75, gather 1572 us (2.10 ms).  The gather issues 132 M vector instructions
// (40 % of the issue slots at four waves per SIMD) and waits for its loads for most of the rest:
// 340 K visits of a roi to a tile and channel group, each 2 to 4 planes of 4 rows.  Steps: the first
// form (blocks of four waves, dynamic loops, weights by scalar loads) 943 us; rows loaded a plane
// ahead and weights fetched by the lanes 680; one wave per block 537; crowded tiles first 500 (-45);
// no spilled registers 445, four rows at a time where bins are smaller than voxels 435.  Without
// `order` an XCD's runs of 8 / 32 / 128 / 512 tiles measured 554 / 535 / 522 / 540 us.  Joining the
// tiles of a block of two or four waves in LDS, to store longer runs, 502 / 520 us against 492; three
// waves per SIMD 542.
// The rules of a launch, by the GPU time of all passes of a call (us; 7^3 bins, 2 samples, rois of
// 4-32 voxels where not said; f: fp32, others 16 bits; "N x" batch items):
//   SPLIT / one wave per tile: 17x24x28, 32 channels, 404 rois of 4-16 (252 blocks) 357 / 1119;
//     26x35x31, 64, 21 of 4-16 (504) 49 / 59; 12x40x40, 200, 90 of 4-24, 3^3 bins (1200) 39 / 60;
//     10x23x65, 256, 213 of 4-16 (1224) 199 / 411; 30x60x60 f, 32, 60 (1800) 58 / 68; 24x48x48, 256,
//     300 of 4-24 (3456) 260 / 322, 30 rois 82 / 77; 32x64x64, 192, 200 rois, 5^3 (6144) 132 / 130.
//     Four blocks per CU: with 64 KB of sums, two, 213 rois took 267 and 21 rois 53.
//   clear_tiles() / every wave stores: 2 x 32x64x64, 256, 64 rois of 4-16 (4096 tiles) 128 / 179; 110 of
//     4-16 168 / 205; 150 of 4-32 213 / 216; f, 16 rois 124 / 208; 2 x 41x50x50, 256, 35 of 4-16, one
//     sample, nearest (3718) 75 / 116, of 4-32 103 / 125; 23x33x89, 250, 46 of 3-18, 3^3 (1242) 44 / 51,
//     f 62 / 66; 24x48x48, 256, 9 rois (864) 46 / 47.  At 27 tiles per roi, rois of 4-30 reach nearly
//     all tiles and lose up to 4 %, rois of 3-12 gain 5 to 30 %.  As a pass of its own before the
//     gather 64 rois took 141.  The clear blocks stand behind the tiles', whose end is the chain of the
//     last crowded ones, or, where one-wave tiles run in up to about three rounds, in their middle, or
//     their own latency is the end (behind / middle / before them: 46 rois above (4968 blocks) 60 / 44
//     / 49, f 71 / 62 / 66; 2 x 23x33x89 f, 80 of 3-18 (9936) 123 / 110 / 113; 2 x 40x50x50, 192, 28 of
//     4-30 (10140) 84 / 78 / 87; 2 x 32x64x64 f, 256, 146 of 3-12, 5^3 (16384) 175 / 194 / 197;
//     24x48x48, 256, 30 of 4-24 (SPLIT) 77 / 83 / 83).
//   Crowded tiles first / in place: 2 x 32x64x64, 256, 512 rois 430 / 459, 400 rois 372 / 371, 300
//     rois 321 / 288, 220 rois 292 / 248; 2 x 40x80x80, 512 rois (8000 tiles) 648 / 610, 300 rois
//     521 / 425: the neighbours' stores then meet in no L2.
template <typename T>
int backward(const void *grad_output, const void *rois, void *grad_input, float *acc, int N, int C, int D, int H,
             int W, int R, int PD, int PH, int PW, float scale, int sr, int order, hipStream_t st) {
  if (gather_fits(C, PD, PH, PW)) {
    const int ntz = tiles_of(D), nty = tiles_of(H), ntx = tiles_of(W);
    const int64_t tiles = (int64_t)N * ntz * nty * ntx, blocks = tiles * ((C + 63) / 64);
    // tiles in runs (at least about four rounds of them over the XCDs), the grid whole rounds
    const int64_t run = blocks >= 32 * kGRun ? kGRun : (blocks + 31) / 32, grid = (blocks + 8 * run - 1) / (8 * run) * (8 * run);
    if (grid >= ((int64_t)1 << 31)) return OPS3D_FDA_EINVAL;
    // workspace: the per-roi axis tables, then grad_output channels-last [R, bins, C]
    float *wt = acc;
    uint32_t *tr = reinterpret_cast<uint32_t *>(acc + (size_t)R * ((size_t)D * PD + (size_t)H * PH + (size_t)W * PW));
    T *top_cl = reinterpret_cast<T *>(reinterpret_cast<char *>(acc) + gather_tables_bytes(R, D, H, W, PD, PH, PW));
    const int bins = PD * PH * PW;
    if (R > 0) {
      hipLaunchKernelGGL((roi_axis_table_kernel<T>), dim3((unsigned)R, 3), dim3(256), 0, st,
                         static_cast<const T *>(rois), wt, tr, D, H, W, PD, PH, PW, R, scale, sr, order);
      const auto copy = [&](auto kern, int cb) {
        hipLaunchKernelGGL(kern, dim3((unsigned)R, (unsigned)((C + cb - 1) / cb)), dim3(256),
                           ((size_t)cb * bins + 16 / sizeof(T)) * sizeof(T), st, static_cast<const T *>(grad_output),
                           top_cl, tr, C, bins, ntz, R);
      };
      constexpr int CB = kCopyChannels<T>;
      if ((int64_t)R * ((C + CB - 1) / CB) < kCopyFewBlocks) copy(grad_channels_last_kernel<T, kCopyFewChannels>, kCopyFewChannels);
      else copy(grad_channels_last_kernel<T, CB>, CB);
    }
    // the tiles' order, in the tables' second part beyond the words that tr takes, where it fits
    const int64_t used = (int64_t)R * (ntz + nty + ntx) * 4, spare = (int64_t)R * (D + H + W) * 4 - used;
    unsigned short *order = nullptr;
    const bool split = blocks <= kGSplitBlocks && R >= kGSplitRois;
    const int64_t clears = ((int64_t)N * ntz * nty * ((C + kGClearChannels - 1) / kGClearChannels) + 7) / 8 * 8;
    const bool cleared = (int64_t)R * kGClearRois <= tiles && grid + clears < (1 << 24);
    if (blocks > kGUnordered && (int64_t)R * kGOrderRois > tiles && tiles <= kGOrdered && tiles * 3 <= spare) {
      order = reinterpret_cast<unsigned short *>(reinterpret_cast<char *>(tr) + used);
      uint8_t *counts = reinterpret_cast<uint8_t *>(order + tiles);
      hipLaunchKernelGGL((roi_tile_count_kernel<T>), dim3((unsigned)((tiles + 3) / 4)), dim3(256), 0, st,
                         static_cast<const T *>(rois), tr, counts, ntz, nty, ntx, R, (int)tiles);
      hipLaunchKernelGGL(roi_tile_order_kernel, dim3(1), dim3(1024), 0, st, counts, order, (int)tiles);
    }
    const auto gather = [&](auto kern, int threads) {
      hipLaunchKernelGGL(kern, dim3((unsigned)(grid + (cleared ? clears : 0))), dim3(threads), 0, st, top_cl,
                         static_cast<const T *>(rois), static_cast<T *>(grad_input), wt, tr, order, N, C, D, H, W, R, PD,
                         PH, PW, (int)blocks, (int)run, (int)(split || blocks > kGClearMiddle ? grid : grid / 16 * 8), cleared ? (int)clears : 0);
    };
    if (split) gather(roi_align3d_backward_gather_kernel<T, true>, 64 * kGSplit);
    else gather(roi_align3d_backward_gather_kernel<T, false>, 64);
    return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
  }
  const int64_t nin = (int64_t)N * C * D * H * W;
  const int64_t vol = (int64_t)D * H * W;
  const int64_t nwaves = (int64_t)R * ((C + 63) / 64) * PD * PH;
  const int64_t fg = (nin + 255) / 256;
  const unsigned fill_grid = (unsigned)(fg < 65536 ? (fg > 0 ? fg : 1) : 65536);
  hipLaunchKernelGGL(fill_zero_kernel, dim3(fill_grid), dim3(256), 0, st, acc, nin);
  if (nwaves > 0)
    hipLaunchKernelGGL((roi_align3d_backward_kernel<T>), dim3((unsigned)((nwaves + kBwdWaves - 1) / kBwdWaves)),
                       dim3(64 * kBwdWaves), 0, st, static_cast<const T *>(grad_output), static_cast<const T *>(rois),
                       acc, N, C, D, H, W, R, PD, PH, PW, scale, sr, order);
  hipLaunchKernelGGL((channels_last_to_ncdhw_kernel<T>), dim3((unsigned)((vol + 63) / 64), (unsigned)((C + 63) / 64), N),
                     dim3(256), 0, st, acc, static_cast<T *>(grad_input), C, vol);
  return hipGetLastError() == hipSuccess ? OPS3D_FDA_OK : OPS3D_FDA_ERUNTIME;
}

bool valid(int dtype, int N, int C, int D, int H, int W, int R, int PD, int PH, int PW, int order) {
  return (dtype == OPS3D_FDA_F32 || dtype == OPS3D_FDA_F16 || dtype == OPS3D_FDA_BF16) && N >= 0 && C >= 0 &&
         D > 0 && H > 0 && W > 0 && R >= 0 && PD > 0 && PH > 0 && PW > 0 && (order == 0 || order == 1) &&
         (int64_t)N * C * D * H * W < ((int64_t)1 << 40);
}

}  // namespace ops3d_roi

using namespace ops3d_roi;

extern "C" {

int ops3d_roi_align3d_forward(const void *features, const void *rois, void *output, int dtype, int N, int C, int D,
                              int H, int W, int R, int PD, int PH, int PW, float spatial_scale, int sampling_ratio,
                              int order, void *stream) {
  if (!valid(dtype, N, C, D, H, W, R, PD, PH, PW, order)) return OPS3D_FDA_EINVAL;
  if ((int64_t)R * C == 0) return OPS3D_FDA_OK;
  if (!features || !rois || !output) return OPS3D_FDA_EINVAL;
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case OPS3D_FDA_F32:
      return forward<float>(features, rois, output, N, C, D, H, W, R, PD, PH, PW, spatial_scale, sampling_ratio, order, st);
    case OPS3D_FDA_F16:
      return forward<__half>(features, rois, output, N, C, D, H, W, R, PD, PH, PW, spatial_scale, sampling_ratio, order, st);
    default:
      return forward<__hip_bfloat16>(features, rois, output, N, C, D, H, W, R, PD, PH, PW, spatial_scale, sampling_ratio,
                                     order, st);
  }
}

int ops3d_roi_align3d_channels_last_supported(int dtype, int C, int D, int H, int W, int PW) {
  const int e = dtype == OPS3D_FDA_F32 ? 4 : (dtype == OPS3D_FDA_F16 || dtype == OPS3D_FDA_BF16 ? 2 : 0);
  // element offsets inside one batch item are 32-bit
  return e > 0 && PW > 0 && D > 0 && H > 0 && W > 0 && cl_supported(C) &&
                 (int64_t)D * H * W * C < ((int64_t)1 << 32)
             ? 1
             : 0;
}

int ops3d_roi_align3d_to_channels_last(const void *features, void *features_cl, int dtype, int N, int C, int D, int H,
                                       int W, void *stream) {
  if (!valid(dtype, N, C, D, H, W, 0, 1, 1, 1, 1) || N > 65535 || (C + 63) / 64 > 65535) return OPS3D_FDA_EINVAL;
  const int64_t V = (int64_t)D * H * W;
  if ((int64_t)N * C * V == 0) return OPS3D_FDA_OK;
  if (!features || !features_cl || (V + 63) / 64 >= ((int64_t)1 << 31)) return OPS3D_FDA_EINVAL;
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case OPS3D_FDA_F32: return to_channels_last<float>(features, features_cl, N, C, V, st);
    case OPS3D_FDA_F16: return to_channels_last<__half>(features, features_cl, N, C, V, st);
    default: return to_channels_last<__hip_bfloat16>(features, features_cl, N, C, V, st);
  }
}

int ops3d_roi_align3d_forward_channels_last(const void *features_cl, const void *rois, void *output, int dtype, int N,
                                            int C, int D, int H, int W, int R, int PD, int PH, int PW,
                                            float spatial_scale, int sampling_ratio, int order, void *stream) {
  if (!valid(dtype, N, C, D, H, W, R, PD, PH, PW, order)) return OPS3D_FDA_EINVAL;
  if (!ops3d_roi_align3d_channels_last_supported(dtype, C, D, H, W, PW)) return OPS3D_FDA_EINVAL;
  if ((int64_t)R * C == 0) return OPS3D_FDA_OK;
  if (!features_cl || !rois || !output || (reinterpret_cast<uintptr_t>(features_cl) & 15u)) return OPS3D_FDA_EINVAL;
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case OPS3D_FDA_F32:
      return forward_cl<float>(features_cl, rois, output, N, C, D, H, W, R, PD, PH, PW, spatial_scale, sampling_ratio,
                               order, st);
    case OPS3D_FDA_F16:
      return forward_cl<__half>(features_cl, rois, output, N, C, D, H, W, R, PD, PH, PW, spatial_scale, sampling_ratio,
                                order, st);
    default:
      return forward_cl<__hip_bfloat16>(features_cl, rois, output, N, C, D, H, W, R, PD, PH, PW, spatial_scale,
                                        sampling_ratio, order, st);
  }
}

size_t ops3d_roi_align3d_backward_workspace_bytes(int dtype, int N, int C, int D, int H, int W, int R, int PD,
                                                 int PH, int PW) {
  (void)dtype;
  if (N <= 0 || C <= 0 || D <= 0 || H <= 0 || W <= 0 || R < 0 || PD <= 0 || PH <= 0 || PW <= 0) return 0;
  if (gather_fits(C, PD, PH, PW))   // the per-roi axis tables and grad_output channels-last
    return R == 0 ? 0
                  : gather_tables_bytes(R, D, H, W, PD, PH, PW) +
                        (size_t)R * C * PD * PH * PW * (dtype == OPS3D_FDA_F32 ? 4 : 2);
  return (size_t)N * C * D * H * W * sizeof(float);
}

int ops3d_roi_align3d_backward(const void *grad_output, const void *rois, void *grad_input, void *workspace,
                               size_t workspace_bytes, int dtype, int N, int C, int D, int H, int W, int R, int PD,
                               int PH, int PW, float spatial_scale, int sampling_ratio, int order, void *stream) {
  if (!valid(dtype, N, C, D, H, W, R, PD, PH, PW, order)) return OPS3D_FDA_EINVAL;
  if ((int64_t)N * C == 0) return OPS3D_FDA_OK;
  if (!grad_input || ((int64_t)R > 0 && (!grad_output || !rois))) return OPS3D_FDA_EINVAL;
  const size_t need = ops3d_roi_align3d_backward_workspace_bytes(dtype, N, C, D, H, W, R, PD, PH, PW);
  if (need > 0 && (workspace_bytes < need || !workspace || (reinterpret_cast<uintptr_t>(workspace) & 15u)))
    return OPS3D_FDA_EINVAL;
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case OPS3D_FDA_F32:
      return backward<float>(grad_output, rois, grad_input, static_cast<float *>(workspace), N, C, D, H, W, R, PD, PH,
                             PW, spatial_scale, sampling_ratio, order, st);
    case OPS3D_FDA_F16:
      return backward<__half>(grad_output, rois, grad_input, static_cast<float *>(workspace), N, C, D, H, W, R, PD, PH,
                              PW, spatial_scale, sampling_ratio, order, st);
    default:
      return backward<__hip_bfloat16>(grad_output, rois, grad_input, static_cast<float *>(workspace), N, C, D, H, W, R,
                                      PD, PH, PW, spatial_scale, sampling_ratio, order, st);
  }
}

}  // extern "C"
