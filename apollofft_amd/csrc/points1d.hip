// points1d.hip -- 1D Kaiser-Bessel spreading (Type-1), interpolation (Type-2)
// and the coordinate gradient.
//
// Replaces the 1D loops of apollo-nufft (type1_into spread, transform/
// dimension_1d.rs:186-197; type2_into gather, :261-275).  The reference
// sorts the points by bucket first (sort_points_1d / sort_positions_1d,
// :54-99); a 1D grid (at most 4096 cells, one FFT line) fits in LDS whole,
// so here each point goes straight to its taps and nothing is sorted.
//
// A workgroup holds the whole grid: spreading as FP64 sums, which LDS adds
// atomically at 7.8 lanes a clock and CU (FP32 ones: 0.33) and which round
// nothing until the sums leave for the grid; interpolation as the FP32 grid,
// with its first cells repeated at the end so that the taps are consecutive.
// Bound by a call's launches up to some 10^4 points, then by the LDS adds
// (24 a point at w = 6) and by the polynomials.  Before, on sorted tiles of
// one wave, and now, the whole call: Type-1 of 4096 points on 512 cells 93
// and 17.5 us (a wave walked a tile's 290 points one by one), of 10^6 points
// on 2018 cells 201 and 60 (238 and 61 clustered), on 128 cells clustered
// 194 and 94 (the adds meet on few cells); Type-2 of 10^6 points on 2018
// cells 77 and 34.
#include <algorithm>

#include "point_device.h"

namespace anufft {
namespace {

// A point's tap weights (DERIV: their derivatives) and first cell.
template <int W, bool DERIV>
__device__ __forceinline__ int point_taps(const PointArgs &pa, const Geom &g, const KbPoly &P,
                                          int64_t j, float (&wt)[2 * W]) {
  int cell;
  const double t = fold_coord(pa.x[j * pa.stride], g.scale[0], g.m[0], g.inv_m[0], cell);
  const float z = (float)(1.0 - 2.0 * (t - (double)cell));
#pragma unroll
  for (int i = 0; i < 2 * W; ++i) {
    float v = DERIV ? P.dc[kPolyCoefs - 1][i] : P.c[kPolyCoefs - 1][i];
#pragma unroll
    for (int d = kPolyCoefs - 2; d >= 0; --d) v = fmaf(v, z, DERIV ? P.dc[d][i] : P.c[d][i]);
    wt[i] = v;
  }
  if (z <= -1.0f) wt[0] = 0.0f;
  if (z >= 1.0f) wt[2 * W - 1] = 0.0f;
  return wrap(cell - W + 1, g.m[0]);
}

template <int W>
__global__ __launch_bounds__(1024) void spread1d_kernel(PointArgs pa, const float2 *values,
                                                        float2 *grid, Geom g, KbPoly poly) {
  extern __shared__ double acc[];  // re, im of each cell
  const int m = g.m[0], nt = blockDim.x;
  for (int i = threadIdx.x; i < 2 * m; i += nt) acc[i] = 0.0;
  __syncthreads();
  for (int64_t j = (int64_t)blockIdx.x * nt + threadIdx.x; j < pa.num_points; j += (int64_t)gridDim.x * nt) {
    const float2 c = values[j];
    float wt[2 * W];
    int x = point_taps<W, false>(pa, g, poly, j, wt);
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) {
      unsafeAtomicAdd(&acc[2 * x], (double)c.x * (double)wt[i]);
      unsafeAtomicAdd(&acc[2 * x + 1], (double)c.y * (double)wt[i]);
      if (++x == m) x = 0;
    }
  }
  __syncthreads();
  // workgroups start at different cells, so that they do not all add to one
  // place of the grid at a time
  const int n = 2 * m, first = (int)((uint32_t)blockIdx.x * 1024u % (uint32_t)n) & ~63;
  for (int i = threadIdx.x; i < n; i += nt) {
    int k = first + i;
    if (k >= n) k -= n;
    const float v = (float)acc[k];
    if (v != 0.f) unsafeAtomicAdd((float *)grid + k, v);
  }
}

template <int W, bool DERIV>
__global__ __launch_bounds__(1024) void interp1d_kernel(PointArgs pa, const float2 *grid,
                                                        const float2 *u, float2 *out, float *gx,
                                                        Geom g, KbPoly poly) {
  extern __shared__ float2 cells[];  // m cells, then the first 2 W - 1 again
  const int m = g.m[0], nt = blockDim.x;
  for (int i = threadIdx.x; i < m + 2 * W - 1; i += nt) cells[i] = grid[i < m ? i : wrap(i, m)];
  __syncthreads();
  for (int64_t j = (int64_t)blockIdx.x * nt + threadIdx.x; j < pa.num_points; j += (int64_t)gridDim.x * nt) {
    float wt[2 * W];
    const float2 *c = cells + point_taps<W, DERIV>(pa, g, poly, j, wt);
    float sr = 0.f, si = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) {
      sr = fmaf(wt[i], c[i].x, sr);
      si = fmaf(wt[i], c[i].y, si);
    }
    if (DERIV) {
      const float2 v = u[j];
      gx[j] = -(float)g.scale[0] * (v.x * sr + v.y * si);
    } else {
      out[j] = make_float2(sr, si);
    }
  }
}

// Workgroups of the launches: 256 points each while that gives every CU at
// most one (short latency at few points), then 1024 lanes for two a CU (the
// zeroing, loading and flushing of the grid is paid by each).
struct Launch {
  int threads, blocks;
  Launch(int64_t n, int cus) {
    threads = n <= 256 * (int64_t)cus ? 256 : 1024;
    blocks = (int)std::max<int64_t>(1, std::min<int64_t>((n + threads - 1) / threads, 2 * (int64_t)cus));
  }
};

template <int W>
struct Spread1 {
  static hipError_t run(const PointArgs &pa, const float2 *values, float2 *grid, const Geom &g,
                        const KbPoly &poly, int cus, hipStream_t s) {
    const Launch l(pa.num_points, cus);
    hipLaunchKernelGGL(spread1d_kernel<W>, dim3(l.blocks), dim3(l.threads),
                       2 * sizeof(double) * g.m[0], s, pa, values, grid, g, poly);
    return hipGetLastError();
  }
};

template <int W>
struct Interp1 {
  static hipError_t run(const PointArgs &pa, const float2 *grid, const float2 *u, float2 *out,
                        float *gx, const Geom &g, const KbPoly &poly, int cus, hipStream_t s) {
    const Launch l(pa.num_points, cus);
    const size_t lds = sizeof(float2) * (g.m[0] + 2 * W - 1);
    if (gx)
      hipLaunchKernelGGL((interp1d_kernel<W, true>), dim3(l.blocks), dim3(l.threads), lds, s, pa, grid,
                         u, out, gx, g, poly);
    else
      hipLaunchKernelGGL((interp1d_kernel<W, false>), dim3(l.blocks), dim3(l.threads), lds, s, pa, grid,
                         u, out, gx, g, poly);
    return hipGetLastError();
  }
};

} // namespace

hipError_t launch_spread1d(int w, const PointArgs &pa, const float2 *values, float2 *grid,
                           const Geom &g, const KbPoly &poly, int cus, hipStream_t s) {
  return dispatch_w<Spread1>(w, pa, values, grid, g, poly, cus, s);
}
hipError_t launch_interp1d(int w, const PointArgs &pa, const float2 *grid, const float2 *u,
                           float2 *out, float *gx, const Geom &g, const KbPoly &poly, int cus,
                           hipStream_t s) {
  return dispatch_w<Interp1>(w, pa, grid, u, out, gx, g, poly, cus, s);
}

} // namespace anufft
