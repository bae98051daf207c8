// spread.hip -- Kaiser-Bessel spreading (Type-1), interpolation (Type-2) and
// the point-coordinate gradient on the vector ALUs, in 3D: subproblems of up
// to max_sub points of one tile.  The matrix-core kernels are in window.hip.
//
// Replaces the per-point T^3 loops of apollo-nufft (type1_into spread,
// transform/dimension_3d.rs:290-327; type2_into gather, :560-601).
//
// 3D spreading is output-stationary: a 1024-thread workgroup owns the padded
// tile of a subproblem, lane (py, pz) owns one (y,z) column and keeps the
// column's bin_x + 2w x-cells in registers; points are staged 256 at a time
// in LDS and each lane adds the 2w x-taps of the points whose support meets
// its column.  Nothing is accumulated through LDS atomics: on gfx950 the LDS
// FP32 atomic add measured 0.33 lane-ops/clk/CU, FP64 7.8, against ~64
// lane-FMAs/clk/CU for register FMAs.  Interpolation loads its padded tile
// into LDS once per subproblem; each wave gathers one point at a time and
// reduces across the wave.
#include "point_device.h"

namespace anufft {
namespace {

constexpr int kStage = 128;        // points staged per round (interp, grad)
constexpr int kSpreadStage = 256;  // points staged per round (spread)
constexpr int kSpreadThreads = 1024;
constexpr int kInterpThreads = 1024;

template <int W>
struct Staging {
  static constexpr int T = 2 * W;
  static constexpr int WS = (3 * T + 3) / 4 * 4; // weights per point, 16-byte rows
};

// Stage one round of points: weights, values, tap origins (3 tasks per point).
template <int W, int NT, bool DERIV>
__device__ __forceinline__ void stage_points(const PointArgs &pa, const Geom &g,
                                             const KbPoly &poly, const float2 *values,
                                             int start, int npts, int org0, int org1, int org2,
                                             float *wts, float *dwts, float2 *cv, int *loc,
                                             int *jidx) {
  constexpr int T = 2 * W;
  constexpr int WS = Staging<W>::WS;
  for (int task = threadIdx.x; task < 3 * npts; task += NT) {
    int ax = task / npts;
    int p = task - ax * npts;
    uint32_t j = pa.perm[start + p];
    const float *cp = ax == 0 ? pa.x : (ax == 1 ? pa.y : pa.z);
    int cell;
    double t = fold_coord(cp[(int64_t)j * pa.stride], g.scale[ax], g.m[ax], g.inv_m[ax], cell);
    float wt[T];
    int i0;
    if (DERIV) {
      float dwt[T];
      i0 = kb_taps_deriv<W>(t, cell, poly, wt, dwt);
#pragma unroll
      for (int i = 0; i < T; ++i) dwts[p * WS + ax * T + i] = dwt[i];
    } else {
      i0 = kb_taps<W>(t, cell, poly, wt);
    }
#pragma unroll
    for (int i = 0; i < T; ++i) wts[p * WS + ax * T + i] = wt[i];
    int org = ax == 0 ? org0 : (ax == 1 ? org1 : org2);
    loc[p * 3 + ax] = i0 - org;
    if (ax == 0) {
      if (values) cv[p] = values[j];
      if (jidx) jidx[p] = (int)j;
    }
  }
}

// Per-point record, in sorted order (floats):
//   [0, 2)          the value (re, im); zero for Type-2
//   [2, 2 + 2w)     x tap weights,  [2 + 2w, 2 + 4w) y,  [2 + 4w, 2 + 6w) z
//   2 + 6w          tile offsets of the first taps (bit pattern of an int:
//                   x register cell | y column << 8 | z column << 16)
// zero-padded to a multiple of 4.  Computing every weight once, in one fully
// parallel pass, leaves the tile kernels only coalesced copies to stage.  The
// vector-ALU spreading kernel reads the value and x weights of a record with
// wave-uniform scalar loads, so they reach its FMAs as scalar operands.
template <int W>
struct XRec {
  static constexpr int T = 2 * W;
  static constexpr int WX = 2, WY = 2 + T, WZ = 2 + 2 * T, OFF = 2 + 3 * T;
  static constexpr int RW = (OFF + 1 + 3) / 4 * 4;  // floats per record
};

// Fill the record and the x offset (cell mod bin_x) of every sorted point.
// Offsets: x register cell of the first tap = cell_x mod bin_x; y (z) tile
// column of the first tap = cell mod bin + 1 (the tile starts w cells before
// its bin).
template <int W>
__global__ __launch_bounds__(256) void point_prep_kernel(PointArgs pa, const float2 *values,
                                                          Geom g, KbPoly poly, float4 *rec,
                                                          uint8_t *xo) {
  using R = XRec<W>;
  constexpr int RW = R::RW;
  const int64_t st = (int64_t)gridDim.x * blockDim.x;
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < pa.num_points; s += st) {
    const int64_t j = (int64_t)pa.perm[s];
    float r[RW];
    int off = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float *cp = a == 0 ? pa.x : (a == 1 ? pa.y : pa.z);
      int cell;
      const double t = fold_coord(cp[j * pa.stride], g.scale[a], g.m[a], g.inv_m[a], cell);
      kb_taps<W>(t, cell, poly, r + R::WX + a * 2 * W);
      const int o = cell - (cell / g.bin[a]) * g.bin[a];
      off |= (a == 0 ? o : o + 1) << (8 * a);
      if (a == 0) xo[s] = (uint8_t)o;
    }
    if (values) {
      const float2 c = values[j];
      r[0] = c.x;
      r[1] = c.y;
    } else {
      r[0] = 0.f;
      r[1] = 0.f;
    }
    r[R::OFF] = __int_as_float(off);
#pragma unroll
    for (int i = R::OFF + 1; i < RW; ++i) r[i] = 0.f;
    float4 *d = rec + s * (RW / 4);
#pragma unroll
    for (int q = 0; q < RW / 4; ++q) d[q] = make_float4(r[4 * q], r[4 * q + 1], r[4 * q + 2], r[4 * q + 3]);
  }
}

// LDS staging of the y and z weights of one point, zero-padded to the 32
// column positions of the padded tile, so a lane reads its weight at its own
// column index.
constexpr int kSpreadRow = 2 * kSpreadCols;  // floats per staged point

// Stage points for spreading: 2 tasks per point (y and z).  Each zero-fills
// its row, stores the 2w weights at the taps' column, and writes a 4-bit
// mask of the 8-column lane blocks the point's support touches; the y task
// also copies the point's x offset.
template <int W, int NT>
__device__ __forceinline__ void stage_spread(const PointArgs &pa, const Geom &g,
                                             const float *pc, const uint8_t *xo, int start,
                                             int npts, int oy, int oz, float *rows, int *rowm,
                                             int *colm, int *xos) {
  constexpr int T = 2 * W;
  for (int task = threadIdx.x; task < 2 * npts; task += NT) {
    const int ax = task < npts ? 1 : 2;
    const int p = task - (ax - 1) * npts;
    const uint32_t j = pa.perm[start + p];
    const float *cp = ax == 1 ? pa.y : pa.z;
    int cell;
    const double t = fold_coord(cp[(int64_t)j * pa.stride], g.scale[ax], g.m[ax], g.inv_m[ax], cell);
    const int l = cell - W + 1 - (ax == 1 ? oy : oz);  // first tap's column, in [1, bin]
    float *r = rows + p * kSpreadRow + (ax - 1) * kSpreadCols;
#pragma unroll
    for (int i = 0; i < kSpreadCols; i += 4) *(float4 *)(r + i) = make_float4(0.f, 0.f, 0.f, 0.f);
    // the taps of kb_taps, stored one by one, with the polynomial
    // coefficients read from the workgroup's LDS copy pc[d][i]
    const float z = (float)(1.0 - 2.0 * (t - (double)cell));
#pragma unroll 1
    for (int i = 0; i < T; ++i) {
      float v = pc[(kPolyCoefs - 1) * kMaxTaps + i];
#pragma unroll
      for (int d = kPolyCoefs - 2; d >= 0; --d) v = fmaf(v, z, pc[d * kMaxTaps + i]);
      if (i == 0 && z <= -1.0f) v = 0.0f;
      if (i == T - 1 && z >= 1.0f) v = 0.0f;
      r[l + i] = v;
    }
    const int m = ((1 << ((l + T - 1) / 8 + 1)) - 1) & ~((1 << (l / 8)) - 1);
    if (ax == 1) {
      rowm[p] = m;
      xos[p] = xo[start + p];
    } else {
      colm[p] = m;
    }
  }
}


// One spreading subproblem (see the file comment): stage, accumulate the
// lane's column in registers, flush it to the grid.
// LDS of the spreading kernels: staged rows, masks and x offsets, then the
// polynomial coefficients (copied once per workgroup by spread_load_poly).
constexpr int kSpreadPolyOfs = kSpreadStage * (kSpreadRow + 3);  // floats

__device__ __forceinline__ void spread_load_poly(const KbPoly &poly, float *sh) {
  float *pc = sh + kSpreadPolyOfs;
  for (int i = threadIdx.x; i < kPolyCoefs * kMaxTaps; i += blockDim.x)
    pc[i] = poly.c[i / kMaxTaps][i % kMaxTaps];
}

template <int W>
__device__ __forceinline__ void spread_subproblem(const PointArgs &pa, const float *rec,
                                                  const uint8_t *xo, float2 *grid, const Geom &g,
                                                  int4 sub, float *sh) {
  constexpr int NT = kSpreadThreads;
  constexpr int T = 2 * W;
  constexpr int PX = kSpreadBinX + T - 1;  // x cells of a tile column
  constexpr int RW = XRec<W>::RW;
  float *rows = sh;
  int *rowm = (int *)(rows + kSpreadStage * kSpreadRow);
  int *colm = rowm + kSpreadStage;
  int *xos = colm + kSpreadStage;
  const float *pc = sh + kSpreadPolyOfs;

  // Wave -> 8 x 8 column block.  Waves are dealt to the 4 SIMDs round-robin;
  // the z block is rotated by the y block so each SIMD holds one block of
  // every row and column of blocks (central blocks see the most points).
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wyb = wave >> 2, wzb = (wave + wyb) & 3;
  const int py = wyb * 8 + (lane >> 3), pz = wzb * 8 + (lane & 7);
  const bool col_ok = py < g.pad[1] && pz < g.pad[2];

  const int bin = sub.x;
  const int bz = bin % g.nbin[2];
  const int by = (bin / g.nbin[2]) % g.nbin[1];
  const int bx = bin / (g.nbin[2] * g.nbin[1]);
  const int bx0 = bx * g.bin[0];
  const int oy = by * g.bin[1] - W, oz = bz * g.bin[2] - W;

  float ar[PX], ai[PX];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    ar[i] = 0.f;
    ai[i] = 0.f;
  }
  for (int c0 = 0; c0 < sub.z; c0 += kSpreadStage) {
    const int npts = min(kSpreadStage, sub.z - c0);
    __syncthreads();
    stage_spread<W, NT>(pa, g, pc, xo, sub.y + c0, npts, oy, oz, rows, rowm, colm, xos);
    __syncthreads();
    const ConstFloatPtr recs = (ConstFloatPtr)(rec + (int64_t)(sub.y + c0) * RW);
    for (int p0 = 0; p0 < npts; p0 += 64) {
      const int q = p0 + lane;
      const bool hit = q < npts && ((rowm[q] >> wyb) & (colm[q] >> wzb) & 1);
      const int o = q < npts ? xos[q] : 0;
      // one pass per x offset, so the register cells it adds to are static
#pragma unroll
      for (int oo = 0; oo < kSpreadBinX; ++oo) {
        uint64_t mask = __ballot(hit && o == oo);
        while (mask) {
          const int k = __ffsll((unsigned long long)mask) - 1;
          mask &= mask - 1;
          const int p = p0 + k;
          const float *r = rows + p * kSpreadRow;
          const float wyz = r[py] * r[kSpreadCols + pz];
          const ConstFloatPtr xr = recs + p * RW;
          const float cr = xr[0] * wyz, ci = xr[1] * wyz;
#pragma unroll
          for (int i = 0; i < T; ++i) {
            const float wx = xr[2 + i];
            ar[oo + i] = fmaf(cr, wx, ar[oo + i]);
            ai[oo + i] = fmaf(ci, wx, ai[oo + i]);
          }
        }
      }
    }
  }

  // add this lane's column to the grid: cell i <-> x = bx0 - W + 1 + i
  if (col_ok) {
    const int gy = wrap(oy + py, g.m[1]);
    const int gz = wrap(oz + pz, g.m[2]);
#pragma unroll
    for (int i = 0; i < PX; ++i) {
      if (ar[i] != 0.f || ai[i] != 0.f) {
        const int gx = wrap(bx0 - W + 1 + i, g.m[0]);
        float2 *dst = grid + ((int64_t)gx * g.m[1] + gy) * g.m[2] + gz;
        unsafeAtomicAdd(&dst->x, ar[i]);
        unsafeAtomicAdd(&dst->y, ai[i]);
      }
    }
  }
}

template <int W>
__global__ __launch_bounds__(kSpreadThreads) void spread3d_kernel(PointArgs pa, const float *rec,
                                                                  const uint8_t *xo, float2 *grid,
                                                                  Geom g, KbPoly poly) {
  extern __shared__ float sh[];
  spread_load_poly(poly, sh);  // ordered before use by the staging barrier
  const uint32_t nsub = *pa.nsub;
  for (uint32_t sidx = blockIdx.x; sidx < nsub; sidx += gridDim.x)
    spread_subproblem<W>(pa, rec, xo, grid, g, pa.subs[sidx], sh);
}

// Batched spreading: one persistent launch over the subproblems of all
// problems.  prefix[p] is the first global subproblem index of problem p
// (prefix[nprob] = total); the problem of a global index is found by a
// uniform binary search and its descriptor read with scalar loads.
template <int W>
__global__ __launch_bounds__(kSpreadThreads) void spread3d_batched_kernel(
    const SpreadProblem *probs, const uint32_t *prefix, int nprob, KbPoly poly) {
  extern __shared__ float sh[];
  spread_load_poly(poly, sh);  // ordered before use by the staging barrier
  const uint32_t total = prefix[nprob];
  for (uint32_t gidx = blockIdx.x; gidx < total; gidx += gridDim.x) {
    int lo = 0, hi = nprob - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (prefix[mid] <= gidx) lo = mid;
      else hi = mid - 1;
    }
    const SpreadProblem &pr = probs[lo];
    spread_subproblem<W>(pr.pa, pr.rec, pr.xo, pr.grid, pr.g, pr.pa.subs[gidx - prefix[lo]], sh);
  }
}

// Write descriptors passed by value into the device table.
__global__ void batch_table_kernel(BatchChunk chunk, SpreadProblem *table) {
  const int i = threadIdx.x;
  if (i < chunk.count) table[chunk.first + i] = chunk.probs[i];
}

// prefix[p] = sum of the subproblem counts of problems < p, and
// prefix[nprob + 1 + p] = sum of their work.
__global__ void batch_prefix_kernel(const SpreadProblem *probs, int nprob, uint32_t *prefix) {
  if (threadIdx.x != 0) return;
  uint32_t acc = 0, accw = 0;
  for (int p = 0; p < nprob; ++p) {
    prefix[p] = acc;
    prefix[nprob + 1 + p] = accw;
    acc += probs[p].pa.nsub[0];
    accw += probs[p].pa.nsub[1];
  }
  prefix[nprob] = acc;
  prefix[2 * nprob + 1] = accw;
}

// Load the padded tile of subproblem origin (ox,oy,oz) from the grid.
__device__ __forceinline__ void load_tile(const float2 *grid, const Geom &g, int ox, int oy,
                                          int oz, float2 *tile, int NT) {
  const int Px = g.pad[0], Py = g.pad[1], Pz = g.pad[2];
  const int P = Px * Py * Pz;
  for (int i = threadIdx.x; i < P; i += NT) {
    const int pz = i % Pz;
    const int t2 = i / Pz;
    const int py = t2 % Py;
    const int px = t2 / Py;
    const int gx = wrap(ox + px, g.m[0]);
    const int gy = wrap(oy + py, g.m[1]);
    const int gz = wrap(oz + pz, g.m[2]);
    tile[i] = grid[((int64_t)gx * g.m[1] + gy) * g.m[2] + gz];
  }
}

template <int W>
__global__ __launch_bounds__(kInterpThreads) void interp3d_kernel(PointArgs pa,
                                                                  const float2 *grid,
                                                                  float2 *out, Geom g,
                                                                  KbPoly poly) {
  constexpr int T = 2 * W;
  constexpr int WS = Staging<W>::WS;
  constexpr int NT = kInterpThreads;
  constexpr int kWaves = NT / 64;
  constexpr int kRounds = (T * T + 63) / 64;
  extern __shared__ float sh[];
  const int Py = g.pad[1], Pz = g.pad[2];
  const int P = g.pad[0] * Py * Pz;
  const int PyPz = Py * Pz;
  float2 *tile = (float2 *)sh;
  float *wts = (float *)(tile + P);
  int *loc = (int *)(wts + kStage * WS);
  int *jidx = loc + 3 * kStage;

  const uint32_t nsub = *pa.nsub;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (uint32_t sidx = blockIdx.x; sidx < nsub; sidx += gridDim.x) {
    const int4 sub = pa.subs[sidx];
    const int bin = sub.x;
    const int bz = bin % g.nbin[2];
    const int by = (bin / g.nbin[2]) % g.nbin[1];
    const int bx = bin / (g.nbin[2] * g.nbin[1]);
    const int ox = bx * g.bin[0] - W, oy = by * g.bin[1] - W, oz = bz * g.bin[2] - W;
    __syncthreads();
    load_tile(grid, g, ox, oy, oz, tile, NT);
    for (int c0 = 0; c0 < sub.z; c0 += kStage) {
      const int npts = min(kStage, sub.z - c0);
      __syncthreads();
      stage_points<W, NT, false>(pa, g, poly, nullptr, sub.y + c0, npts, ox, oy, oz, wts,
                                 nullptr, nullptr, loc, jidx);
      __syncthreads();
      for (int p = wave; p < npts; p += kWaves) {
        const float *wp = wts + p * WS;
        const int lx = loc[3 * p], ly = loc[3 * p + 1], lz = loc[3 * p + 2];
        float ar = 0.f, ai = 0.f;
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
          const int q = lane + 64 * r;
          if (q < T * T) {
            const int ty = q / T, tz = q - (q / T) * T;
            const float wyz = wp[T + ty] * wp[2 * T + tz];
            const float2 *tp = tile + (lx * Py + ly + ty) * Pz + lz + tz;
            float sr = 0.f, si = 0.f;
#pragma unroll
            for (int tx = 0; tx < T; ++tx) {
              const float2 v = tp[tx * PyPz];
              sr = fmaf(wp[tx], v.x, sr);
              si = fmaf(wp[tx], v.y, si);
            }
            ar = fmaf(wyz, sr, ar);
            ai = fmaf(wyz, si, ai);
          }
        }
        ar = wave_sum(ar);
        ai = wave_sum(ai);
        if (lane == 0) out[jidx[p]] = make_float2(ar, ai);
      }
    }
  }
}

// d/dx of the interpolant, contracted with conj(u_j):
// grad[a][j] = Re(conj(u_j) * (-scale_a) * sum dphi_a phi_b phi_c G).
template <int W>
__global__ __launch_bounds__(kInterpThreads) void grad3d_kernel(PointArgs pa,
                                                                const float2 *grid,
                                                                const float2 *u, float *gx,
                                                                float *gy, float *gz, Geom g,
                                                                KbPoly poly) {
  constexpr int T = 2 * W;
  constexpr int WS = Staging<W>::WS;
  constexpr int NT = kInterpThreads;
  constexpr int kWaves = NT / 64;
  constexpr int kRounds = (T * T + 63) / 64;
  extern __shared__ float sh[];
  const int Py = g.pad[1], Pz = g.pad[2];
  const int P = g.pad[0] * Py * Pz;
  const int PyPz = Py * Pz;
  float2 *tile = (float2 *)sh;
  float *wts = (float *)(tile + P);
  float *dwts = wts + kStage * WS;
  int *loc = (int *)(dwts + kStage * WS);
  int *jidx = loc + 3 * kStage;

  const uint32_t nsub = *pa.nsub;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (uint32_t sidx = blockIdx.x; sidx < nsub; sidx += gridDim.x) {
    const int4 sub = pa.subs[sidx];
    const int bin = sub.x;
    const int bz = bin % g.nbin[2];
    const int by = (bin / g.nbin[2]) % g.nbin[1];
    const int bx = bin / (g.nbin[2] * g.nbin[1]);
    const int ox = bx * g.bin[0] - W, oy = by * g.bin[1] - W, oz = bz * g.bin[2] - W;
    __syncthreads();
    load_tile(grid, g, ox, oy, oz, tile, NT);
    for (int c0 = 0; c0 < sub.z; c0 += kStage) {
      const int npts = min(kStage, sub.z - c0);
      __syncthreads();
      stage_points<W, NT, true>(pa, g, poly, nullptr, sub.y + c0, npts, ox, oy, oz, wts, dwts,
                                nullptr, loc, jidx);
      __syncthreads();
      for (int p = wave; p < npts; p += kWaves) {
        const float *wp = wts + p * WS;
        const float *dp = dwts + p * WS;
        const int lx = loc[3 * p], ly = loc[3 * p + 1], lz = loc[3 * p + 2];
        float sx[2] = {0.f, 0.f}, sy[2] = {0.f, 0.f}, sz[2] = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
          const int q = lane + 64 * r;
          if (q < T * T) {
            const int ty = q / T, tz = q - (q / T) * T;
            const float2 *tp = tile + (lx * Py + ly + ty) * Pz + lz + tz;
            float ar = 0.f, ai = 0.f, dr = 0.f, di = 0.f;
#pragma unroll
            for (int tx = 0; tx < T; ++tx) {
              const float2 v = tp[tx * PyPz];
              ar = fmaf(wp[tx], v.x, ar);
              ai = fmaf(wp[tx], v.y, ai);
              dr = fmaf(dp[tx], v.x, dr);
              di = fmaf(dp[tx], v.y, di);
            }
            const float wy = wp[T + ty], wz = wp[2 * T + tz];
            const float dy = dp[T + ty], dz = dp[2 * T + tz];
            const float wyz = wy * wz, dyz = dy * wz, wydz = wy * dz;
            sx[0] = fmaf(wyz, dr, sx[0]);
            sx[1] = fmaf(wyz, di, sx[1]);
            sy[0] = fmaf(dyz, ar, sy[0]);
            sy[1] = fmaf(dyz, ai, sy[1]);
            sz[0] = fmaf(wydz, ar, sz[0]);
            sz[1] = fmaf(wydz, ai, sz[1]);
          }
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          sx[c] = wave_sum(sx[c]);
          sy[c] = wave_sum(sy[c]);
          sz[c] = wave_sum(sz[c]);
        }
        if (lane == 0) {
          const int j = jidx[p];
          const float2 uj = u[j];
          // Re(conj(u) * (-s) * S) = -s (u.x S.x + u.y S.y)
          gx[j] = -(float)g.scale[0] * (uj.x * sx[0] + uj.y * sx[1]);
          if (gy) gy[j] = -(float)g.scale[1] * (uj.x * sy[0] + uj.y * sy[1]);
          if (gz) gz[j] = -(float)g.scale[2] * (uj.x * sz[0] + uj.y * sz[1]);
        }
      }
    }
  }
}

template <int W>
size_t spread_lds(const Geom &) {
  return ((size_t)kSpreadPolyOfs + kPolyCoefs * kMaxTaps) * sizeof(float);
}

template <int W>
size_t interp_lds(const Geom &g, bool grad) {
  const size_t P = (size_t)g.pad[0] * g.pad[1] * g.pad[2];
  const size_t ws = (size_t)kStage * Staging<W>::WS * (grad ? 2 : 1);
  return P * sizeof(float2) + ws * sizeof(float) + 4 * kStage * sizeof(int);
}

template <int W>
struct PointPrep {
  static hipError_t run(const PointArgs &pa, const float2 *values, const Geom &g,
                        const KbPoly &poly, float *rec, uint8_t *xo, hipStream_t s) {
    if (pa.num_points <= 0) return hipSuccess;
    int64_t blocks = (pa.num_points + 255) / 256;
    if (blocks > 16384) blocks = 16384;
    hipLaunchKernelGGL(point_prep_kernel<W>, dim3((unsigned)blocks), dim3(256), 0, s, pa, values,
                       g, poly, (float4 *)rec, xo);
    return hipGetLastError();
  }
};

template <int W>
struct Spread3 {
  static hipError_t run(const PointArgs &pa, const float *rec, const uint8_t *xo, float2 *grid,
                        const Geom &g, const KbPoly &poly, int nblk, hipStream_t s) {
    size_t lds = spread_lds<W>(g);
    hipError_t e = hipFuncSetAttribute((const void *)spread3d_kernel<W>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(spread3d_kernel<W>, dim3(nblk), dim3(kSpreadThreads), lds, s, pa, rec, xo,
                       grid, g, poly);
    return hipGetLastError();
  }
};

template <int W>
struct Spread3Batched {
  static hipError_t run(const SpreadProblem *probs, const uint32_t *prefix, int nprob,
                        const KbPoly &poly, int nblk, hipStream_t s) {
    const Geom g{};
    size_t lds = spread_lds<W>(g);
    hipError_t e = hipFuncSetAttribute((const void *)spread3d_batched_kernel<W>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(spread3d_batched_kernel<W>, dim3(nblk), dim3(kSpreadThreads), lds, s,
                       probs, prefix, nprob, poly);
    return hipGetLastError();
  }
};

template <int W>
struct Interp3 {
  static hipError_t run(const PointArgs &pa, const float2 *grid, float2 *out, const Geom &g,
                        const KbPoly &poly, int nblk, hipStream_t s) {
    size_t lds = interp_lds<W>(g, false);
    hipError_t e = hipFuncSetAttribute((const void *)interp3d_kernel<W>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(interp3d_kernel<W>, dim3(nblk), dim3(kInterpThreads), lds, s, pa, grid,
                       out, g, poly);
    return hipGetLastError();
  }
};

template <int W>
struct Grad3 {
  static hipError_t run(const PointArgs &pa, const float2 *grid, const float2 *u, float *gx,
                        float *gy, float *gz, const Geom &g, const KbPoly &poly, int nblk,
                        hipStream_t s) {
    size_t lds = interp_lds<W>(g, true);
    hipError_t e = hipFuncSetAttribute((const void *)grad3d_kernel<W>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(grad3d_kernel<W>, dim3(nblk), dim3(kInterpThreads), lds, s, pa, grid, u,
                       gx, gy, gz, g, poly);
    return hipGetLastError();
  }
};

template <int W>
struct LdsSize {
  static hipError_t run(const Geom &g, int kind, size_t *out) {
    *out = kind == 0 ? spread_lds<W>(g) : interp_lds<W>(g, kind == 2);
    return hipSuccess;
  }
};

} // namespace

int point_rec_floats(int w) { return (2 + 6 * w + 1 + 3) / 4 * 4; }


hipError_t launch_point_prep(int w, const PointArgs &pa, const float2 *values, const Geom &g,
                             const KbPoly &poly, float *rec, uint8_t *xo, hipStream_t s) {
  return dispatch_w<PointPrep>(w, pa, values, g, poly, rec, xo, s);
}

int spread_bin_x(int w, int method) {
  return method == kSpreadMfma ? win_bin_x(w) : kSpreadBinX;
}

hipError_t launch_spread3d(int w, const PointArgs &pa, const float *rec, const uint8_t *xo,
                           float2 *grid, const Geom &g, const KbPoly &poly, int nblk,
                           hipStream_t s) {
  return dispatch_w<Spread3>(w, pa, rec, xo, grid, g, poly, nblk, s);
}
hipError_t launch_spread3d_batched(int w, const SpreadProblem *host_probs, int nprob,
                                   SpreadProblem *dev_table, uint32_t *dev_prefix,
                                   const KbPoly &poly, int nblk, hipStream_t s) {
  for (int first = 0; first < nprob; first += kBatchChunk) {
    BatchChunk chunk{};
    chunk.first = first;
    chunk.count = nprob - first < kBatchChunk ? nprob - first : kBatchChunk;
    for (int i = 0; i < chunk.count; ++i) chunk.probs[i] = host_probs[first + i];
    hipLaunchKernelGGL(batch_table_kernel, dim3(1), dim3(64), 0, s, chunk, dev_table);
  }
  hipLaunchKernelGGL(batch_prefix_kernel, dim3(1), dim3(64), 0, s, dev_table, nprob, dev_prefix);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return dispatch_w<Spread3Batched>(w, (const SpreadProblem *)dev_table, (const uint32_t *)dev_prefix,
                                    nprob, poly, nblk, s);
}
hipError_t launch_interp3d(int w, const PointArgs &pa, const float2 *grid, float2 *out,
                           const Geom &g, const KbPoly &poly, int nblk, hipStream_t s) {
  return dispatch_w<Interp3>(w, pa, grid, out, g, poly, nblk, s);
}
hipError_t launch_grad3d(int w, const PointArgs &pa, const float2 *grid, const float2 *u, float *gx,
                         float *gy, float *gz, const Geom &g, const KbPoly &poly, int nblk,
                         hipStream_t s) {
  return dispatch_w<Grad3>(w, pa, grid, u, gx, gy, gz, g, poly, nblk, s);
}
size_t spread_lds_bytes(int w, int method, const Geom &g) {
  size_t v = 0;  // the matrix-core kernels' LDS is static
  if (method != kSpreadMfma) (void)dispatch_w<LdsSize>(w, g, 0, &v);
  return v;
}
size_t interp_lds_bytes(int w, const Geom &g, bool grad) {
  size_t v = 0;
  (void)dispatch_w<LdsSize>(w, g, grad ? 2 : 1, &v);
  return v;
}

} // namespace anufft
