// block_spread.hip -- Type-1 spreading on blocks of 32 x 32 cells, for the
// entry points that return FP64 results (host FP64 storage).
//
// Replaces the per-point T^3 loop of apollo-nufft (type1_into spread,
// transform/dimension_3d.rs:290-327).
//
// A dense grid cell sums hundreds to thousands of FP32 terms, and the
// rounding of such a sum depends on the order of its terms: runs of this kernel
// differ by 2e-7 (the order of the atomic additions), and the windows of
// window.hip, the spreading of the other entry points, are 4e-7 from it.  It is
// kept for one reason: callers who hold results in FP64 compare them more closely
// than FP32 ones, and with it they stay as they have been to within what two runs
// differ by.  Neither accuracy nor speed is the reason: against 64-bit sums
// the windows are off by less (32^3 modes, w = 6, 100,000 points 3.48e-7 here and
// 3.08e-7; 24^3, 400,000 clustered 2.65e-7 and 2.02e-7; 16^3, w = 7, 400,000
// 1.13e-6 and 7.2e-7), and a call with them takes 220 us instead of 247.
//
// The order: tiles of PX x cells x 32 y x 32 z along x pencils, the points of a
// tile in input order, 16 a step.
//
// For each x cell the (y, z) plane is one output block of
// v_mfma_f32_32x32x16_f16: A[y][k] = wx_k wy_k(y) times B[k][z] = c_k wz_k(z).
#include "point_device.h"

namespace anufft {
namespace {

// Tap polynomials staged in LDS as rows of kPolyRow floats per tap (the
// kPolyCoefs coefficients, lowest degree first, zero padded), so that a lane
// evaluates all taps of a point with broadcast reads of uniform addresses.
constexpr int kPolyRow = 12;
__device__ __forceinline__ void stage_poly_rows(const float (*__restrict__ coef)[kMaxTaps], int T,
                                                float *rows) {
  for (int k = threadIdx.x; k < T * kPolyRow; k += blockDim.x) {
    const int tap = k / kPolyRow, d = k - tap * kPolyRow;
    rows[k] = d < kPolyCoefs ? coef[d][tap] : 0.f;
  }
}

// Weights of all 2W taps at two arguments z0, z1 from the mirrored
// polynomials (tap 2W-1-i at z is tap i at -z): each pair from the even part
// E(z^2) and odd part O(z^2) of tap i, P_i = E + z O, P_{2W-1-i} = E - z O;
// kb_taps's endpoint rule.
static_assert(kPolyCoefs == 11, "taps2_sym splits degree-10 polynomials into even and odd parts");
template <int W>
__device__ __forceinline__ void taps2_sym(const float *__restrict__ rows, float z0, float z1,
                                          float (&v0)[2 * W], float (&v1)[2 * W]) {
  const float u0 = z0 * z0, u1 = z1 * z1;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    float c[kPolyRow];
#pragma unroll
    for (int d = 0; d < kPolyRow; d += 4) *(float4 *)(c + d) = *(const float4 *)(rows + i * kPolyRow + d);
    float e0 = c[10], e1 = c[10], o0 = c[9], o1 = c[9];
#pragma unroll
    for (int d = 8; d >= 0; d -= 2) {
      e0 = fmaf(e0, u0, c[d]);
      e1 = fmaf(e1, u1, c[d]);
    }
#pragma unroll
    for (int d = 7; d >= 1; d -= 2) {
      o0 = fmaf(o0, u0, c[d]);
      o1 = fmaf(o1, u1, c[d]);
    }
    v0[i] = fmaf(z0, o0, e0);
    v1[i] = fmaf(z1, o1, e1);
    v0[2 * W - 1 - i] = fmaf(-z0, o0, e0);
    v1[2 * W - 1 - i] = fmaf(-z1, o1, e1);
  }
  if (z0 <= -1.0f) v0[0] = 0.f;
  if (z1 <= -1.0f) v1[0] = 0.f;
  if (z0 >= 1.0f) v0[2 * W - 1] = 0.f;
  if (z1 >= 1.0f) v1[2 * W - 1] = 0.f;
}

// Each FP32 operand is split into FP16 hi + lo (split8) and a product is
// hi hi + hi lo + lo hi, accumulated in FP32.  The strengths of a subproblem
// are scaled by a power of two so that max |c| is in [1/2, 1); the flush
// undoes the scale exactly.  A wave owns XW = 4 consecutive x cells (4 x 2
// accumulator blocks); the B operands of a point group are shared by the
// wave's cells, A is rebuilt per cell from the staged y and x weights.
template <int W>
struct BSpread {
  static constexpr int NW = W >= 8 ? 8 : 4;    // waves per workgroup
  static constexpr int XW = 4;                 // x cells per wave
  static constexpr int PX = NW * XW;           // x cells of a tile
  static constexpr int BINX = PX - 2 * W + 1;  // tile interior along x
  static constexpr int NT = 64 * NW;
};
constexpr int kMNP = 128;       // points staged per round
constexpr int kMWY = kMNP + 4;  // row stride (floats) of the y / x weight tables
constexpr int kMBT = kMNP + 8;  // row stride (halves) of the B operand tables
// LDS layout (bytes), for a tile of PX x cells.
constexpr int kMWZ = 33;        // row stride (floats) of the staged z weights
template <int PX>
struct BLds {
  static constexpr int WY = 0;                                 // float [32][kMWY]
  static constexpr int WX = WY + 32 * kMWY * 4;                // float [PX][kMWY]
  static constexpr int BT = WX + PX * kMWY * 4;                // half [4][32][kMBT]
  static constexpr int C = BT + 4 * 32 * kMBT * 2;             // float2 [kMNP]
  static constexpr int WZ = C + kMNP * 8;                      // float [kMNP][kMWZ]
  static constexpr int ZS = WZ + kMNP * kMWZ * 4;              // float [3][kMNP]
  static constexpr int OFS = ZS + 3 * kMNP * 4;                // int [kMNP]
  static constexpr int RED = OFS + kMNP * 4;                   // float [8]
  static constexpr int POLY = RED + 8 * 4;                     // float [kMaxTaps][kPolyRow]
  static constexpr int SIZE = POLY + kMaxTaps * kPolyRow * 4;
};
// two 4-wave workgroups per CU for w <= 7
static_assert(2 * BLds<16>::SIZE <= 160 * 1024, "block spreading LDS");

// Tile of a spreading subproblem.  The accumulators of a workgroup form a
// ring of PX x columns: column x lives in slot x mod PX, so a workgroup that
// moves on to the next tile along x keeps the columns both tiles cover and
// flushes only those it leaves behind.
struct BTile {
  int pencil;       // y-z tile row (by * nbin_z + bz)
  int bx;           // x tile index
  int xlo, oy, oz;  // grid cell of tile column 0, row 0, layer 0
};

template <int W>
__device__ __forceinline__ BTile block_tile(const Geom &g, int bin) {
  const int bz = bin % g.nbin[2];
  const int by = (bin / g.nbin[2]) % g.nbin[1];
  const int bx = bin / (g.nbin[2] * g.nbin[1]);
  return BTile{by * g.nbin[2] + bz, bx, bx * g.bin[0] - W + 1, by * g.bin[1] - W,
               bz * g.bin[2] - W};
}

// Power-of-two scale of a subproblem's strengths: e with max |c| 2^-e in
// [1/2, 1), clamped to [-120, 120] so that both scales stay finite and normal.
template <int NW>
__device__ __forceinline__ int block_strength_exp(const ZRec &zr, int4 sub, float *red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int NT = 64 * NW, B = 4;  // B values per thread loaded before any is used
  const float2 *vals = zr.v + sub.y;
  float mx = 0.f;
  for (int p0 = threadIdx.x; p0 < sub.z; p0 += NT * B) {
    float2 c[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int p = p0 + u * NT;
      c[u] = vals[p < sub.z ? p : 0];
    }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (p0 + u * NT < sub.z) mx = fmaxf(mx, fmaxf(fabsf(c[u].x), fabsf(c[u].y)));
  }
  mx = wave_max_nonneg(mx);
  __syncthreads();  // earlier readers of red[] are done
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) mx = fmaxf(mx, red[i]);
  int e = 0;
  if (mx > 0.f) (void)frexpf(mx, &e);
  return max(-120, min(120, e));
}

// Add the points of one subproblem, strengths scaled by s_in, to the ring
// accumulators; base = tile column 0's ring slot.
template <int W>
__device__ __forceinline__ void block_accumulate(f32x16 (&acc)[BSpread<W>::XW][2], const ZRec &zr,
                                                const WinPoly *__restrict__ dpoly, int4 sub,
                                                int base, float s_in, char *sh) {
  using MS = BSpread<W>;
  constexpr int NT = MS::NT, XW = MS::XW, PX = MS::PX, T = 2 * W;
  using L = BLds<PX>;
  float *WY = (float *)(sh + L::WY);
  float *WX = (float *)(sh + L::WX);
  _Float16 *BT = (_Float16 *)(sh + L::BT);
  float2 *C = (float2 *)(sh + L::C);
  float *WZ = (float *)(sh + L::WZ);
  float *ZS = (float *)(sh + L::ZS);
  int *OFS = (int *)(sh + L::OFS);

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = lane >> 5, l32 = lane & 31;

  for (int c0 = 0; c0 < sub.z; c0 += kMNP) {
    const int npts = min(kMNP, sub.z - c0);
    const int ng = (npts + 15) >> 4;
    const int np16 = ng << 4;
    const int start = sub.y + c0;
    __syncthreads();  // the previous round's operand reads are done
    // pass 0: zero the operand tables; the points' polynomial arguments,
    // tile offsets and scaled values into LDS (padding points: z = 0,
    // offsets 0, value 0, so their finite weights meet zero B rows)
    for (int p = threadIdx.x; p < np16; p += NT) {
#pragma unroll
      for (int i = 0; i < PX; ++i) WX[i * kMWY + p] = 0.f;
#pragma unroll
      for (int y = 0; y < 32; ++y) WY[y * kMWY + p] = 0.f;
#pragma unroll
      for (int zz = 0; zz < 32; ++zz) WZ[p * kMWZ + zz] = 0.f;
      const bool ok = p < npts;
      const float4 z = ok ? zr.r[start + p] : make_float4(0.f, 0.f, 0.f, 0.f);
      const float2 c = ok ? zr.v[start + p] : make_float2(0.f, 0.f);
      ZS[p] = z.x;
      ZS[kMNP + p] = z.y;
      ZS[2 * kMNP + p] = z.z;
      OFS[p] = __float_as_int(z.w);
      C[p] = make_float2(c.x * s_in * kOpScale, c.y * s_in * kOpScale);
    }
    __syncthreads();
    // pass 1: tap weights; a task evaluates all taps of one axis for two
    // points (p, p + np16 / 2).  The x weights go to ring slot (tile column
    // + base) mod PX.
    {
      const float *PL = (const float *)(sh + L::POLY);
      const int hn = np16 >> 1;
      for (int u = threadIdx.x; u < 3 * hn; u += NT) {
        const int a = (u >= hn) + (u >= 2 * hn);
        const int p0 = u - a * hn, p1 = p0 + hn;
        const int o0 = (OFS[p0] >> (8 * a)) & 255, o1 = (OFS[p1] >> (8 * a)) & 255;
        float v0[T], v1[T];
        taps2_sym<W>(PL, ZS[a * kMNP + p0], ZS[a * kMNP + p1], v0, v1);
        if (a == 0) {
#pragma unroll
          for (int i = 0; i < T; ++i) {
            WX[((o0 + i + base) & (PX - 1)) * kMWY + p0] = v0[i] * kOpScale;
            WX[((o1 + i + base) & (PX - 1)) * kMWY + p1] = v1[i] * kOpScale;
          }
        } else if (a == 1) {
#pragma unroll
          for (int i = 0; i < T; ++i) {
            WY[(o0 + i) * kMWY + p0] = v0[i];
            WY[(o1 + i) * kMWY + p1] = v1[i];
          }
        } else {
#pragma unroll
          for (int i = 0; i < T; ++i) {
            WZ[p0 * kMWZ + o0 + i] = v0[i];
            WZ[p1 * kMWZ + o1 + i] = v1[i];
          }
        }
      }
    }
    __syncthreads();
    // pass 2: B operands c_k wz_k(z), split, 8 points per task
    for (int t = threadIdx.x; t < 32 * (np16 >> 3); t += NT) {
      const int z = t & 31, pb = (t >> 5) << 3;
      float br[8], bi[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float w = WZ[(pb + j) * kMWZ + z];
        const float2 c = C[pb + j];
        br[j] = c.x * w;
        bi[j] = c.y * w;
      }
      half8 rh, rl, ih, il;
      split8(br, rh, rl);
      split8(bi, ih, il);
      *(half8 *)(BT + (0 * 32 + z) * kMBT + pb) = rh;
      *(half8 *)(BT + (1 * 32 + z) * kMBT + pb) = rl;
      *(half8 *)(BT + (2 * 32 + z) * kMBT + pb) = ih;
      *(half8 *)(BT + (3 * 32 + z) * kMBT + pb) = il;
    }
    __syncthreads();
    // MFMA: 16 points per step; lane (l32, h) holds A row y = l32 and
    // B column z = l32 for the points kb .. kb + 7; wave w owns ring
    // slots w XW .. w XW + XW - 1
    for (int gi = 0; gi < ng; ++gi) {
      const int kb = (gi << 4) + (h << 3);
      const half8 brh = *(const half8 *)(BT + (0 * 32 + l32) * kMBT + kb);
      const half8 brl = *(const half8 *)(BT + (1 * 32 + l32) * kMBT + kb);
      const half8 bih = *(const half8 *)(BT + (2 * 32 + l32) * kMBT + kb);
      const half8 bil = *(const half8 *)(BT + (3 * 32 + l32) * kMBT + kb);
      float wy[8];
      *(float4 *)wy = *(const float4 *)(WY + l32 * kMWY + kb);
      *(float4 *)(wy + 4) = *(const float4 *)(WY + l32 * kMWY + kb + 4);
      half8 ah[XW], al[XW];
#pragma unroll
      for (int q = 0; q < XW; ++q) {
        const int ix = wave * XW + q;
        float a[8];
        *(float4 *)a = *(const float4 *)(WX + ix * kMWY + kb);
        *(float4 *)(a + 4) = *(const float4 *)(WX + ix * kMWY + kb + 4);
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] *= wy[j];
        split8(a, ah[q], al[q]);
      }
      // one split term at a time over all 2 XW accumulators: 2 XW
      // independent MFMA chains
#pragma unroll
      for (int q = 0; q < XW; ++q) {
        acc[q][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[q], brh, acc[q][0], 0, 0, 0);
        acc[q][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[q], bih, acc[q][1], 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < XW; ++q) {
        acc[q][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[q], brl, acc[q][0], 0, 0, 0);
        acc[q][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[q], bil, acc[q][1], 0, 0, 0);
      }
#pragma unroll
      for (int q = 0; q < XW; ++q) {
        acc[q][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[q], brh, acc[q][0], 0, 0, 0);
        acc[q][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[q], bih, acc[q][1], 0, 0, 0);
      }
    }
  }
}

// Add the ring columns x in [t.xlo, t.xlo + ncol) to the grid (scaled by
// s_out) and zero them.  Accumulator r of lane (l32, h) is tile cell (y, z)
// with y = 8 (r / 4) + 4 h + r % 4, z = l32.
template <int W>
__device__ __forceinline__ void block_flush(f32x16 (&acc)[BSpread<W>::XW][2], float2 *grid,
                                           const Geom &g, const BTile &t, int ncol, float s_out) {
  using MS = BSpread<W>;
  constexpr int XW = MS::XW, PX = MS::PX;
  int lane = threadIdx.x & 63;
  // an opaque copy: keeps the per-row index arithmetic below from being
  // hoisted out of the subproblem loop, where it would stay live in
  // registers for the whole kernel
  asm volatile("" : "+v"(lane));
  const int wave = threadIdx.x >> 6;
  const int h = lane >> 5, l32 = lane & 31;
  int m0 = __builtin_amdgcn_readfirstlane(g.m[0]);
  int m1 = __builtin_amdgcn_readfirstlane(g.m[1]);
  int m2 = __builtin_amdgcn_readfirstlane(g.m[2]);
  asm volatile("" : "+s"(m0), "+s"(m1), "+s"(m2));  // no hoisted divisions by m
  const int base = t.xlo & (PX - 1);
  const bool zok = l32 < g.pad[2];
  const int gz = wrap(t.oz + l32, m2);
#pragma unroll
  for (int q = 0; q < XW; ++q) {
    const int ix = (wave * XW + q - base) & (PX - 1);  // tile column of the slot
    if (ix >= ncol) continue;
    if (zok) {
      const int gx = wrap(t.xlo + ix, m0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int y = ((r >> 2) << 3) + (h << 2) + (r & 3);
        const float vr = acc[q][0][r] * s_out, vi = acc[q][1][r] * s_out;
        if (y < g.pad[1] && (vr != 0.f || vi != 0.f)) {
          const int gy = wrap(t.oy + y, m1);
          float2 *dst = grid + ((int64_t)gx * m1 + gy) * m2 + gz;
          unsafeAtomicAdd(&dst->x, vr);
          unsafeAtomicAdd(&dst->y, vi);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[q][0][r] = 0.f;
      acc[q][1][r] = 0.f;
    }
  }
}

// Longest run of points accumulated in registers between full flushes.
constexpr int kMaxChain = 8192;

// Ring window of one workgroup: the open tile and its scale.
struct BWindow {
  bool open = false;
  BTile t{};
  int e = 0;
};

// Columns of the open window to flush before the window moves to tile n at
// strength exponent e (PX = all): a tile further along the
// same pencil keeps the columns both cover, unless the scales are so far
// apart that rescaling the kept sums could leave the normal FP32 range.
template <int W>
__device__ __forceinline__ int block_flush_cols(const BWindow &w, const BTile &n, int e, const Geom &g) {
  constexpr int PX = BSpread<W>::PX;
  if (w.t.pencil != n.pencil || n.bx < w.t.bx || abs(e - w.e) > 32) return PX;
  return min(PX, (n.bx - w.t.bx) * g.bin[0]);
}

template <int W>
__device__ __forceinline__ void block_rescale(f32x16 (&acc)[BSpread<W>::XW][2], float f) {
#pragma unroll
  for (int q = 0; q < BSpread<W>::XW; ++q) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[q][0][r] *= f;
      acc[q][1][r] *= f;
    }
  }
}

// Spread a workgroup's share of the list with one ring window: a tile further along the pencil keeps the columns both cover;
// everything left is flushed at the end.
template <int W>
__device__ __forceinline__ void block_run(const int4 *__restrict__ subs, const XcdChunk &r,
                                                const ZRec &zr, float2 *grid, const Geom &g,
                                                const WinPoly *__restrict__ dpoly, char *shm) {
  using MS = BSpread<W>;
  float *red = (float *)(shm + BLds<MS::PX>::RED);
  f32x16 acc[MS::XW][2];
#pragma unroll
  for (int q = 0; q < MS::XW; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[q][0][r] = acc[q][1][r] = 0.f;
  BWindow win;
  int chain = 0;  // points accumulated since the last full flush
  for (uint32_t sidx = r.begin; sidx < r.end; ++sidx) {
    const int4 sub = r.part(sidx, subs[sidx]);
    const BTile t = block_tile<W>(g, sub.x);
    const int e = block_strength_exp<MS::NW>(zr, sub, red);
    if (win.open) {
      int ncol = block_flush_cols<W>(win, t, e, g);
      // bound the FP32 accumulation chains (rounding error grows with their
      // length) as a full flush per subproblem of kMaxChain points would
      if (chain + sub.z > kMaxChain) ncol = MS::PX;
      block_flush<W>(acc, grid, g, win.t, ncol, ldexpf(1.0f, win.e) * kProdUnscale);
      if (ncol < MS::PX && e != win.e) block_rescale<W>(acc, ldexpf(1.0f, win.e - e));
      if (ncol == MS::PX) chain = 0;
    }
    chain += sub.z;
    win.open = true;
    win.t = t;
    win.e = e;
    block_accumulate<W>(acc, zr, dpoly, sub, t.xlo & (MS::PX - 1), ldexpf(1.0f, -e), shm);
  }
  if (win.open)
    block_flush<W>(acc, grid, g, win.t, MS::PX, ldexpf(1.0f, win.e) * kProdUnscale);
}

template <int W>
__global__ __launch_bounds__(BSpread<W>::NT, 2) void block_spread_kernel(
    PointArgs pa, ZRec zr, float2 *grid, Geom g, const WinPoly *__restrict__ dpoly) {
  using MS = BSpread<W>;
  extern __shared__ __align__(16) char shm[];
  stage_poly_rows(dpoly->p.c, 2 * W, (float *)(shm + BLds<MS::PX>::POLY));  // ordered by the first barrier
  const XcdChunk r(pa);
  block_run<W>(pa.subs, r, zr, grid, g, dpoly, shm);
}

template <int W>
struct BlockSpread {
  static hipError_t run(const PointArgs &pa, ZRec zr, float2 *grid, const Geom &g,
                        const WinPoly *dpoly, int nblk, hipStream_t s) {
    constexpr int lds = BLds<BSpread<W>::PX>::SIZE;
    hipError_t e = hipFuncSetAttribute((const void *)block_spread_kernel<W>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(block_spread_kernel<W>, dim3(nblk), dim3(BSpread<W>::NT), lds, s, pa, zr, grid,
                       g, dpoly);
    return hipGetLastError();
  }
};
template <int W>
struct BlockShape {
  static hipError_t run(int *binx) {
    *binx = BSpread<W>::BINX;
    return hipSuccess;
  }
};

} // namespace

int block_bin_x(int w) {
  int v = 1;
  (void)dispatch_w<BlockShape>(w, &v);
  return v;
}
hipError_t launch_block_spread(int w, const PointArgs &pa, ZRec zr, float2 *grid, const Geom &g,
                               const WinPoly *dpoly, int num_blocks, hipStream_t s) {
  return dispatch_w<BlockSpread>(w, pa, zr, grid, g, dpoly, num_blocks, s);
}

} // namespace anufft
