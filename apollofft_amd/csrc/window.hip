// window.hip -- the 3D matrix-core point kernels: Kaiser-Bessel spreading
// (Type-1), interpolation (Type-2) and the coordinate gradient on 16-row
// windows of the grid.
//
// Replaces the per-point T^3 loops of apollo-nufft (type1_into spread,
// transform/dimension_3d.rs:290-327; type2_into gather, :560-601) and the
// O(grid x points) WGSL passes fast_type1_spread_3d /
// fast_type2_interpolate_3d (apollo-nufft-wgpu .../shaders/
// nufft_fast_3d.wgsl:130-161, :268-299).
//
// A window is PX x cells x 16 y rows x 32 z cells: the points of one tile
// whose y offsets lie in one class of at most 17 - 2w consecutive offsets
// (class_sort_kernel) have all their taps inside it.  For each x cell the
// products run on v_mfma_f32_16x16x32_f16:
//   spreading       G_i[y][z] += sum_k (wx_k(i) wy_k(y)) (c_k wz_k(z)), K = 32 points,
//                   four blocks of 16 y rows x 8 complex z cells;
//   interpolation   D_i[y][k] = sum_z G_i[y][z] wz_k(z), K = the 32 z cells,
//                   16 points, contracted over y and x on the vector ALUs.
// Each FP32 operand is split into FP16 hi + lo (hi = fp16(a), lo =
// fp16(a - hi)) and a product is hi hi + hi lo + lo hi with FP32
// accumulation: about 22 significant bits.
//
// The entries of one (x, z) pencil of tiles follow each other along y, so a
// workgroup's window slides: rows are kept as a ring (row y at y mod 16), and
// a step flushes (spreading) or loads (interpolation) only the rows the
// window leaves or gains, 17 - 2w of 16.  The window is PX x cells wide,
// 17 - 2w of them and more interior: unlike y and z, x cells cost matrix work
// one by one, so PX is chosen for the flush against the products (below).
//
// Against blocks of 32 x 32 cells with two planes of 16 points a step
// (block_spread.hip), a window executes 6144 f16 flops per point and x cell
// its group reaches instead of 12288, over 14 to 16 cells instead of 16 to
// 32.  What bounds the kernels is the matrix work and the vector work beside
// it, which overlap little on a SIMD, then the flush of spreading (17 G
// 64-byte atomic requests a second) and the loading of interpolation's
// windows.  Measured, blocks or the class lists that each
// interpolation workgroup built for itself, and now: spreading 2e6 points,
// 64^3 modes, w = 7, 400 and 250 us; 16e6 points, 127^3 modes, w = 4, 2650
// and 1250; interpolation 2e6, w = 7, 400 and 280; 16e6, 100^3, w = 8, 5310
// and 2440; gradient 1e6, 64^3, w = 6, 447 and 258.
//
// Points are staged kWinPts at a time; each wave evaluates the taps of one
// axis for them (a lane is a point), with the polynomial coefficients in
// scalar registers, and clears the tables it writes itself, so a round needs
// two barriers.
#include <algorithm>

#include "point_device.h"

namespace anufft {
namespace {

// x cells per wave: of the windows, and of the wide spreading windows for
// few points a cell (anufft_plan::spread_bins).
constexpr int win_cells(int w) { return w >= 7 ? 5 : (w >= 5 ? 4 : 3); }
constexpr int wide_cells(int w) { return w >= 5 ? 7 : 6; }

template <int W, int XC = win_cells(W)>
struct Win {
  static constexpr int T = 2 * W;
  static constexpr int CW = 17 - T;  // y offsets of a class at most
  static constexpr int NW = 4;       // waves
  static constexpr int NT = 64 * NW;
  static constexpr int XW = XC;      // x cells per wave
  static constexpr int PX = NW * XW;
  static constexpr int BINX = PX - T + 1;
  static_assert(BINX >= 1 && CW >= 1, "window shape");
};

constexpr int kWinPts = 64;  // points staged per round, one per lane

// All 2W taps at argument z from the mirrored polynomials (tap 2W-1-i at z is
// tap i at -z, negated for the derivative, ODD): each pair from the even part
// E(z^2) and odd part O(z^2) of tap i, P_i = E + z O, P_{2W-1-i} = E - z O
// (ODD: z O - E), with the coefficients c[d * kMaxTaps + tap] in scalar
// registers; the endpoint rule of kb_taps.
static_assert(kPolyCoefs == 11, "degree-10 polynomials split into even and odd parts");
template <int W, bool ODD = false>
__device__ __forceinline__ void taps_scalar(ConstFloatPtr c, float z, float (&v)[2 * W]) {
  // In two parts, each loading its coefficients where they are used: hoisted
  // out of the loops, or all at once, they would push the loops' scalars out
  // to vector lanes.
  constexpr int H = W > 4 ? (W + 1) / 2 : W;
  const float u = z * z;
#pragma unroll
  for (int i0 = 0; i0 < W; i0 += H) {
    if (i0 == 0) asm volatile("" : "+s"(c));
    else asm volatile("" : "+s"(c), "+v"(v[0]), "+v"(v[H - 1]));
#pragma unroll
    for (int i = i0; i < W && i < i0 + H; ++i) {
      float e = c[10 * kMaxTaps + i], o = c[9 * kMaxTaps + i];
#pragma unroll
      for (int d = 8; d >= 0; d -= 2) e = fmaf(e, u, c[d * kMaxTaps + i]);
#pragma unroll
      for (int d = 7; d >= 1; d -= 2) o = fmaf(o, u, c[d * kMaxTaps + i]);
      v[i] = fmaf(z, o, e);
      v[2 * W - 1 - i] = ODD ? fmaf(z, o, -e) : fmaf(-z, o, e);
    }
  }
  if (z <= -1.0f) v[0] = 0.f;
  if (z >= 1.0f) v[2 * W - 1] = 0.f;
}

// hi = fp16(a), lo = fp16(a - hi) of two values (split8's rounding).
__device__ __forceinline__ void split2(float a, float b, half2v &hi, half2v &lo) {
  const float2v x = {a, b};
  hi = __builtin_convertvector(x, half2v);
  typedef __fp16 fp16x2 __attribute__((ext_vector_type(2)));
  const fp16x2 l = __builtin_amdgcn_cvt_pkrtz(a - (float)hi[0], b - (float)hi[1]);
  lo[0] = (_Float16)l[0];
  lo[1] = (_Float16)l[1];
}

// Window of one class of a tile.
struct WTile {
  int xlo, y0, z0;  // grid cell of column 0, row 0, layer 0
  int o1;           // tile y offset of row 0's first tap
};

template <int W>
__device__ __forceinline__ WTile win_tile(const Geom &g, int bin, int cls, int cw) {
  const int bz = bin % g.nbin[2], t = bin / g.nbin[2];
  const int by = t % g.nbin[1], bx = t / g.nbin[1];
  WTile w;
  w.o1 = 1 + cls * cw;
  w.xlo = bx * g.bin[0] - W + 1;
  w.y0 = by * g.bin[1] - W + w.o1;
  w.z0 = bz * g.bin[2] - W;
  return w;
}

// A walk over the classes of a workgroup's share of the subproblem list:
// entries [lo, hi) of the class list hold the points of class `cls` of tile
// `bin` that are the workgroup's.
struct ClassWalk {
  const XcdChunk &r;
  ConstInt4Ptr subs;
  const uint16_t *start;
  int ncls;
  uint32_t i;
  int bin, cls, lo, hi;
  int y, p0, p1;  // the subproblem's first entry; its entries that are this workgroup's
  uint32_t st;    // lane k: first entry of class k (lane ncls: the count)
  __device__ __forceinline__ ClassWalk(const XcdChunk &r_, const PointArgs &pa)
      : r(r_), subs((ConstInt4Ptr)pa.subs), start(pa.cstart), ncls(pa.ncls), i(r_.begin) {
    load();
  }
  __device__ __forceinline__ void load() {
    const int4v e = subs[i];
    const int4 s = make_int4(e.x, e.y, e.z, e.w), q = r.part(i, s);
    bin = s.x;
    y = s.y;
    p0 = q.y - s.y;
    p1 = p0 + q.z;
    const int lane = threadIdx.x & 63;
    st = lane < ncls ? (uint32_t)start[(int64_t)i * ncls + lane] : (uint32_t)s.z;
    cls = -1;
    next_class();
  }
  __device__ __forceinline__ void next_class() {
    do {  // some class has points in [p0, p1)
      ++cls;
      lo = max((int)__builtin_amdgcn_readlane(st, cls), p0);
      hi = min((int)__builtin_amdgcn_readlane(st, cls + 1), p1);
    } while (lo >= hi && cls + 1 < ncls);
    lo += y;
    hi += y;
  }
  // To the next class with points; false at the end of the share.
  __device__ __forceinline__ bool next() {
    if (hi - y < p1) {
      next_class();
      return true;
    }
    if (i + 1 >= r.end) return false;
    ++i;
    load();
    return true;
  }
};

// The rounds of kWinPts points ahead of the one being worked on: the list
// entries of the points two rounds ahead and the records of the next round
// are loaded while a round runs.
struct Rounds {
  ClassWalk w;
  uint32_t off;  // (lists end at 2^31 - 1 points, and the rounds go on past the share's end)
  __device__ __forceinline__ Rounds(const XcdChunk &r, const PointArgs &pa) : w(r, pa), off((uint32_t)w.lo) {}
  // List position of point p of the round (a valid one past the end too).
  __device__ __forceinline__ int pos(int p) const { return (int)min(off + (uint32_t)p, (uint32_t)w.hi - 1u); }
  __device__ __forceinline__ void advance() {
    off += kWinPts;
    if (off >= (uint32_t)w.hi && w.next()) off = (uint32_t)w.lo;
  }
};

// The x cells of a group: a wave's cells q (window column 4 q + wave) that the
// group's points reach, c0 <= 4 q < c1.  body(q0, q1) runs once with compile-
// time bounds that cover them: all cells, or all but the first, the last or
// both (a kernel spans most of the window, so more is rarely left out), each
// a straight line the scheduler can pipeline.
template <int N>
struct IntConst {
  __device__ constexpr operator int() const { return N; }
};
template <int XW, class F>
__device__ __forceinline__ void reached_cells(int c0, int c1, F body) {
  const bool first = c0 <= 0, last = c1 > 4 * (XW - 1);  // whether they are reached
  if (first) {
    if (last) body(IntConst<0>(), IntConst<XW>());
    else body(IntConst<0>(), IntConst<XW - 1>());
  } else {
    if (last) body(IntConst<1>(), IntConst<XW>());
    else body(IntConst<1>(), IntConst<XW - 1>());
  }
}

// ---- spreading ---------------------------------------------------------------
constexpr int kSLd = kWinPts + 8;   // row stride (halves) of the B operand table
constexpr int kSLdF = kWinPts + 4;  // row stride (floats) of the weight tables
template <int PX>
struct SLds {
  static constexpr int X = 0;                             // float [PX][kSLdF]: x weights
  static constexpr int Y = X + PX * kSLdF * 4;            // float [16][kSLdF]: y weights
  static constexpr int B = Y + 16 * kSLdF * 4;            // half [hi, lo][32 z][re, im][kSLd]
  static constexpr int R = B + 2 * 64 * kSLd * 2;         // int [groups]: x cells reached
  static constexpr int SIZE = R + 16;
};
template <int W, int XC>
using SpreadAcc = f32x4[XC][4];  // [slot][block of 8 z cells]

// Ring rows and z cells of the accumulators.  Register r of lane (i16, g4)
// of a block is ring row 4 r + g4, so that the (few, consecutive) rows of a
// flush lie in few registers, each used by all four lane groups; its column
// is z cell 8 b + i16 / 2 of 32, re or im by i16 & 1.  The z cells sit at z
// mod 32: blocks of 8 cells start at multiples of 64 bytes of a grid row
// (whose length is a multiple of 8 cells in most grids), and re and im lie
// side by side as in the grid, so the 16 lanes of a row are one aligned
// 64-byte atomic request.  Such requests bound the flush: 17 G/s measured
// whatever they hold (61 M floats: 222 us in aligned 64-byte requests, 370
// misaligned, 442 in 32-byte ones).
//
// Add rows [0, nrow) of the window t to the grid (times 2^e_out) and zero
// them.
template <int W, int XC>
__device__ __forceinline__ void win_flush(SpreadAcc<W, XC> &acc, float2 *grid, const Geom &g,
                                          const WTile &t, int wave, int i16, int g4, int nrow,
                                          int e_out) {
  using WN = Win<W, XC>;
  int m0 = __builtin_amdgcn_readfirstlane(g.m[0]), m1 = __builtin_amdgcn_readfirstlane(g.m[1]);
  int m2 = __builtin_amdgcn_readfirstlane(g.m[2]);
  asm volatile("" : "+v"(i16), "+v"(g4), "+s"(m0), "+s"(m1), "+s"(m2));
  uint32_t z[4];  // byte offsets in a grid row
#pragma unroll
  for (int b = 0; b < 4; ++b)
    z[b] = 8 * wrap(t.z0 + ((8 * b + (i16 >> 1) - t.z0) & 31), m2) + 4 * (i16 & 1);
  uint64_t plane[WN::XW];  // byte addresses, wave-uniform
#pragma unroll
  for (int q = 0; q < WN::XW; ++q)
    plane[q] = (uint64_t)grid + (uint64_t)wrap(t.xlo + 4 * q + wave, m0) * ((uint64_t)m1 * m2 * 8);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = (4 * r + g4 - t.y0) & 15;
    if (row < nrow) {
      const uint32_t y = (uint32_t)(wrap(t.y0 + row, m1) * m2) * 8;
#pragma unroll
      for (int q = 0; q < WN::XW; ++q)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float v = ldexpf(acc[q][b][r], e_out);
          if (v != 0.f) unsafeAtomicAdd((float *)(plane[q] + (y + z[b])), v);
          acc[q][b][r] = 0.f;
        }
    }
  }
}

// Longest run of points accumulated in registers between full flushes
// (bounds the FP32 rounding of a cell's sum).
constexpr int kMaxChain = 8192;

// Clear N rows (N a multiple of 4) of the weight tables by one wave.
template <int N>
__device__ __forceinline__ void clear_rows(float *f, int lane) {
  static_assert(N % 4 == 0 && kWinPts == 64, "four rows a store of the wave");
#pragma unroll
  for (int i = 0; i < N / 4; ++i)
    *(float4 *)(f + (4 * i + (lane >> 4)) * kSLdF + (lane & 15) * 4) = make_float4(0.f, 0.f, 0.f, 0.f);
}

// hi and lo of s v[i] to z cell i of the B table (re or im rows).
template <int T>
__device__ __forceinline__ void store_split(_Float16 *f, const float (&v)[T], float s) {
#pragma unroll
  for (int i = 0; i < T; i += 2) {
    half2v h, l;
    split2(v[i] * s, v[i + 1] * s, h, l);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      f[(i + d) * 2 * kSLd] = h[d];
      f[(32 + i + d) * 2 * kSLd] = l[d];
    }
  }
}

// The x cells the points of a group reach, first | last + 1 << 16: the list
// is ordered by x offset within a class, so the group's first and last point
// have the extreme ones.  (off: the lanes' offset words.)
template <int T>
__device__ __forceinline__ int cells_reached(int off, int first, int last) {
  return (__builtin_amdgcn_readlane(off, first) & 255) |
         ((__builtin_amdgcn_readlane(off, last) & 255) + T) << 16;
}

// Weights of the staged points, window relative: role 0 x and 1 y, a lane a
// point; 2 and 3 the B operands of the first and second 32 points, lanes 0-31
// re and 32-63 im (staged_point).  Lanes past the round's points leave their
// column of the tables zero.
template <int W, int XC>
__device__ __forceinline__ void spread_stage(char *sh, int role, int lane, int npts, float4 ra,
                                             float2 cv, const WinPoly *poly, const WTile &w) {
  using WN = Win<W, XC>;
  constexpr int T = WN::T, PX = WN::PX;
  using L = SLds<PX>;
  const int off = __float_as_int(ra.w);
  if (role == 0) {
    const int r0 = cells_reached<T>(off, 0, min(npts, 32) - 1);
    const int r1 = cells_reached<T>(off, 32, max(npts, 33) - 1);
    if (lane < 2) ((int *)(sh + L::R))[lane] = lane == 0 ? r0 : r1;
  }
  // opaque copies here and in the flush: keep their address arithmetic from
  // being hoisted out of the loops, where it would hold registers throughout
  asm volatile("" : "+v"(lane));
  const bool ok = lane < npts;
  float v[T];
  if (role < 2) {  // (the x weights carry the product's scale)
    float *F = (float *)(sh + (role == 0 ? L::X : L::Y));
    if (role == 0) clear_rows<PX>(F, lane);
    else clear_rows<16>(F, lane);
    taps_scalar<W>((ConstFloatPtr)(role == 0 ? &poly->op[0][0] : &poly->p.c[0][0]), role == 0 ? ra.x : ra.y, v);
    F += (role == 0 ? off & 255 : ((off >> 8) & 255) - w.o1) * kSLdF + lane;
    if (ok)
#pragma unroll
      for (int i = 0; i < T; ++i) F[i * kSLdF] = v[i];
  } else if (32 * (role - 2) < npts) {
    _Float16 *B = (_Float16 *)(sh + L::B) + 32 * (role - 2);
#pragma unroll
    for (int i = 0; i < 2 * 64 / 16; ++i)
      *(float4 *)(B + (16 * i + (lane >> 2)) * kSLd + (lane & 3) * 8) = make_float4(0.f, 0.f, 0.f, 0.f);
    taps_scalar<W>((ConstFloatPtr)&poly->p.c[0][0], ra.z, v);
    if (32 * (role - 2) + (lane & 31) < npts)
      store_split<T>(B + (((off >> 16) & 255) * 2 + (lane >> 5)) * kSLd + (lane & 31), v,
                     lane < 32 ? cv.x : cv.y);
  }
}

// The point of a round a lane stages in a role.
__device__ __forceinline__ int staged_point(int role, int lane) {
  return role < 2 ? lane : 32 * (role - 2) + (lane & 31);
}

// The products of the staged points, 32 a step: lane (i16, g4) holds A row
// i16 (the ring row whose sums its lane group keeps, win_flush) and B column
// i16 for the points 8 g4 .. 8 g4 + 7.  x cells the 32 points do not reach
// are left out.
template <int W, int XC>
__device__ __forceinline__ void spread_products(SpreadAcc<W, XC> &acc, const char *sh, int ng,
                                                const WTile &t, int wave, int i16, int g4) {
  using WN = Win<W, XC>;
  using L = SLds<WN::PX>;
  constexpr int XW = WN::XW;
  asm volatile("" : "+v"(i16), "+v"(g4));
  const float *X = (const float *)(sh + L::X) + wave * kSLdF;
  // ring row 4 (i16 % 4) + i16 / 4 and z cell 8 b + i16 / 2, window relative
  const float *Y = (const float *)(sh + L::Y) + ((4 * (i16 & 3) + (i16 >> 2) - t.y0) & 15) * kSLdF;
  const _Float16 *B[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
    B[b] = (const _Float16 *)(sh + L::B) + (((8 * b + (i16 >> 1) - t.z0) & 31) * 2 + (i16 & 1)) * kSLd;
  for (int gi = 0; gi < ng; ++gi) {
    const int kb = 32 * gi + 8 * g4;
    const int cells = __builtin_amdgcn_readfirstlane(((const int *)(sh + L::R))[gi]);
    const int c0 = (cells & 0xffff) - wave, c1 = (cells >> 16) - wave;  // reached: c0 <= 4 q < c1
    half8 bh[4], bl[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      bh[b] = *(const half8 *)(B[b] + kb);
      bl[b] = *(const half8 *)(B[b] + 64 * kSLd + kb);
    }
    float y[8];
    *(float4 *)y = *(const float4 *)(Y + kb);
    *(float4 *)(y + 4) = *(const float4 *)(Y + kb + 4);
#pragma unroll
    for (int q = 0; q < XW; ++q) {
      if (4 * q < c0 || 4 * q >= c1) continue;
      // A = wx wy, the FP32 product split once.  (Split factors multiplied
      // with FP16 FMAs take 16 vector instructions a cell instead of 24, but
      // lose bits: against 64 bits 2000 points on 32^3 cells 2.8e-7 and 2.6e-7;
      // and their staging takes what the products save: a Type-1 call of 2e6
      // points, w = 7, 353 us and 354, w = 4, 244 and 244.)
      float a[8];
      *(float4 *)a = *(const float4 *)(X + 4 * q * kSLdF + kb);
      *(float4 *)(a + 4) = *(const float4 *)(X + 4 * q * kSLdF + kb + 4);
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] *= y[j];
      half8 ah, al;
      split8(a, ah, al);
      // four independent chains of three products
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[q][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bh[b], acc[q][b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[q][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl[b], acc[q][b], 0, 0, 0);
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[q][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh[b], acc[q][b], 0, 0, 0);
    }
  }
}

// Power-of-two exponent of a maximum kept in slots: e with max 2^-e in
// [1/2, 1), 128 for an infinite one.  Strengths and sums are scaled by ldexpf:
// over the range of finite floats 2^(bits - e) and its inverse need not be
// finite (strengths of 1e-36).
__device__ __forceinline__ int max_exp(const float *slots, int lane) {
  static_assert(kMaxSlots == 64, "a slot a lane");
  const float mx = wave_max(slots[lane * kMaxStride]);
  int e = 0;
  if (mx > 0.f) (void)frexpf(mx, &e);
  return __builtin_amdgcn_readfirstlane(mx < INFINITY ? e : 128);
}

// Spread the share r of one problem's list.
template <int W, int XC>
__device__ __forceinline__ void spread_run(const PointArgs &pa, const ZRec &zr, float2 *grid,
                                           const Geom &g, const XcdChunk &r, const WinPoly *poly,
                                           char *sh) {
  using WN = Win<W, XC>;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g4 = lane >> 4;
  if (r.begin >= r.end) return;
  SpreadAcc<W, XC> acc;
#pragma unroll
  for (int q = 0; q < WN::XW; ++q)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[q][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int e = max_exp((const float *)pa.vmax, lane);
  const int e_in = kValBits - e, e_out = e - kProdBits;

  const uint32_t *perm = pa.cperm;
  Rounds ahead(r, pa);
  float4 ra;
  float2 cv = make_float2(0.f, 0.f);
  // the staging roles move round the waves (SIMDs) from round to round
  int role = wave;
  uint32_t np = perm[ahead.pos(staged_point(role, lane))];
  ra = zr.r[np];
  if (role >= 2) cv = zr.v[np];
  ahead.advance();
  np = perm[ahead.pos(staged_point((role + 1) & 3, lane))];
  ClassWalk cw(r, pa);
  WTile t = win_tile<W>(g, cw.bin, cw.cls, pa.cw);
  int chain = 0;  // points accumulated since the last full flush
  for (;;) {
    const int n = cw.hi - cw.lo;
    chain += n;
    for (int c0 = 0; c0 < n; c0 += kWinPts) {
      const int npts = min(kWinPts, n - c0);
      spread_stage<W, XC>(sh, role, lane, npts, ra, make_float2(ldexpf(cv.x, e_in), ldexpf(cv.y, e_in)), poly, t);
      __syncthreads();
      role = (role + 1) & 3;
      ra = zr.r[np];
      if (role >= 2) cv = zr.v[np];
      ahead.advance();
      np = perm[ahead.pos(staged_point((role + 1) & 3, lane))];
      spread_products<W, XC>(acc, sh, (npts + 31) >> 5, t, wave, i16, g4);
      __syncthreads();
    }
    if (!cw.next()) break;
    const WTile w = win_tile<W>(g, cw.bin, cw.cls, pa.cw);
    // the loads in flight are waited for before the atomics are issued (a
    // wait after them would wait for them too)
    asm volatile("" : "+v"(ra.x), "+v"(ra.w), "+v"(cv.x), "+v"(np));
    const bool slide = w.xlo == t.xlo && w.z0 == t.z0 && w.y0 >= t.y0 && chain + cw.hi - cw.lo <= kMaxChain;
    const int nrow = slide ? min(16, w.y0 - t.y0) : 16;
    if (nrow > 0) win_flush<W, XC>(acc, grid, g, t, wave, i16, g4, nrow, e_out);
    if (nrow == 16) chain = 0;
    t = w;
  }
  win_flush<W, XC>(acc, grid, g, t, wave, i16, g4, 16, e_out);
}

// Workgroups resident on a CU: as many as the registers (16 XW a lane for the
// accumulators) hold, or all but: 3, with 3 x cells 4, at which 6 registers
// spill (batched 17; w = 7 and 8 batched 6 at 3).  Type-1 calls, 4 against 3: 2e6
// points on 128^3 cells w = 2 202 and 205 us, w = 3 229 and 234, w = 4 243 and
// 252; 16 problems w = 4 1433 and 1482; 800,000 points, where the flush counts
// for more, w = 4 171 and 169.  (w = 6 at 4: spreading 226 to 306 us, the spills
// queue behind the atomics.)
constexpr int spread_groups_per_cu(int cells) { return cells <= 3 ? 4 : cells <= 5 ? 3 : 2; }

template <int W, int XC>
__global__ __launch_bounds__(Win<W>::NT, spread_groups_per_cu(XC)) void win_spread_kernel(
    PointArgs pa, ZRec zr, float2 *grid, Geom g, const WinPoly *__restrict__ dpoly) {
  __shared__ __align__(16) char sh[SLds<Win<W, XC>::PX>::SIZE];
  const XcdChunk r(pa);
  spread_run<W, XC>(pa, zr, grid, g, r, dpoly, sh);
}

// A descriptor read through the scalar cache (its fields stay in scalar
// registers, as kernel arguments do).
template <class T>
__device__ __forceinline__ T load_scalar(const T *p) {
  typedef const int __attribute__((address_space(4))) *ConstIntPtr;
  static_assert(sizeof(T) % 4 == 0, "whole dwords");
  const ConstIntPtr s = (ConstIntPtr)p;
  struct {
    int d[sizeof(T) / 4];
  } v;
#pragma unroll
  for (unsigned i = 0; i < sizeof(T) / 4; ++i) v.d[i] = s[i];
  return __builtin_bit_cast(T, v);
}

// Batched form: one persistent launch over the lists of all problems
// (wpre[p] = work of the problems before p, wpre[nprob] = total).
template <int W, int XC>
__global__ __launch_bounds__(Win<W>::NT, spread_groups_per_cu(XC)) void win_spread_batched_kernel(
    const SpreadProblem *probs, const uint32_t *wpre, int nprob, const WinPoly *__restrict__ dpoly) {
  __shared__ __align__(16) char sh[SLds<Win<W, XC>::PX>::SIZE];
  uint32_t w0, w1;
  xcd_work_range(wpre[nprob], w0, w1);
  if (w0 >= w1) return;
  int p = 0;
  {  // last problem with wpre <= w0
    int hi = nprob - 1;
    while (p < hi) {
      const int mid = (p + hi + 1) >> 1;
      if (wpre[mid] <= w0) p = mid;
      else hi = mid - 1;
    }
  }
  // each problem the range meets: its share of the problem's own list
  for (; p < nprob && wpre[p] < w1; ++p) {
    const uint32_t lo = wpre[p], hi = wpre[p + 1];
    if (hi <= w0) continue;  // no work of this problem in the range
    const SpreadProblem pr = load_scalar(probs + p);
    const XcdChunk part(pr.pa.subs, pr.pa.nsub[0], hi - lo, max(w0, lo) - lo, min(w1, hi) - lo);
    spread_run<W, XC>(pr.pa, pr.zr, pr.grid, pr.g, part, dpoly, sh);
  }
}

// ---- interpolation and coordinate gradient -------------------------------------
//
// The window of the grid lives in registers as FP16 hi + lo A operands: lane
// (i16, g4) of a wave holds ring row i16 (row y at y mod 16), z cells 8 g4 ..
// 8 g4 + 7 of the window's 32, for each of the wave's x cells.  It is scaled
// by the power of two of the grid's largest component, which leaves 22 bits to
// cells down to 2^-15 of it and an absolute 2^-37 of it below, far under the
// rounding of the FFT that wrote the grid; so rows carry over while the window
// slides along a pencil of tiles.  Only rows the window gains are loaded (the
// lanes of the others sit the loads out).  (Scales of each tile's own maximum
// took LDS atomics in the last FFT pass and a launch of their own: Type-2 of
// 2e6 points, w = 7, 394 us and now 371, 200,000 ragged ones, w = 4, 113 and
// 95.)
constexpr int kIRow = 40;   // row stride (halves) of a staged point's z weights (32 cells)
constexpr int kIRowY = 20;  // row stride (floats) of its y weights (16 ring rows; 32: + 16)
template <int W>
struct ILds {
  using WN = Win<W>;
  static constexpr int ROWX = WN::PX <= 12 ? 12 : 20;  // row stride (floats) of the x weights
};
// Window origin along z: even, so that aligned rows load 16 bytes at a time
// (z offsets start at 1: no tap of the tile lies in a skipped first cell).
__device__ __forceinline__ int even_z0(int z0) { return z0 + (z0 & 1); }

// The exponent windows are scaled with, whose 2^(kValBits - e) is finite: the
// loads multiply by it (ldexpf there took 1 % of a Type-2 call, 2e6 points on
// 128^3 cells 334.6 and 338.1 us).  Grids below 2^-111 are scaled by 2^126 and
// so split to 2^-150, finer than FP32 subnormals lie.
__device__ __forceinline__ int grid_exp(const float *gmax, int lane) {
  return max(max_exp(gmax, lane), kValBits - 126);
}

// H windows of 16 rows on top of each other: H = 2, tall windows, hold every
// point of a tile (bin_y + 2 W <= 32 rows) for twice the products a point; row
// y at y mod 16 H.
constexpr int kWinBuf = 256;  // 16 rows of 16 pairs
template <int W, int H>
struct GridWin {
  static constexpr int XW = Win<W>::XW;
  half8 rh[H][XW], rl[H][XW], ih[H][XW], il[H][XW];

  // Load rows `first` .. 16 H - 1 of window t (scaled by s); the other rows
  // keep their content.  buf: kWinBuf float4 of LDS, the wave's own.
  //
  // A lane needs 64 bytes of its row (z cells 8 g4 .. 8 g4 + 7), but 64 lanes
  // each reading 16 bytes 64 apart are 64 accesses of the first-level cache,
  // one a clock: they bound calls of few points a window (1.3 M loads of 29
  // accesses, 150k of 230k clocks, at 17,000 points on 128^3).  So 16 lanes
  // load a row's 32 cells (4 rows a load, only rows that are new), and the
  // wave turns them in LDS (XORed places: no bank conflicts).  Lanes as the
  // products need them, and so: interpolation of 17,000 points 95 and 57 us,
  // 1e6 on 128^3, w = 6, 155 and 129, 2e6, w = 7, 310 and 287; gradient 1e6
  // 267 and 258.  AHEAD: the next cell's loads run during this one's turn,
  // where registers are left for them (w = 5, 6 at 4 workgroups: 25 spilled).
  template <bool AHEAD>
  __device__ __forceinline__ void load(const float2 *grid, const Geom &g, const WTile &t, int first,
                                       float s, int wave, int i16, int g4, float4 *buf) {
#pragma unroll
    for (int h = 0; h < H; ++h) load_half<AHEAD>(h, grid, g, t, first, s, wave, i16, g4, buf);
  }
  template <bool AHEAD>
  __device__ __forceinline__ void load_half(int h, const float2 *grid, const Geom &g, const WTile &t,
                                            int first, float s, int wave, int i16, int g4,
                                            float4 *buf) {
    int m0 = __builtin_amdgcn_readfirstlane(g.m[0]), m1 = __builtin_amdgcn_readfirstlane(g.m[1]);
    int m2 = __builtin_amdgcn_readfirstlane(g.m[2]);
    asm volatile("" : "+v"(i16), "+v"(g4), "+s"(m0), "+s"(m1), "+s"(m2));
    // as a loader: cells z, z + 1 of ring rows 16 h + 4 r + g4
    const int z = wrap(even_z0(t.z0) + 2 * i16, m2);
    const bool pairs = (m2 & 1) == 0;  // aligned, and none crosses the end
    const int next = z + 1 < m2 ? 8 : 8 - 8 * m2;  // bytes from z to z + 1
    int at[4];  // byte offset in a plane (below 2^27), -1: not loaded
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (16 * h + 4 * r + g4 - t.y0) & (16 * H - 1);
      at[r] = row < first ? -1 : 8 * (wrap(t.y0 + row, m1) * m2 + z);
    }
    const bool mine = ((16 * h + i16 - t.y0) & (16 * H - 1)) >= first;
    auto fetch = [&](int q, float4 (&u)[4]) {
      const char *plane = (const char *)(grid + (int64_t)wrap(t.xlo + 4 * q + wave, m0) * m1 * m2);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (at[r] < 0) continue;
        if (pairs) {
          u[r] = *(const float4 *)(plane + (uint32_t)at[r]);
        } else {
          const float2 a = *(const float2 *)(plane + (uint32_t)at[r]);
          const float2 b = *(const float2 *)(plane + (uint32_t)(at[r] + next));
          u[r] = make_float4(a.x, a.y, b.x, b.y);
        }
      }
    };
    float4 u[4], un[4];
    if (AHEAD) fetch(0, un);
#pragma unroll
    for (int q = 0; q < XW; ++q) {
      if (AHEAD) {
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] = un[r];
        if (q + 1 < XW) fetch(q + 1, un);
      } else {
        fetch(q, u);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      int i = i16, k = g4;
      if (!AHEAD) asm volatile("" : "+v"(i), "+v"(k));  // places not kept: no registers left
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + k;
        if (at[r] >= 0) buf[16 * row + (i ^ row)] = u[r];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (!mine) continue;
      float2 v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 c = buf[16 * i + ((4 * k + j) ^ i)];
        v[2 * j] = make_float2(c.x, c.y);
        v[2 * j + 1] = make_float2(c.z, c.w);
      }
      float tr[8], ti[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        tr[j] = v[j].x * s;
        ti[j] = v[j].y * s;
      }
      split8(tr, rh[h][q], rl[h][q]);
      split8(ti, ih[h][q], il[h][q]);
    }
  }
};

// Sums over the four lane groups of a wave: a's in lanes 0-31, b's in 32-63.
__device__ __forceinline__ float sum_groups(float a, float b) {
  typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
  // lower halves of a and b, upper halves of a and b
  const uint2v h = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  const float s = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const uint2v r = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The x cells reached by each group of 16 of the staged points (cells_reached).
template <int W>
__device__ __forceinline__ void stage_reach(int *reach, int off, int npts, int lane) {
  int r[kWinPts / 16];
#pragma unroll
  for (int i = 0; i < kWinPts / 16; ++i)
    r[i] = cells_reached<2 * W>(off, 16 * i, max(min(npts, 16 * i + 16), 16 * i + 1) - 1);
  if (lane == 0) *(int4 *)reach = make_int4(r[0], r[1], r[2], r[3]);
}

// One axis' taps of a staged point into its float row (x: window columns; y:
// ring rows), cleared first.
template <int W, bool ODD>
__device__ __forceinline__ void interp_stage_x(float *row, bool ok, float z, int o, const float *poly) {
#pragma unroll
  for (int i = 0; i < Win<W>::PX; i += 4) *(float4 *)(row + i) = make_float4(0.f, 0.f, 0.f, 0.f);
  float v[2 * W];
  taps_scalar<W, ODD>((ConstFloatPtr)poly, z, v);
  if (ok) {
    row += o;
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) row[i] = v[i];
  }
}
template <int W, int H, bool ODD>
__device__ __forceinline__ void interp_stage_y(float *row, bool ok, float z, int first, const float *poly) {
#pragma unroll
  for (int i = 0; i < 16 * H; i += 4) *(float4 *)(row + i) = make_float4(0.f, 0.f, 0.f, 0.f);
  float v[2 * W];
  taps_scalar<W, ODD>((ConstFloatPtr)poly, z, v);
  if (ok) {
    const int r0 = first & (16 * H - 1), cut = 16 * H - r0;  // taps from `cut` on wrap around
    float *a = row + r0, *b = a - 16 * H;
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) (i < cut ? a : b)[i] = v[i];
  }
}
// z taps (scaled) as FP16 hi and lo B rows.
template <int W, bool ODD>
__device__ __forceinline__ void interp_stage_z(_Float16 *rh, _Float16 *rl, bool ok, float z, int o,
                                               const float *poly) {
#pragma unroll
  for (int i = 0; i < 32; i += 8) {
    *(float4 *)(rh + i) = make_float4(0.f, 0.f, 0.f, 0.f);
    *(float4 *)(rl + i) = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float v[2 * W];
  taps_scalar<W, ODD>((ConstFloatPtr)poly, z, v);
  if (ok) {
    rh += o;
    rl += o;
#pragma unroll
    for (int i = 0; i < 2 * W; i += 2) {
      half2v h, l;
      split2(v[i], v[i + 1], h, l);
      rh[i] = h[0];
      rh[i + 1] = h[1];
      rl[i] = l[0];
      rl[i + 1] = l[1];
    }
  }
}

// As many workgroups on a CU as the registers hold: 4 up to w = 6 (2e6 points
// on 64^3, w = 6: 252 to 230 us), 3 above (w = 7 at 4: 296 to 372, spilled).
// Tall windows need twice the operand registers.
constexpr int interp_groups_per_cu(int cells, int h) { return (cells <= 4 ? 4 : 3) - (h - 1); }

template <int W, int H>
__global__ __launch_bounds__(Win<W>::NT, interp_groups_per_cu(win_cells(W), H)) void win_interp_kernel(
    PointArgs pa, ZRec zr, const float2 *grid, const float *gmax, float2 *out, Geom g,
    const WinPoly *__restrict__ dpoly) {
  using WN = Win<W>;
  using L = ILds<W>;
  constexpr int XW = WN::XW, ROWY = kIRowY + 16 * (H - 1);
  __shared__ __align__(16) _Float16 BH[kWinPts * kIRow], BL[kWinPts * kIRow];
  __shared__ __align__(16) float WY[kWinPts * ROWY], WX[kWinPts * L::ROWX];
  __shared__ float RED[4][2][kWinPts];  // per wave: re, im of each point
  __shared__ float4 WB[4 * kWinBuf];    // window rows on their way to the lanes
  __shared__ __align__(16) int REACH[kWinPts / 16];   // x cells each group of 16 points reaches
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g4 = lane >> 4;
  const XcdChunk r(pa);
  if (r.begin >= r.end) return;

  const uint32_t *perm = pa.cperm;
  Rounds ahead(r, pa);
  uint32_t np = perm[ahead.pos(lane)];
  float4 ra = zr.r[np];
  // staging roles (0 x, 1 y, 2 z, 3 writes the outputs) move round the waves
  int role = wave;
  uint32_t j = 0, jn = 0;
  if (role == 3) jn = zr.i[np];
  ahead.advance();
  np = perm[ahead.pos(lane)];

  GridWin<W, H> win;
  const int e = grid_exp(gmax, lane), e_out = e - kProdBits;
  const float s_in = ldexpf(1.0f, kValBits - e);
  ClassWalk cw(r, pa);
  WTile t{};
  bool open = false;
  do {
    const WTile n = win_tile<W>(g, cw.bin, cw.cls, pa.cw);
    // rows carry over along a pencil, ascending classes
    const int first = open && n.xlo == t.xlo && n.z0 == t.z0 && n.y0 >= t.y0
                          ? 16 * H - min(16 * H, n.y0 - t.y0) : 0;
    open = true;
    t = n;
    if (first < 16 * H) win.template load<interp_groups_per_cu(XW, H) < 4 || XW < 4>(grid, g, t, first, s_in, wave,
                                                                   i16, g4, WB + wave * kWinBuf);
    const int oz = t.z0 - even_z0(t.z0);
    const int npt = cw.hi - cw.lo;
    for (int c0 = 0; c0 < npt; c0 += kWinPts) {
      const int npts = min(kWinPts, npt - c0);
      const bool ok = lane < npts;
      {
        int p = lane;
        asm volatile("" : "+v"(p));  // no hoisted row addresses
        const int off = __float_as_int(ra.w);
        if (role == 0) {
          stage_reach<W>(REACH, off, npts, lane);
          interp_stage_x<W, false>(WX + p * L::ROWX, ok, ra.x, off & 255, &dpoly->p.c[0][0]);
        } else if (role == 1) {
          interp_stage_y<W, H, false>(WY + p * ROWY, ok, ra.y, ((off >> 8) & 255) - t.o1 + t.y0,
                                   &dpoly->p.c[0][0]);
        } else if (role == 2) {
          interp_stage_z<W, false>(BH + p * kIRow, BL + p * kIRow, ok, ra.z, ((off >> 16) & 255) + oz,
                                   &dpoly->op[0][0]);
        } else {
          j = jn;
        }
      }
      __syncthreads();
      const bool writer = role == 3;
      role = (role + 1) & 3;
      ra = zr.r[np];
      if (role == 3) jn = zr.i[np];
      ahead.advance();
      np = perm[ahead.pos(lane)];
      for (int gi = 0; gi < (npts + 15) >> 4; ++gi) {
        const int k = 16 * gi + i16;  // this lane's point
        const half8 bh = *(const half8 *)(BH + k * kIRow + 8 * g4);
        const half8 bl = *(const half8 *)(BL + k * kIRow + 8 * g4);
        // wy at this lane's D rows (ring rows 4 g4 .. 4 g4 + 3 of each half), wx
        // at the wave's cells
        float4 wy[H];
#pragma unroll
        for (int h = 0; h < H; ++h) wy[h] = *(const float4 *)(WY + k * ROWY + 16 * h + 4 * g4);
        float wx[XW];
#pragma unroll
        for (int q = 0; q < XW; ++q) wx[q] = WX[k * L::ROWX + 4 * q + wave];
        // cells the group reaches: c0 <= 4 q < c1 (the others' weights are zero)
        const int cells = __builtin_amdgcn_readfirstlane(REACH[gi]);
        const int c0 = (cells & 0xffff) - wave, c1 = (cells >> 16) - wave;
        float accr = 0.f, acci = 0.f;
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        reached_cells<XW>(c0, c1, [&](auto q0, auto q1) {
          f32x4 dr[2], di[2];
          // products of one cell (and half) are issued before the contraction of
          // the one before
#pragma unroll
          for (int u = q0 * H; u <= q1 * H; ++u) {
            if (u < q1 * H) {
              const int q = u / H, h = u % H;
              f32x4 &a = dr[u & 1], &b = di[u & 1];
              a = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rh[h][q], bh, zero, 0, 0, 0);
              b = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.ih[h][q], bh, zero, 0, 0, 0);
              a = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rh[h][q], bl, a, 0, 0, 0);
              b = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.ih[h][q], bl, b, 0, 0, 0);
              a = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rl[h][q], bh, a, 0, 0, 0);
              b = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.il[h][q], bh, b, 0, 0, 0);
            }
            if (u > q0 * H) {
              const int q = (u - 1) / H, h = (u - 1) % H;
              const f32x4 &a = dr[(u - 1) & 1], &b = di[(u - 1) & 1];
              const float4 y = wy[h];
              const float pr = fmaf(y.x, a[0], fmaf(y.y, a[1], fmaf(y.z, a[2], y.w * a[3])));
              const float pi = fmaf(y.x, b[0], fmaf(y.y, b[1], fmaf(y.z, b[2], y.w * b[3])));
              accr = fmaf(wx[q], pr, accr);
              acci = fmaf(wx[q], pi, acci);
            }
          }
        });
        const float s = sum_groups(accr, acci);
        if ((g4 & 1) == 0) RED[wave][g4 >> 1][k] = s;
      }
      __syncthreads();
      if (writer && ok) {
        const float re = (RED[0][0][lane] + RED[1][0][lane]) + (RED[2][0][lane] + RED[3][0][lane]);
        const float im = (RED[0][1][lane] + RED[1][1][lane]) + (RED[2][1][lane] + RED[3][1][lane]);
        out[j] = make_float2(ldexpf(re, e_out), ldexpf(im, e_out));
      }
    }
  } while (cw.next());
}

// Coordinate gradient: with D_i[y][k] = sum_z G_i[y][z] wz_k(z) and E_i[y][k] =
// sum_z G_i[y][z] wz'_k(z) the three derivative sums are
//   Sx_k = sum_i wx'_k(i) sum_y wy_k(y) D_i,  Sy_k = sum_i wx_k(i) sum_y wy'_k(y) D_i,
//   Sz_k = sum_i wx_k(i) sum_y wy_k(y) E_i,
// and grad_a = -scale_a Re(conj(u_k) S_a), u_k from the point's record (the
// binning stores u in the value fields).  Twelve products per x cell.
template <int W>
constexpr int grad_groups_per_cu() { return 2; }

template <int W>
__global__ __launch_bounds__(Win<W>::NT, grad_groups_per_cu<W>()) void win_grad_kernel(
    PointArgs pa, ZRec zr, const float2 *grid, const float *gmax, float *gx, float *gy, float *gz,
    Geom g, const WinPoly *__restrict__ dpoly) {
  using WN = Win<W>;
  using L = ILds<W>;
  constexpr int XW = WN::XW;
  __shared__ __align__(16) _Float16 BH[kWinPts * kIRow], BL[kWinPts * kIRow];
  __shared__ __align__(16) _Float16 DH[kWinPts * kIRow], DL[kWinPts * kIRow];
  __shared__ __align__(16) float WY[kWinPts * kIRowY], WX[kWinPts * L::ROWX];
  __shared__ __align__(16) float DY[kWinPts * kIRowY], DX[kWinPts * L::ROWX];
  __shared__ float RED[4][6][kWinPts];
  __shared__ float4 WB[4 * kWinBuf];
  __shared__ __align__(16) int REACH[kWinPts / 16];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g4 = lane >> 4;
  const XcdChunk r(pa);
  if (r.begin >= r.end) return;

  const uint32_t *perm = pa.cperm;
  Rounds ahead(r, pa);
  uint32_t np = perm[ahead.pos(lane)];
  float4 ra = zr.r[np];
  // staging roles (0 x, 1 y, 2 z values, 3 z derivatives) move round the
  // waves; role 2 also writes the outputs
  int role = wave;
  float2 u = make_float2(0.f, 0.f), un = u;  // writer: the point's u and index
  uint32_t j = 0, jn = 0;
  if (role == 2) un = zr.v[np], jn = zr.i[np];
  ahead.advance();
  np = perm[ahead.pos(lane)];

  GridWin<W, 1> win;
  const int e = grid_exp(gmax, lane), e_out = e - kProdBits, e_outd = e - kProdBitsD;
  const float s_in = ldexpf(1.0f, kValBits - e);
  ClassWalk cw(r, pa);
  WTile t{};
  bool open = false;
  do {
    const WTile n = win_tile<W>(g, cw.bin, cw.cls, pa.cw);
    // rows carry over along a pencil, ascending classes
    const int first = open && n.xlo == t.xlo && n.z0 == t.z0 && n.y0 >= t.y0 ? 16 - min(16, n.y0 - t.y0) : 0;
    open = true;
    t = n;
    if (first < 16) win.template load<true>(grid, g, t, first, s_in, wave, i16, g4, WB + wave * kWinBuf);
    const int oz = t.z0 - even_z0(t.z0);
    const int npt = cw.hi - cw.lo;
    for (int c0 = 0; c0 < npt; c0 += kWinPts) {
      const int npts = min(kWinPts, npt - c0);
      const bool ok = lane < npts;
      {
        int p = lane;
        asm volatile("" : "+v"(p));
        const int off = __float_as_int(ra.w);
        if (role == 0) {
          stage_reach<W>(REACH, off, npts, lane);
          interp_stage_x<W, false>(WX + p * L::ROWX, ok, ra.x, off & 255, &dpoly->p.c[0][0]);
          interp_stage_x<W, true>(DX + p * L::ROWX, ok, ra.x, off & 255, &dpoly->p.dc[0][0]);
        } else if (role == 1) {
          const int s = ((off >> 8) & 255) - t.o1 + t.y0;
          interp_stage_y<W, 1, false>(WY + p * kIRowY, ok, ra.y, s, &dpoly->p.c[0][0]);
          interp_stage_y<W, 1, true>(DY + p * kIRowY, ok, ra.y, s, &dpoly->p.dc[0][0]);
        } else if (role == 2) {
          u = un;
          j = jn;
          interp_stage_z<W, false>(BH + p * kIRow, BL + p * kIRow, ok, ra.z, ((off >> 16) & 255) + oz,
                                   &dpoly->op[0][0]);
        } else {
          interp_stage_z<W, true>(DH + p * kIRow, DL + p * kIRow, ok, ra.z, ((off >> 16) & 255) + oz,
                                  &dpoly->dop[0][0]);
        }
      }
      __syncthreads();
      const bool writer = role == 2;
      role = (role + 1) & 3;
      ra = zr.r[np];
      if (role == 2) un = zr.v[np], jn = zr.i[np];
      ahead.advance();
      np = perm[ahead.pos(lane)];
      for (int gi = 0; gi < (npts + 15) >> 4; ++gi) {
        const int k = 16 * gi + i16;  // this lane's point
        const half8 bh = *(const half8 *)(BH + k * kIRow + 8 * g4);
        const half8 bl = *(const half8 *)(BL + k * kIRow + 8 * g4);
        const half8 dh = *(const half8 *)(DH + k * kIRow + 8 * g4);
        const half8 dl = *(const half8 *)(DL + k * kIRow + 8 * g4);
        const float4 wy = *(const float4 *)(WY + k * kIRowY + 4 * g4);
        const float4 dy = *(const float4 *)(DY + k * kIRowY + 4 * g4);
        float wx[XW], dx[XW];
#pragma unroll
        for (int q = 0; q < XW; ++q) wx[q] = WX[k * L::ROWX + 4 * q + wave];
#pragma unroll
        for (int q = 0; q < XW; ++q) dx[q] = DX[k * L::ROWX + 4 * q + wave];
        float sv[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};  // Sx, Sy, Sz (re, im)
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        // cells the group reaches: c0 <= 4 q < c1 (the others' weights are zero)
        const int cells = __builtin_amdgcn_readfirstlane(REACH[gi]);
        const int c0 = (cells & 0xffff) - wave, c1 = (cells >> 16) - wave;
        reached_cells<XW>(c0, c1, [&](auto q0, auto q1) {
          f32x4 dr[2], di[2], er[2], ei[2];
#pragma unroll
          for (int q = q0; q <= q1; ++q) {
            if (q < q1) {
              f32x4 &a = dr[q & 1], &b = di[q & 1], &c = er[q & 1], &d = ei[q & 1];
              a = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rh[0][q], bh, zero, 0, 0, 0);
              b = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.ih[0][q], bh, zero, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rh[0][q], dh, zero, 0, 0, 0);
              d = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.ih[0][q], dh, zero, 0, 0, 0);
              a = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rh[0][q], bl, a, 0, 0, 0);
              b = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.ih[0][q], bl, b, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rh[0][q], dl, c, 0, 0, 0);
              d = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.ih[0][q], dl, d, 0, 0, 0);
              a = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rl[0][q], bh, a, 0, 0, 0);
              b = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.il[0][q], bh, b, 0, 0, 0);
              c = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.rl[0][q], dh, c, 0, 0, 0);
              d = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.il[0][q], dh, d, 0, 0, 0);
            }
            if (q > q0) {
              const f32x4 &a = dr[(q - 1) & 1], &b = di[(q - 1) & 1];
              const f32x4 &c = er[(q - 1) & 1], &d = ei[(q - 1) & 1];
              const float xw = wx[q - 1], xd = dx[q - 1];
              const float ar = fmaf(wy.x, a[0], fmaf(wy.y, a[1], fmaf(wy.z, a[2], wy.w * a[3])));
              const float ai = fmaf(wy.x, b[0], fmaf(wy.y, b[1], fmaf(wy.z, b[2], wy.w * b[3])));
              const float br = fmaf(dy.x, a[0], fmaf(dy.y, a[1], fmaf(dy.z, a[2], dy.w * a[3])));
              const float bi = fmaf(dy.x, b[0], fmaf(dy.y, b[1], fmaf(dy.z, b[2], dy.w * b[3])));
              const float cr = fmaf(wy.x, c[0], fmaf(wy.y, c[1], fmaf(wy.z, c[2], wy.w * c[3])));
              const float ci = fmaf(wy.x, d[0], fmaf(wy.y, d[1], fmaf(wy.z, d[2], wy.w * d[3])));
              sv[0] = fmaf(xd, ar, sv[0]);
              sv[1] = fmaf(xd, ai, sv[1]);
              sv[2] = fmaf(xw, br, sv[2]);
              sv[3] = fmaf(xw, bi, sv[3]);
              sv[4] = fmaf(xw, cr, sv[4]);
              sv[5] = fmaf(xw, ci, sv[5]);
            }
          }
        });
#pragma unroll
        for (int c = 0; c < 6; c += 2) {
          const float s = sum_groups(sv[c], sv[c + 1]);
          if ((g4 & 1) == 0) RED[wave][c + (g4 >> 1)][k] = s;
        }
      }
      __syncthreads();
      if (writer && ok) {
        float sv[6];
#pragma unroll
        for (int c = 0; c < 6; ++c)
          sv[c] = ldexpf((RED[0][c][lane] + RED[1][c][lane]) + (RED[2][c][lane] + RED[3][c][lane]),
                         c < 4 ? e_out : e_outd);
        // Re(conj(u) * (-s) * S) = -s (u.x S.x + u.y S.y)
        gx[j] = -(float)g.scale[0] * (u.x * sv[0] + u.y * sv[1]);
        if (gy) gy[j] = -(float)g.scale[1] * (u.x * sv[2] + u.y * sv[3]);
        if (gz) gz[j] = -(float)g.scale[2] * (u.x * sv[4] + u.y * sv[5]);
      }
    }
  } while (cw.next());
}

// Write descriptors passed by value into the device table.
__global__ void batch_table_kernel(BatchChunk chunk, SpreadProblem *table) {
  const int i = threadIdx.x;
  if (i < chunk.count) table[chunk.first + i] = chunk.probs[i];
}

// prefix[p] = work of the problems < p, prefix[nprob] = total.
__global__ void batch_work_kernel(const SpreadProblem *probs, int nprob, uint32_t *prefix) {
  if (threadIdx.x != 0) return;
  uint32_t acc = 0;
  for (int p = 0; p < nprob; ++p) {
    prefix[p] = acc;
    acc += probs[p].pa.nsub[1];
  }
  prefix[nprob] = acc;
}

template <int W>
struct WinSpread {
  static hipError_t run(const PointArgs &pa, ZRec zr, float2 *grid, const Geom &g,
                        const WinPoly *dpoly, int nblk, hipStream_t s) {
    if (g.bin[0] > Win<W>::BINX)
      hipLaunchKernelGGL((win_spread_kernel<W, wide_cells(W)>), dim3(nblk), dim3(Win<W>::NT), 0, s, pa,
                         zr, grid, g, dpoly);
    else
      hipLaunchKernelGGL((win_spread_kernel<W, win_cells(W)>), dim3(nblk), dim3(Win<W>::NT), 0, s, pa,
                         zr, grid, g, dpoly);
    return hipGetLastError();
  }
};

template <int W>
struct WinSpreadBatched {
  static hipError_t run(const SpreadProblem *probs, const uint32_t *wpre, int nprob,
                        const WinPoly *dpoly, int nblk, hipStream_t s) {
    hipLaunchKernelGGL((win_spread_batched_kernel<W, win_cells(W)>), dim3(nblk), dim3(Win<W>::NT), 0, s, probs,
                       wpre, nprob, dpoly);
    return hipGetLastError();
  }
};

template <int W>
struct WinInterp {
  static hipError_t run(const PointArgs &pa, ZRec zr, const float2 *grid, const float *gmax,
                        float2 *out, const Geom &g, const WinPoly *dpoly, int nblk, hipStream_t s) {
    if constexpr (W >= 7) {  // (anufft_plan::interp_bins takes them from there on)
      if (pa.cw > Win<W>::CW) {
        hipLaunchKernelGGL((win_interp_kernel<W, 2>), dim3(nblk), dim3(Win<W>::NT), 0, s, pa, zr, grid,
                           gmax, out, g, dpoly);
        return hipGetLastError();
      }
    }
    if (pa.cw > Win<W>::CW) return hipErrorInvalidValue;
    hipLaunchKernelGGL((win_interp_kernel<W, 1>), dim3(nblk), dim3(Win<W>::NT), 0, s, pa, zr, grid,
                       gmax, out, g, dpoly);
    return hipGetLastError();
  }
};

template <int W>
struct WinGrad {
  static hipError_t run(const PointArgs &pa, ZRec zr, const float2 *grid, const float *gmax,
                        float *gx, float *gy, float *gz, const Geom &g, const WinPoly *dpoly,
                        int nblk, hipStream_t s) {
    hipLaunchKernelGGL(win_grad_kernel<W>, dim3(nblk), dim3(Win<W>::NT), 0, s, pa, zr, grid, gmax, gx,
                       gy, gz, g, dpoly);
    return hipGetLastError();
  }
};

template <int W>
struct WinShape {
  static hipError_t run(bool wide, int *binx) {
    *binx = wide ? Win<W, wide_cells(W)>::BINX : Win<W>::BINX;
    return hipSuccess;
  }
};

} // namespace

int win_bin_x(int w, bool wide) {
  int v = 1;
  (void)dispatch_w<WinShape>(w, wide, &v);
  return v;
}

// Workgroups per CU: the resident ones, times what the points allow.  More
// workgroups than fit even out their finishing times, and each costs its
// first and last window.  At 16e6 points, w = 8, 15 instead of 3 per CU cut
// spreading from 2.85 to 2.36 ms and interpolation from 2.80 to 2.53 (w = 4:
// 1.23 to 1.42 at 16, as a spreading workgroup flushes a whole window for few
// products; interpolation 1.40 to 1.15); at 1e6 points more than the resident
// ones lose (w = 6: 155 us at 3, 185 at 6).
static int groups(int64_t num_points, int cus, int resident, int most) {
  const int64_t per_cu = num_points / (1250 * (int64_t)std::max(cus, 1));
  return (int)std::min<int64_t>(std::max<int64_t>(per_cu / resident * resident, resident), most);
}
template <int W>
struct WinGroups {
  static hipError_t run(int which, int64_t num_points, int cus, int *v) {
    constexpr int R = spread_groups_per_cu(win_cells(W)), I = interp_groups_per_cu(win_cells(W), 1),
                  G = grad_groups_per_cu<W>();
    *v = which == 0   ? groups(num_points, cus, R, W >= 7 ? 5 * R : W >= 5 ? 2 * R : R)
         : which == 1 ? groups(num_points, cus, I, 16 / I * I)
                      : groups(num_points, cus, G, 16 / G * G);
    return hipSuccess;
  }
};
static int win_groups(int which, int w, int64_t num_points, int cus) {
  int v = 1;
  (void)dispatch_w<WinGroups>(w, which, num_points, cus, &v);
  return v;
}
int win_spread_groups(int w, const Geom &g, int64_t num_points, int cus) {
  if (g.bin[0] > win_bin_x(w)) return spread_groups_per_cu(wide_cells(w));  // few points
  return win_groups(0, w, num_points, cus);
}
int win_interp_groups(int w, int cw, int64_t num_points, int cus) {
  if (cw > 17 - 2 * w) return interp_groups_per_cu(win_cells(w), 2);  // few points
  return win_groups(1, w, num_points, cus);
}
int win_grad_groups(int w, int64_t num_points, int cus) { return win_groups(2, w, num_points, cus); }

hipError_t launch_win_interp(int w, const PointArgs &pa, ZRec zr, const float2 *grid,
                             const float *gmax, float2 *out, const Geom &g, const WinPoly *dpoly,
                             int num_blocks, hipStream_t s) {
  return dispatch_w<WinInterp>(w, pa, zr, grid, gmax, out, g, dpoly, num_blocks, s);
}
hipError_t launch_win_grad(int w, const PointArgs &pa, ZRec zr, const float2 *grid,
                           const float *gmax, float *gx, float *gy, float *gz, const Geom &g,
                           const WinPoly *dpoly, int num_blocks, hipStream_t s) {
  return dispatch_w<WinGrad>(w, pa, zr, grid, gmax, gx, gy, gz, g, dpoly, num_blocks, s);
}

hipError_t launch_win_spread(int w, const PointArgs &pa, ZRec zr, float2 *grid, const Geom &g,
                             const WinPoly *dpoly, int num_blocks, hipStream_t s) {
  return dispatch_w<WinSpread>(w, pa, zr, grid, g, dpoly, num_blocks, s);
}

hipError_t launch_win_spread_batched(int w, const SpreadProblem *host_probs, int nprob,
                                     SpreadProblem *dev_table, uint32_t *dev_prefix,
                                     const WinPoly *dpoly, int num_blocks, hipStream_t s) {
  for (int first = 0; first < nprob; first += kBatchChunk) {
    BatchChunk chunk{};
    chunk.first = first;
    chunk.count = std::min(kBatchChunk, nprob - first);
    for (int i = 0; i < chunk.count; ++i) chunk.probs[i] = host_probs[first + i];
    hipLaunchKernelGGL(batch_table_kernel, dim3(1), dim3(64), 0, s, chunk, dev_table);
  }
  hipLaunchKernelGGL(batch_work_kernel, dim3(1), dim3(64), 0, s, (const SpreadProblem *)dev_table,
                     nprob, dev_prefix);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return dispatch_w<WinSpreadBatched>(w, (const SpreadProblem *)dev_table,
                                      (const uint32_t *)dev_prefix, nprob, dpoly, num_blocks, s);
}

} // namespace anufft
