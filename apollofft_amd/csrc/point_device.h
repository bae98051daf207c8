// point_device.h -- device helpers shared by the point kernels (spread.hip,
// window.hip, block_spread.hip): periodic indices, wave reductions, tap polynomials, the FP16
// split of FP32 operands and the work shares of the persistent launches.
#pragma once

#include "internal.h"

namespace anufft {

// Periodic index; padded tiles may exceed the grid by more than one period
// when the grid is not much larger than the kernel support.
__device__ __forceinline__ int wrap(int v, int m) {
  if (v < 0) v += m;  // tiles start less than m cells before the grid
  if (v >= m) v -= m;
  if (v < 0 || v >= m) v = v < 0 ? (v % m + m) % m : v % m;  // rarely taken
  return v;
}

template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xf, false));
}

// Sum over the 64 lanes of a wave with DPP (quad swaps, row mirrors, row
// broadcasts) instead of LDS permutes; the total is read from lane 63.
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<0xB1>(v);        // quad_perm [1,0,3,2]
  v += dpp<0x4E>(v);        // quad_perm [2,3,0,1]
  v += dpp<0x141>(v);       // row_half_mirror
  v += dpp<0x140>(v);       // row_mirror: every lane holds its row's sum
  v += dpp<0x142, 0xa>(v);  // row_bcast15 into rows 1 and 3
  v += dpp<0x143, 0xc>(v);  // row_bcast31 into rows 2 and 3
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

typedef const float __attribute__((address_space(4))) *ConstFloatPtr;
typedef int int4v __attribute__((ext_vector_type(4)));
typedef const int4v __attribute__((address_space(4))) *ConstInt4Ptr;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// hi = fp16(a) (round to nearest, packed pairs), lo = fp16(a - hi) (round
// toward zero, packed pairs).  Both halves of a register are written by one
// packed conversion: split sequences that wrote the low and high halves of a
// register with separate half-register instructions gave sporadically wrong
// low parts on gfx950, while packed conversions of the same values did not.
__device__ __forceinline__ void split8(const float *a, half8 &hi, half8 &lo) {
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    const float2v v = {a[j], a[j + 1]};
    const half2v h = __builtin_convertvector(v, half2v);
    typedef __fp16 fp16x2 __attribute__((ext_vector_type(2)));
    const fp16x2 l = __builtin_amdgcn_cvt_pkrtz(a[j] - (float)h[0], a[j + 1] - (float)h[1]);
    hi[j] = h[0];
    hi[j + 1] = h[1];
    lo[j] = (_Float16)l[0];
    lo[j + 1] = (_Float16)l[1];
  }
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// Maximum of non-negative values over the 64 lanes (the DPP steps of
// wave_sum; lanes a step does not write read 0, which is neutral here).
__device__ __forceinline__ float wave_max_nonneg(float v) {
  v = fmaxf(v, dpp<0xB1>(v));
  v = fmaxf(v, dpp<0x4E>(v));
  v = fmaxf(v, dpp<0x141>(v));
  v = fmaxf(v, dpp<0x140>(v));
  v = fmaxf(v, dpp<0x142, 0xa>(v));
  v = fmaxf(v, dpp<0x143, 0xc>(v));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}


// Work range [w0, w1) of this workgroup out of total work wt: each XCD
// takes one contiguous eighth (blocks are dealt to the XCDs round-robin,
// block b on XCD b mod 8) and splits it evenly among its blocks, so a
// workgroup walks consecutive tiles of a pencil and the XCD's tiles meet in
// its L2.
__device__ __forceinline__ void xcd_work_range(uint32_t wt, uint32_t &w0, uint32_t &w1) {
  constexpr uint32_t kXcd = 8;
  const uint32_t g = gridDim.x, b = blockIdx.x;
  if (g < kXcd) {
    w0 = (uint32_t)((uint64_t)wt * b / g);
    w1 = (uint32_t)((uint64_t)wt * (b + 1) / g);
    return;
  }
  const uint32_t x = b % kXcd, j = b / kXcd;
  const uint32_t per = (g - x + kXcd - 1) / kXcd;  // blocks on XCD x
  const uint64_t lo = (uint64_t)wt * x / kXcd, hi = (uint64_t)wt * (x + 1) / kXcd;
  w0 = (uint32_t)(lo + (hi - lo) * j / per);
  w1 = (uint32_t)(lo + (hi - lo) * (j + 1) / per);
}

// First subproblems a, b in [0, n] whose work prefix subs[i].w is >= wa, wb
// (n if none): each step of the search is one load of 64 entries by a wave's
// lanes, for both at once (a list of 1857 entries: 2 dependent loads where
// bisection had 22, some 0.7 us each before a workgroup's first point).
__device__ __forceinline__ void work_lower_bounds(const int4 *subs, uint32_t n, uint32_t wa,
                                                  uint32_t wb, uint32_t &a, uint32_t &b) {
  const uint32_t lane = threadIdx.x & 63u;
  uint32_t lo[2] = {0, 0}, hi[2] = {n, n};
  while (lo[0] < hi[0] || lo[1] < hi[1]) {
    uint32_t step[2], v[2], p[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      step[k] = (hi[k] - lo[k] + 63u) >> 6;
      p[k] = lo[k] + lane * step[k];
      v[k] = (uint32_t)subs[min(p[k], n - 1)].w;
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (lo[k] >= hi[k]) continue;
      // the probes below the bound come first
      const uint32_t c = (uint32_t)__popcll(__ballot(p[k] < hi[k] && v[k] < (k == 0 ? wa : wb)));
      const uint32_t l = lo[k];
      lo[k] = c == 0 ? l : l + (c - 1) * step[k] + 1;
      hi[k] = min(hi[k], l + c * step[k]);
    }
  }
  a = lo[0];
  b = lo[1];
}

// The share of the subproblem list of this workgroup: the work range
// [w0, w1) of xcd_work_range over the list's work prefix W (W(i) =
// subs[i].w).  Subproblem i spans the work interval [W(i), W(i + 1)): its
// fixed cost first, then one unit per kWorkUnit points.  The workgroup owns the points whose units fall in
// its range, so the subproblems at the two ends of its run may be split with
// the neighbouring workgroups (each pays the fixed cost) and every
// workgroup gets the same work however coarse the subproblems are; every
// unit lies in exactly one range, so the shares partition the points.
// begin .. end - 1 are the subproblems whose intervals meet the range;
// points [h0, h1) of subproblem begin and [0, t1) of subproblem end - 1 are
// this workgroup's, every subproblem between is whole.
struct XcdChunk {
  uint32_t begin, end;
  int h0, h1, t1;
  __device__ __forceinline__ XcdChunk(const PointArgs &pa) {
    uint32_t w0, w1;
    xcd_work_range(pa.nsub[1], w0, w1);
    init(pa.subs, pa.nsub[0], pa.nsub[1], w0, w1);
  }
  // The share [w0, w1) of a list of n subproblems of total work wt.
  __device__ __forceinline__ XcdChunk(const int4 *subs, uint32_t n, uint32_t wt, uint32_t w0,
                                      uint32_t w1) {
    init(subs, n, wt, w0, w1);
  }
  __device__ __forceinline__ void init(const int4 *subs, uint32_t n, uint32_t wt, uint32_t w0,
                                       uint32_t w1) {
    uint32_t b;
    work_lower_bounds(subs, n, w0 + 1, w1, b, end);  // b: first i with W(i) > w0
    begin = b > 0 ? b - 1 : 0;
    // drop a head or tail subproblem of which no point is this workgroup's
    // (the range starts past its points, or ends inside its fixed cost), so
    // that every subproblem of the run has points
    h0 = h1 = t1 = 0;
    int t0;
    if (begin < end) {
      owned(subs, n, wt, begin, w0, w1, h0, h1);
      if (h1 <= h0 && ++begin < end) owned(subs, n, wt, begin, w0, w1, h0, h1);
      if (h1 <= h0) begin = end;
    }
    if (end - begin > 1) {
      owned(subs, n, wt, end - 1, w0, w1, t0, t1);
      if (t1 <= 0 && --end - begin > 1) owned(subs, n, wt, end - 1, w0, w1, t0, t1);
    }
    begin = __builtin_amdgcn_readfirstlane(begin);
    end = __builtin_amdgcn_readfirstlane(end);
    h0 = __builtin_amdgcn_readfirstlane(h0);
    h1 = __builtin_amdgcn_readfirstlane(h1);
    t1 = __builtin_amdgcn_readfirstlane(t1);
  }
  // Points [p0, p1) of subproblem i whose units fall in [w0, w1).
  __device__ __forceinline__ static void owned(const int4 *subs, uint32_t n, uint32_t wt, uint32_t i,
                                               uint32_t w0, uint32_t w1, int &p0, int &p1) {
    const int4 sub = subs[i];
    const uint32_t wi = (uint32_t)sub.w, wn = i + 1 < n ? (uint32_t)subs[i + 1].w : wt;
    const uint32_t u = ((uint32_t)sub.z + kWorkUnit - 1) / kWorkUnit;
    const uint32_t a = wi + (wn - wi > u ? wn - wi - u : 0u);  // unit 0's place
    const uint32_t last = wn - 1;  // unit k sits at min(a + k, last)
    auto first = [&](uint32_t w) { return last < w ? u : (w <= a ? 0u : min(u, w - a)); };
    p0 = (int)(first(w0) * kWorkUnit);
    p1 = min(sub.z, (int)(first(w1) * kWorkUnit));
  }
  // Subproblem i (sub = subs[i]) of begin .. end - 1 narrowed to this
  // workgroup's points (at least one).
  __device__ __forceinline__ int4 part(uint32_t i, int4 sub) const {
    const int y = i == begin ? sub.y + h0 : sub.y;
    const int z = i == begin ? h1 - h0 : (i + 1 == end ? t1 : sub.z);
    // wave-uniform values: kept in scalar registers
    return make_int4(sub.x, __builtin_amdgcn_readfirstlane(y), __builtin_amdgcn_readfirstlane(z),
                     sub.w);
  }
};

// F<w>::run for the kernel widths built.
template <template <int> class F, typename... A>
hipError_t dispatch_w(int w, A &&...args) {
  switch (w) {
  case 2: return F<2>::run(args...);
  case 3: return F<3>::run(args...);
  case 4: return F<4>::run(args...);
  case 5: return F<5>::run(args...);
  case 6: return F<6>::run(args...);
  case 7: return F<7>::run(args...);
  case 8: return F<8>::run(args...);
  default: return hipErrorInvalidValue;
  }
}

} // namespace anufft
