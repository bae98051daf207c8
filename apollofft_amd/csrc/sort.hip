// sort.hip -- point binning by counting sorts on integer tile keys.
//
// Replaces the comparison sorts sort_points_{1d,3d} / sort_positions_{1d,3d}
// of apollo-nufft (transform/dimension_1d.rs:54-99, dimension_3d.rs:74-161):
// the reference orders points by bucket with float tie-breaks; here the key is
// the spreading tile of the point, from an FP64 fold of its coordinates.  Each
// binning ends in a list of subproblems of at most max_sub points of a tile,
// tiles in pencil order (along y, or along x).  One stream, no host
// synchronisation.
//
// * Tile binning, with a class list (matrix-core kernels, up to kTileMaxBins
//   tiles): places from LDS counters, ties in any order; up to kSmallPoints
//   points in one workgroup.
// * One-pass binning (up to kOneMaxBins tiles): stable, on the whole key.
// * Digit passes (any tile count): a stable LSD counting sort,
//     keys   : key[j] = tile of point j, per-chunk histogram of digit 0
//     per digit: per-digit scan of the chunk counts -> stable scatter
//              (histogram of the next digit)
//     bounds : bin_start[b] = lower_bound(sorted keys, b)
//     subproblems (one block): scan of per-tile subproblem counts, the list
//   (with records for the matrix-core kernels, then their class list).
// In the stable ones ties keep the input order, so the permutation is a
// deterministic function of the coordinates that a CPU replay reproduces bit
// for bit.
#include <algorithm>

#include "internal.h"

namespace anufft {
namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ uint32_t tile_key(const PointArgs &pa, const Geom &g, int dim,
                                             int64_t j) {
  int cx, cy = 0, cz = 0;
  fold_coord(pa.x[j * pa.stride], g.scale[0], g.m[0], g.inv_m[0], cx);
  if (dim == 3) {
    fold_coord(pa.y[j * pa.stride], g.scale[1], g.m[1], g.inv_m[1], cy);
    fold_coord(pa.z[j * pa.stride], g.scale[2], g.m[2], g.inv_m[2], cz);
  }
  uint32_t bx = (uint32_t)(cx / g.bin[0]);
  uint32_t by = (uint32_t)(cy / g.bin[1]);
  uint32_t bz = (uint32_t)(cz / g.bin[2]);
  return (bx * (uint32_t)g.nbin[1] + by) * (uint32_t)g.nbin[2] + bz;
}

// keys + digit-0 histogram of each chunk, written digit-major.
__global__ __launch_bounds__(kSortThreads) void keys_kernel(PointArgs pa, Geom g, int dim,
                                                            uint32_t *keys, uint32_t *cnt,
                                                            int nchunks, uint32_t *vmax) {
  __shared__ uint32_t hist[kRadix];
  if (vmax && blockIdx.x == 0 && threadIdx.x < kMaxSlots) vmax[threadIdx.x * kMaxStride] = 0u;
  for (int d = threadIdx.x; d < kRadix; d += kSortThreads) hist[d] = 0;
  __syncthreads();
  int64_t base = (int64_t)blockIdx.x * kSortChunk;
  for (int i = threadIdx.x; i < kSortChunk; i += kSortThreads) {
    int64_t j = base + i;
    if (j < pa.num_points) {
      uint32_t k = tile_key(pa, g, dim, j);
      keys[j] = k;
      atomicAdd(&hist[k & (kRadix - 1)], 1u);
    }
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kRadix; d += kSortThreads)
    cnt[(int64_t)d * nchunks + blockIdx.x] = hist[d];
}

// Keys of the current order: a key array, or the key field of the records.
struct KeySrc {
  const uint32_t *k;
  const float4 *r;
  __device__ __forceinline__ uint32_t operator[](int64_t j) const {
    return r ? __float_as_uint(r[2 * j + 1].z) : k[j];
  }
};

// Per-chunk histogram of digit `shift` (passes after the first).
__global__ __launch_bounds__(kSortThreads) void hist_kernel(KeySrc keys, int64_t n, int shift,
                                                            uint32_t *cnt, int nchunks) {
  __shared__ uint32_t hist[kRadix];
  for (int d = threadIdx.x; d < kRadix; d += kSortThreads) hist[d] = 0;
  __syncthreads();
  int64_t base = (int64_t)blockIdx.x * kSortChunk;
  for (int i = threadIdx.x; i < kSortChunk; i += kSortThreads) {
    int64_t j = base + i;
    if (j < n) atomicAdd(&hist[(keys[j] >> shift) & (kRadix - 1)], 1u);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < kRadix; d += kSortThreads)
    cnt[(int64_t)d * nchunks + blockIdx.x] = hist[d];
}

// ---- exclusive scan of a uint32 array (reduce, scan block sums, apply) ----
// Exclusive scan over a block of NT threads (NT / 64 waves): wave scans by
// shuffles, wave totals through LDS (sh: NT / 64 entries); two barriers.
template <int NT>
__device__ __forceinline__ uint32_t block_scan_waves(uint32_t v, uint32_t *sh, uint32_t &total) {
  constexpr int NWV = NT / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < NWV; ++w) {
    const uint32_t t = sh[w];
    before += w < wave ? t : 0u;
    total += t;
  }
  __syncthreads();  // sh may be reused
  return before + x - v;
}

// Exclusive scan of each digit's row of chunk counts, in place: one block per
// digit, the row walked in tiles of kScanTile with a running carry;
// tot[d] = the row's total.  The scatter adds the digit's base (the totals
// of the smaller digits) itself, so one launch replaces a whole-array scan.
__global__ __launch_bounds__(kScanThreads) void scan_rows_kernel(uint32_t *cnt, int nchunks,
                                                                 uint32_t *tot) {
  __shared__ uint32_t sh[kScanThreads / 64];
  uint32_t *row = cnt + (int64_t)blockIdx.x * nchunks;
  uint32_t carry = 0;
  for (int base = 0; base < nchunks; base += kScanTile) {
    uint32_t v[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
      const int j = base + threadIdx.x * kScanItems + i;
      v[i] = j < nchunks ? row[j] : 0u;
      s += v[i];
    }
    uint32_t total;
    uint32_t ex = block_scan_waves<kScanThreads>(s, sh, total) + carry;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
      const int j = base + threadIdx.x * kScanItems + i;
      if (j < nchunks) row[j] = ex;
      ex += v[i];
    }
    carry += total;
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

// ---- stable scatter of one digit --------------------------------------------
// One block per chunk; the chunk is walked in input order, kSortThreads points
// per step.  Ranks inside a wave come from matching digits with per-bit
// ballots; ranks across the waves of a step from per-wave digit counts.
// With REC the pass moves 32-byte records instead of separate keys and
// indices: the first pass builds each point's record from its coordinates
// and value (keys_in holds the keys of the input order), later passes read
// the records of the current order from `in`; all write to `out`.
struct RecMove {
  ZRec in, out;
  const float2 *values;  // value field present (Type-1) or null
  PointArgs pa;
  Geom g;
  int first, last;
  uint32_t *vmax;        // first pass with values: their largest component, or null
};

__device__ __forceinline__ void value_max(float mx, uint32_t *vmax);

template <bool REC>
__global__ __launch_bounds__(kSortThreads) void scatter_kernel(
    const uint32_t *keys_in, const uint32_t *idx_in, uint32_t *keys_out, uint32_t *idx_out,
    int64_t n, int shift, const uint32_t *offs, const uint32_t *tot, int nchunks, RecMove rm) {
  constexpr int kWaves = kSortThreads / 64;
  static_assert(kSortThreads == kRadix, "one thread per digit");
  __shared__ uint32_t running[kRadix];
  __shared__ uint32_t wcount[kWaves][kRadix];
  __shared__ uint32_t sh[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  {
    // start of digit tid in this chunk: digits below it, then its earlier chunks
    uint32_t all;
    const uint32_t dbase = block_scan_waves<kSortThreads>(tot[tid], sh, all);
    running[tid] = dbase + offs[(int64_t)tid * nchunks + blockIdx.x];
    for (int w = 0; w < kWaves; ++w) wcount[w][tid] = 0;
  }
  __syncthreads();
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  int64_t base = (int64_t)blockIdx.x * kSortChunk;
  float mx = 0.f;
  for (int step = 0; step < kSortItems; ++step) {
    int64_t j = base + (int64_t)step * kSortThreads + tid;
    bool valid = j < n;
    uint32_t key = 0u, idx = 0u;
    float4 ra = make_float4(0.f, 0.f, 0.f, 0.f), rb = ra;
    if (!REC) {
      key = valid ? keys_in[j] : 0u;
      idx = valid ? (idx_in ? idx_in[j] : (uint32_t)j) : 0u;
    } else if (valid) {
      if (rm.first) {
        key = keys_in[j];
        idx = (uint32_t)j;
        float z[3];
        int off;
        point_zrec(rm.pa, rm.g, j, z, off);
        const float2 c = rm.values ? rm.values[j] : make_float2(0.f, 0.f);
        ra = make_float4(z[0], z[1], z[2], __int_as_float(off));
        rb = make_float4(c.x, c.y, __uint_as_float(key), __uint_as_float(idx));
        mx = fmaxf(mx, fmaxf(fabsf(c.x), fabsf(c.y)));
      } else {
        ra = rm.in.r[2 * j];
        rb = rm.in.r[2 * j + 1];
        key = __float_as_uint(rb.z);
      }
    }
    uint32_t d = (key >> shift) & (kRadix - 1);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kRadixBits; ++b) {
      bool bit = (d >> b) & 1u;
      uint64_t m = __ballot(valid && bit);
      peers &= bit ? m : ~m;
    }
    uint32_t rank = (uint32_t)__popcll(peers & lt);
    if (valid && (peers & lt) == 0ull) wcount[wave][d] = (uint32_t)__popcll(peers);
    __syncthreads();
    if (valid) {
      uint32_t pos = running[d] + rank;
      for (int w = 0; w < wave; ++w) pos += wcount[w][d];
      if (REC && rm.last) {
        rm.out.r[pos] = ra;
        if (rm.out.v) rm.out.v[pos] = make_float2(rb.x, rb.y);
        if (rm.out.i) rm.out.i[pos] = __float_as_uint(rb.w);
        keys_out[pos] = key;
      } else if (REC) {
        rm.out.r[2 * (int64_t)pos] = ra;
        rm.out.r[2 * (int64_t)pos + 1] = rb;
      } else {
        keys_out[pos] = key;
        idx_out[pos] = idx;
      }
    }
    __syncthreads();
    for (int dd = tid; dd < kRadix; dd += kSortThreads) {
      uint32_t s = 0;
      for (int w = 0; w < kWaves; ++w) {
        s += wcount[w][dd];
        wcount[w][dd] = 0;
      }
      running[dd] += s;
    }
    __syncthreads();
  }
  if (REC && rm.vmax) value_max(mx, rm.vmax);
}

// bin_start[b] = first sorted position with key >= b, b in [0, nbins].
__global__ void bounds_kernel(KeySrc keys, int64_t n, uint32_t *bin_start, int nbins) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b > nbins) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < (uint32_t)b) lo = mid + 1;
    else hi = mid;
  }
  bin_start[b] = (uint32_t)lo;
}

// The subproblem list runs over the tiles in pencil order -- y fastest, then
// z, then x, so that consecutive entries are neighbouring tiles along y, or
// (along_x) x, z, y; q is the position of a tile in that order.
__device__ __forceinline__ int pencil_bin(int q, int3 nb, bool along_x) {
  if (along_x) {
    const int bx = q % nb.x, pz = q / nb.x;
    return (bx * nb.y + pz / nb.z) * nb.z + pz % nb.z;
  }
  const int by = q % nb.y, t = q / nb.y;
  const int bx = t / nb.z;
  return (bx * nb.y + by) * nb.z + (t - bx * nb.z);
}

// 64-bit exclusive scan over a block of NT threads (see block_scan_waves).
template <int NT>
__device__ __forceinline__ uint64_t block_scan_waves64(uint64_t v, uint64_t *sh, uint64_t &total) {
  constexpr int NWV = NT / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  uint64_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < NWV; ++w) {
    const uint64_t t = sh[w];
    before += w < wave ? t : 0ull;
    total += t;
  }
  __syncthreads();  // sh may be reused
  return before + x - v;
}

// Subproblem list in one block: tiles in pencil order, ceil(count / max_sub)
// subproblems each, exclusive scan of those counts in rounds of kSubRound
// tiles (kSubPer consecutive tiles per thread).  subs[i].w = work before
// subproblem i in list order, in units of kWorkUnit points, a subproblem
// weighing exactly ceil(count / kWorkUnit) + sub_work (its fixed cost); nsub[0] =
// number of subproblems, nsub[1] = total work.  The subproblem counts and
// the work are scanned together (one 64-bit scan: counts in the high word).
// The entries of a round are written by the whole block, each finding its
// tile by a binary search of the tiles' first entries (a tile of a dense
// cluster can hold hundreds of subproblems).
// With from_tot (the tile totals tot of the one-pass binning) the kernel
// first writes bin_start[b] = sum of tot[d] over d < b, b in [0, nbins];
// tot == NULL with no points means all tiles are empty.
constexpr int kSubThreads = 1024;
// LDS of the list for a block of NT threads (rounds of NT * kSubPer tiles).
template <int NT, int kSubPer = 4>
struct SubLds {
  static constexpr int kRound = NT * kSubPer;
  uint32_t sh[NT / 64];
  uint64_t sh64[NT / 64];
  uint32_t first[kRound];  // first entry of each tile of the round
  int4 tinfo[kRound];      // tile: bin, first point, count, work before it
};
template <int NT, int kSubPer = 4>
__device__ __forceinline__ void subproblems_body(SubLds<NT, kSubPer> &L, uint32_t *bin_start,
                                                 const uint32_t *tot, int from_tot, int nbins,
                                                 int3 nb, bool along_x, int max_sub, int sub_work,
                                                 uint32_t *nsub, int4 *subs) {
  constexpr int kSubRound = SubLds<NT, kSubPer>::kRound;
  uint32_t *sh = L.sh;
  uint64_t *sh64 = L.sh64;
  uint32_t *first = L.first;
  int4 *tinfo = L.tinfo;
  if (from_tot) {
    uint32_t run = 0;
    for (int base = 0; base <= nbins; base += kSubRound) {
      const int b0 = base + threadIdx.x * kSubPer;
      uint32_t v[kSubPer], sum = 0;
#pragma unroll
      for (int i = 0; i < kSubPer; ++i) {
        v[i] = (tot && b0 + i < nbins) ? tot[b0 + i] : 0u;
        sum += v[i];
      }
      uint32_t total;
      uint32_t ex = run + block_scan_waves<NT>(sum, sh, total);
#pragma unroll
      for (int i = 0; i < kSubPer; ++i) {
        if (b0 + i <= nbins) bin_start[b0 + i] = ex;
        ex += v[i];
      }
      run += total;
    }
    __syncthreads();  // bin_start is read below by other threads of the block
  }
  const uint32_t ms = (uint32_t)max_sub;
  const uint32_t sw = (uint32_t)sub_work;
  const uint32_t wfull = (ms + kWorkUnit - 1) / kWorkUnit + sw;  // a full subproblem
  uint32_t carry = 0, carry_w = 0;
  for (int base = 0; base < nbins; base += kSubRound) {
    const int q0 = base + threadIdx.x * kSubPer;
    int b[kSubPer];
    uint32_t start[kSubPer], c[kSubPer], k[kSubPer], wk[kSubPer];
    uint64_t sum = 0;
#pragma unroll
    for (int i = 0; i < kSubPer; ++i) {
      b[i] = 0;
      start[i] = c[i] = k[i] = wk[i] = 0u;
      if (q0 + i < nbins) {
        b[i] = pencil_bin(q0 + i, nb, along_x);
        start[i] = bin_start[b[i]];
        c[i] = bin_start[b[i] + 1] - start[i];
        k[i] = (c[i] + ms - 1) / ms;
        // k - 1 full subproblems and the rest: each interval of the work
        // prefix is its fixed cost plus its own units, for any max_sub
        const uint32_t rest = k[i] > 0 ? c[i] - (k[i] - 1) * ms : 0u;
        wk[i] = k[i] > 0 ? (k[i] - 1) * wfull + (rest + kWorkUnit - 1) / kWorkUnit + sw : 0u;
      }
      sum += ((uint64_t)k[i] << 32) | wk[i];
    }
    uint64_t total64;
    const uint64_t ex = block_scan_waves64<NT>(sum, sh64, total64);
    uint32_t o = (uint32_t)(ex >> 32), w = carry_w + (uint32_t)ex;
#pragma unroll
    for (int i = 0; i < kSubPer; ++i) {
      first[threadIdx.x * kSubPer + i] = o;
      tinfo[threadIdx.x * kSubPer + i] = make_int4(b[i], (int)start[i], (int)c[i], (int)w);
      o += k[i];
      w += wk[i];
    }
    __syncthreads();
    const uint32_t total = (uint32_t)(total64 >> 32), total_w = (uint32_t)total64;
    for (uint32_t t = threadIdx.x; t < total; t += NT) {
      // owner = last tile with first <= t; it has t - first < its count
      int lo = 0, hi = kSubRound - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= t) lo = mid;
        else hi = mid - 1;
      }
      const int4 ti = tinfo[lo];
      const uint32_t tl = t - first[lo];
      const uint32_t cnt = min((uint32_t)ti.z - tl * ms, ms);
      subs[carry + t] = make_int4(ti.x, (int)((uint32_t)ti.y + tl * ms), (int)cnt,
                                  (int)((uint32_t)ti.w + tl * wfull));
    }
    carry += total;
    carry_w += total_w;
  }
  if (threadIdx.x == 0) {
    nsub[0] = carry;
    nsub[1] = carry_w;
  }
}

__global__ __launch_bounds__(kSubThreads) void subproblems_kernel(uint32_t *bin_start,
                                                                  const uint32_t *tot, int from_tot,
                                                                  int nbins, int3 nb, bool along_x,
                                                                  int max_sub, int sub_work, uint32_t *nsub,
                                                                  int4 *subs) {
  __shared__ SubLds<kSubThreads> L;
  subproblems_body<kSubThreads>(L, bin_start, tot, from_tot, nbins, nb, along_x, max_sub, sub_work,
                                nsub, subs);
}

// ---- one-pass binning (tile count <= kOneMaxBins) ---------------------------
// A stable counting sort on the whole tile key in one scatter: chunks of
// kOneChunk points in input order, each split into kOneWaves contiguous runs
// of kOneSteps x 64 points, one run per wave.
//   chunk_count   : per-chunk tile histogram, cnt[chunk][tile]
//   chunk_scan    : per-tile exclusive scan over the chunks (in place) and
//                   the tile totals
//   subproblems   : bin_start = exclusive scan of the totals, and the list
//                   (up to kFusedMaxBins tiles: block 0 of the scatter
//                   launch, the chunks then scan the totals themselves)
//   chunk_scatter : each wave ranks its run's points among equal tiles with
//                   ballots (earlier lanes, then earlier steps through a
//                   per-wave LDS row of counts); the rows are scanned across
//                   the waves; a point's place is bin_start[tile] + its
//                   chunk's offset + its wave's offset + its rank.
// Ties keep input order, so the result equals the LSD passes' (and
// numpy.argsort(keys, kind="stable")).

// Largest |component| of a wave's values into the slot of its block, as bits
// (non-negative floats order like their bit patterns).
__device__ __forceinline__ void value_max(float mx, uint32_t *vmax) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0)
    atomicMax(vmax + (blockIdx.x % kMaxSlots) * kMaxStride, __float_as_uint(mx));
}

// Peers of this lane (lanes of the wave with the same key among `valid`
// lanes), from one ballot per key bit.
__device__ __forceinline__ uint64_t key_peers(uint32_t key, bool valid, int bits) {
  uint64_t peers = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool bit = (key >> b) & 1u;
    const uint64_t m = __ballot(valid && bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

// Coordinates of point j (zeros past the end; dim 1 keeps x only).  The
// loads are unconditional, from point 0 past the end (callers launch only
// with points; 1D point arguments alias y and z to x), so that no branch
// around a load makes the compiler wait for it there: all loads of a
// thread stay in flight together.
__device__ __forceinline__ void load_point(const PointArgs &pa, int dim, int64_t j, bool valid,
                                           float (&c)[3]) {
  const int64_t o = (valid ? j : 0) * pa.stride;
  const float x = pa.x[o], y = pa.y[o], z = pa.z[o];
  c[0] = valid ? x : 0.f;
  c[1] = (valid && dim == 3) ? y : 0.f;
  c[2] = (valid && dim == 3) ? z : 0.f;
}

// Tile key of a point from its coordinates (tile_key's arithmetic); with
// REC also the record fields of point_zrec (polynomial arguments, offsets).
template <bool REC>
__device__ __forceinline__ uint32_t fold_point(const float (&c)[3], const Geom &g, int dim,
                                               float (&z)[3], int &off) {
  int cell[3] = {0, 0, 0};
  off = 0;
  z[0] = z[1] = z[2] = 0.f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (a > 0 && dim != 3) break;
    const double t = fold_coord(c[a], g.scale[a], g.m[a], g.inv_m[a], cell[a]);
    if (REC) z[a] = (float)(1.0 - 2.0 * (t - (double)cell[a]));
  }
  int b[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    b[a] = (a > 0 && dim != 3) ? 0 : cell_div(cell[a], g, a);
    if (REC && (a == 0 || dim == 3)) {
      const int o = cell[a] - b[a] * g.bin[a];
      off |= (a == 0 ? o : o + 1) << (8 * a);
    }
  }
  return ((uint32_t)b[0] * (uint32_t)g.nbin[1] + (uint32_t)b[1]) * (uint32_t)g.nbin[2] + (uint32_t)b[2];
}

// Tile histogram of one chunk: every thread loads its points' coordinates
// first (all loads in flight at once), then folds them and counts each in
// LDS (the sums do not depend on the order of the atomic adds).
constexpr int kCountThreads = 1024;
constexpr int kCountPer = kOneChunk / kCountThreads;
__global__ __launch_bounds__(kCountThreads) void chunk_count_kernel(BinProblem pr) {
  extern __shared__ uint32_t hist[];  // nbins
  const uint32_t chunk = blockIdx.x;
  const int nbins = pr.nbins, dim = pr.dim;
  const PointArgs &pa = pr.pa;
  for (int d = threadIdx.x; d < nbins; d += kCountThreads) hist[d] = 0;
  const int64_t base = (int64_t)chunk * kOneChunk + threadIdx.x;
  float c[kCountPer][3];
#pragma unroll
  for (int s = 0; s < kCountPer; ++s) {
    const int64_t j = base + (int64_t)s * kCountThreads;
    load_point(pa, dim, j, j < pa.num_points, c[s]);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < kCountPer; ++s) {
    const int64_t j = base + (int64_t)s * kCountThreads;
    const bool valid = j < pa.num_points;
    float z[3];
    int off;
    if (valid) atomicAdd(&hist[fold_point<false>(c[s], pr.g, dim, z, off)], 1u);
  }
  __syncthreads();
  uint32_t *row = pr.cnt + (int64_t)chunk * nbins;
  for (int d = threadIdx.x; d < nbins; d += kCountThreads) row[d] = hist[d];
}

// cnt[c][d] -> sum of cnt[c'][d] over c' < c (in place); tot[d] = the total.
// A block takes 16 tiles; its 1024 threads split the chunks into 64
// segments per tile (lane group of 16 = 16 consecutive tiles of one chunk),
// so each thread has one short run of loads in flight.
constexpr int kScanDigits = 16;
constexpr int kChunkScanSegs = 64;
__device__ __forceinline__ void chunk_scan(const BinProblem &pr, uint32_t blk) {
  __shared__ uint32_t seg[kChunkScanSegs][kScanDigits];
  uint32_t *cnt = pr.cnt;
  const int nchunks = pr.nchunks, nbins = pr.nbins;
  const int dl = threadIdx.x & (kScanDigits - 1), sg = threadIdx.x / kScanDigits;
  const int d = (int)blk * kScanDigits + dl;
  const int per = (nchunks + kChunkScanSegs - 1) / kChunkScanSegs;
  const int c0 = min(nchunks, sg * per), c1 = min(nchunks, c0 + per);
  uint32_t s = 0;
  if (d < nbins) {
#pragma unroll 8
    for (int c = c0; c < c1; ++c) s += cnt[(int64_t)c * nbins + d];
  }
  seg[sg][dl] = s;
  __syncthreads();
  uint32_t before = 0, total = 0;
#pragma unroll 16
  for (int k = 0; k < kChunkScanSegs; ++k) {
    const uint32_t v = seg[k][dl];
    before += k < sg ? v : 0u;
    total += v;
  }
  if (d < nbins) {
#pragma unroll 8
    for (int c = c0; c < c1; ++c) {
      uint32_t *q = cnt + (int64_t)c * nbins + d;
      const uint32_t v = *q;
      *q = before;
      before += v;
    }
    if (sg == 0) pr.tot[d] = total;
  }
}
__global__ __launch_bounds__(kScanDigits * kChunkScanSegs) void chunk_scan_kernel(BinProblem pr) {
  chunk_scan(pr, blockIdx.x);
}

// Fused list (pr.fused): block 0 writes bin_start and the
// subproblem list from the tile totals, beside the scatter; every other
// block scans the totals into LDS for the tile starts of its own points.
// Otherwise bin_start comes from the list launch before this one.
// Dynamic LDS: kOneWaves rows of nbins 16-bit counts, then (fused) nbins
// 32-bit tile starts; block 0 uses it as a SubLds<kOneThreads>.
constexpr int kFusedTotPer = 16;  // tile totals per thread in the fused scan
// Largest tile count of the fused list: 16 + 4 bytes of LDS per tile within
// the 160 KiB of a workgroup (and kFusedTotPer totals per thread).
constexpr int kFusedMaxBins = 8176;
static_assert(kFusedMaxBins <= kFusedTotPer * kOneThreads, "fused scan covers the tiles");
static_assert(20 * kFusedMaxBins + 4 * kOneWaves <= 160 * 1024, "fused scatter LDS");
static_assert(sizeof(SubLds<kOneThreads>) + 4 * kOneWaves <= 160 * 1024, "list LDS");
template <bool REC>
__global__ __launch_bounds__(kOneThreads) void chunk_scatter_kernel(BinProblem pr) {
  extern __shared__ uint4 scatter_lds[];
  __shared__ uint32_t wsum[kOneWaves];
  uint16_t *rows = (uint16_t *)scatter_lds;
  const bool fused = pr.fused;
  if (fused && blockIdx.x == 0) {
    const int3 nb = pr.dim == 3 ? make_int3(pr.g.nbin[0], pr.g.nbin[1], pr.g.nbin[2])
                                : make_int3(1, 1, 1);
    subproblems_body<kOneThreads>(*(SubLds<kOneThreads> *)scatter_lds, pr.bin_start, pr.tot, 1,
                                  pr.nbins, nb, pr.along_x, pr.max_sub, pr.sub_work, pr.nsub, pr.subs);
    return;
  }
  const uint32_t chunk = blockIdx.x - (fused ? 1u : 0u);
  const int nbins = pr.nbins, dim = pr.dim, bits = pr.bits;
  const PointArgs &pa = pr.pa;
  for (int i = threadIdx.x; i < kOneWaves / 2 * nbins; i += kOneThreads) ((uint32_t *)rows)[i] = 0u;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  uint16_t *row = rows + wave * nbins;
  uint32_t *bst = (uint32_t *)(rows + kOneWaves * nbins);
  const int64_t j0 = (int64_t)chunk * kOneChunk + (int64_t)wave * (64 * kOneSteps) + lane;
  // the wave's coordinates and values, all loads in flight at once
  float c[kOneSteps][3];
  float2 val[kOneSteps];
#pragma unroll
  for (int s = 0; s < kOneSteps; ++s) {
    const int64_t j = j0 + 64 * s;
    const bool valid = j < pa.num_points;
    load_point(pa, dim, j, valid, c[s]);
    val[s] = (REC && pr.values) ? pr.values[valid ? j : 0] : make_float2(0.f, 0.f);
  }
  // fused: this thread's run of tile totals (clamped indices, no branch)
  const int per = (nbins + kOneThreads - 1) / kOneThreads;
  const int t0 = threadIdx.x * per;
  uint32_t tv[kFusedTotPer];
  if (fused) {
#pragma unroll
    for (int i = 0; i < kFusedTotPer; ++i) tv[i] = pr.tot[min(t0 + i, nbins - 1)];
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kFusedTotPer; ++i) sum += (i < per && t0 + i < nbins) ? tv[i] : 0u;
    uint32_t total;
    uint32_t ex = block_scan_waves<kOneThreads>(sum, wsum, total);  // its barriers: rows zeroed
#pragma unroll
    for (int i = 0; i < kFusedTotPer; ++i) {
      if (i < per && t0 + i < nbins) bst[t0 + i] = ex;
      ex += (i < per && t0 + i < nbins) ? tv[i] : 0u;
    }
  } else {
    __syncthreads();  // rows zeroed
  }
  const uint32_t *coff = pr.cnt + (int64_t)chunk * nbins;
  const uint32_t *bin_start = pr.bin_start;
  uint32_t key[kOneSteps], rk[kOneSteps], pos[kOneSteps];
  float zr[kOneSteps][3];
  int off[kOneSteps];
#pragma unroll
  for (int s = 0; s < kOneSteps; ++s) {
    const int64_t j = j0 + 64 * s;
    const bool valid = j < pa.num_points;
    const uint32_t k = valid ? fold_point<REC>(c[s], pr.g, dim, zr[s], off[s]) : 0u;
    // the chunk's offset (and without the fused scan the tile start): loads
    // in flight during the ranking
    pos[s] = coff[k] + (fused ? 0u : bin_start[k]);
    const uint64_t peers = key_peers(k, valid, bits);
    const uint64_t below = peers & lt;
    uint32_t b0 = 0;
    if (valid && below == 0ull) {  // the first lane of each key claims the step's slots
      b0 = row[k];
      row[k] = (uint16_t)(b0 + (uint32_t)__popcll(peers));
    }
    const int leader = valid ? __ffsll((unsigned long long)peers) - 1 : lane;
    b0 = __shfl(b0, leader);
    key[s] = k;
    rk[s] = b0 + (uint32_t)__popcll(below);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < nbins; d += kOneThreads) {
    uint32_t run = 0;
#pragma unroll
    for (int w = 0; w < kOneWaves; ++w) {
      const uint32_t v = rows[w * nbins + d];
      rows[w * nbins + d] = (uint16_t)run;
      run += v;
    }
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < kOneSteps; ++s) {
    const uint32_t k = key[s];
    pos[s] += (fused ? bst[k] : 0u) + (uint32_t)row[k] + rk[s];
  }
#pragma unroll
  for (int s = 0; s < kOneSteps; ++s) {
    const int64_t j = j0 + 64 * s;
    if (j >= pa.num_points) continue;
    if (REC) {
      pr.out.r[pos[s]] = make_float4(zr[s][0], zr[s][1], zr[s][2], __int_as_float(off[s]));
      if (pr.out.v) pr.out.v[pos[s]] = val[s];
      if (pr.out.i) pr.out.i[pos[s]] = (uint32_t)j;
    } else {
      pr.keys_out[pos[s]] = key[s];
      pr.idx_out[pos[s]] = (uint32_t)j;
    }
  }
}

// ---- tile binning (records with a class list) -------------------------------
// The matrix-core kernels order a tile's points by class and x offset
// themselves (class_sort_kernel), so their records need no stable order
// inside a tile: a point takes its place from an LDS counter of its tile
// instead of a rank by ballots, and a chunk can be as long as keeps every CU
// busy with two (the counts of (chunk, tile) pairs stay small).
//   tile_count    : per-chunk tile histogram, cnt[chunk][tile]
//   tile_scan     : per-tile exclusive scan over the chunks (in place) and the
//                   tile totals; left out for a single chunk
//   tile_scatter  : every block scans the totals in LDS for the tile starts;
//                   the first writes the subproblem list, the others add their
//                   chunk's offsets and stream their points to their places
// The scatter is bound by its writes of 20 to 28 bytes a point to scattered
// places.  Measured, count, scan, scatter and class list together against the
// stable one-pass binning: 2e6 points, 1368 tiles, 92 and 75 us; 16e6
// clustered, 6176 tiles, 850 and 480 (with places in input order, no scatter,
// 55 and 316).  (Places from global counters, 490 chunks meeting on each: 26 us
// more at 2e6, 125 at 16e6.)
constexpr int kTileThreads = 1024;

// The problem of this block: the one passed by value, or (BATCH) the last
// table entry whose first block is at most blockIdx.x; first block of entry
// i: chunk0 (COUNT), scan0 (SCAN), or chunk0 + i (SCATTER: a list block each).
enum TileStep { kTileCount, kTileScan, kTileScatter };
template <bool BATCH, TileStep STEP>
__device__ __forceinline__ const BinProblem &tile_problem(const BinProblem &one,
                                                           const BinProblem *table, int nprob,
                                                           uint32_t &local) {
  local = blockIdx.x;
  if (!BATCH) return one;
  auto first = [&](int i) {
    return STEP == kTileScan ? table[i].scan0 : table[i].chunk0 + (STEP == kTileScatter ? i : 0);
  };
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first(mid) <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  local = blockIdx.x - first(lo);
  return table[lo];
}

template <bool BATCH>
__global__ __launch_bounds__(kTileThreads) void tile_count_kernel(BinProblem one,
                                                                  const BinProblem *table,
                                                                  int nprob) {
  extern __shared__ uint32_t hist[];  // nbins
  uint32_t chunk;
  const BinProblem &pr = tile_problem<BATCH, kTileCount>(one, table, nprob, chunk);
  if (!BATCH && chunk >= (uint32_t)pr.nchunks) {  // blocks past the chunks zero pr.zero
    const int64_t st = (int64_t)(gridDim.x - pr.nchunks) * kTileThreads;
    float4 *q = (float4 *)pr.zero;
    const int64_t n4 = pr.zero_n / 2;
    for (int64_t i = (int64_t)(chunk - pr.nchunks) * kTileThreads + threadIdx.x; i < n4; i += st)
      q[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (chunk == (uint32_t)pr.nchunks && threadIdx.x == 0 && (pr.zero_n & 1))
      pr.zero[pr.zero_n - 1] = make_float2(0.f, 0.f);
    return;
  }
  const int nbins = pr.nbins;
  const PointArgs &pa = pr.pa;
  if (chunk == 0 && threadIdx.x < kMaxSlots) pr.cls.vmax[threadIdx.x * kMaxStride] = 0u;
  for (int d = threadIdx.x; d < nbins; d += kTileThreads) hist[d] = 0;
  const int64_t end = min(pa.num_points, (int64_t)(chunk + 1) * pr.chunk);
  int64_t j = (int64_t)chunk * pr.chunk + threadIdx.x;
  float c[3], cn[3];
  load_point(pa, 3, j, j < end, c);
  __syncthreads();
  for (; j < end; j += kTileThreads) {
    load_point(pa, 3, j + kTileThreads, j + kTileThreads < end, cn);
    float z[3];
    int off;
    atomicAdd(&hist[fold_point<false>(c, pr.g, 3, z, off)], 1u);
#pragma unroll
    for (int a = 0; a < 3; ++a) c[a] = cn[a];
  }
  __syncthreads();
  uint32_t *row = pr.cnt + (int64_t)chunk * nbins;
  for (int d = threadIdx.x; d < nbins; d += kTileThreads) row[d] = hist[d];
}

template <bool BATCH>
__global__ __launch_bounds__(kScanDigits * kChunkScanSegs) void tile_scan_kernel(
    BinProblem one, const BinProblem *table, int nprob) {
  uint32_t blk;
  const BinProblem &pr = tile_problem<BATCH, kTileScan>(one, table, nprob, blk);
  chunk_scan(pr, blk);
}

typedef SubLds<kTileThreads, 1> TileSubLds;
// LDS of the scatter: the tile starts (nbins + 1), then (list block) the list's.
static size_t tile_scatter_lds(int nbins) {
  return sizeof(uint32_t) * (((size_t)nbins + 4) & ~(size_t)3) + sizeof(TileSubLds);
}

template <bool BATCH>
__global__ __launch_bounds__(kTileThreads) void tile_scatter_kernel(BinProblem one,
                                                                    const BinProblem *table,
                                                                    int nprob) {
  extern __shared__ uint4 tile_lds[];
  __shared__ float wmax[kTileThreads / 64];
  __shared__ uint32_t sh[kTileThreads / 64];
  uint32_t chunk;
  const BinProblem &pr = tile_problem<BATCH, kTileScatter>(one, table, nprob, chunk);
  const int nbins = pr.nbins;
  const PointArgs &pa = pr.pa;
  uint32_t *place = (uint32_t *)tile_lds;  // next place of each tile
  // tile starts: the totals' exclusive scan, a run of tiles per thread
  for (int d = threadIdx.x; d < nbins; d += kTileThreads) place[d] = pr.tot[d];
  __syncthreads();
  {
    const int per = (nbins + kTileThreads - 1) / kTileThreads;
    const int d0 = min(nbins, (int)threadIdx.x * per), d1 = min(nbins, d0 + per);
    uint32_t sum = 0, total;
    for (int d = d0; d < d1; ++d) sum += place[d];
    uint32_t at = block_scan_waves<kTileThreads>(sum, sh, total);
    for (int d = d0; d < d1; ++d) {
      const uint32_t v = place[d];
      place[d] = at;
      at += v;
    }
    if (threadIdx.x == 0) place[nbins] = total;
  }
  __syncthreads();
  if (chunk == 0) {
    subproblems_body<kTileThreads, 1>(*(TileSubLds *)(place + ((nbins + 4) & ~3)), place, nullptr, 0,
                                      nbins, make_int3(pr.g.nbin[0], pr.g.nbin[1], pr.g.nbin[2]),
                                      pr.along_x, pr.max_sub, pr.sub_work, pr.nsub, pr.subs);
    return;
  }
  --chunk;
  {  // consecutive chunks on one XCD (blocks are dealt to the XCDs in turn):
     // the runs they write in a tile join in its L2 (2e6 points: 79 to 75 us)
    const uint32_t n = (uint32_t)pr.nchunks, x = chunk & 7u;
    chunk = x * (n >> 3) + min(x, n & 7u) + (chunk >> 3);
  }
  const int64_t end = min(pa.num_points, (int64_t)(chunk + 1) * pr.chunk);
  int64_t j = (int64_t)chunk * pr.chunk + threadIdx.x;
  const bool vals = pr.out.v != nullptr;
  float c[3], cn[3];
  float2 v = make_float2(0.f, 0.f), vn = v;
  load_point(pa, 3, j, j < end, c);
  if (vals) v = pr.values[j < end ? j : 0];
  if (pr.nchunks > 1) {
    const uint32_t *coff = pr.cnt + (int64_t)chunk * nbins;
    for (int d = threadIdx.x; d < nbins; d += kTileThreads) place[d] += coff[d];
    __syncthreads();
  }
  float mx = 0.f;
  for (; j < end; j += kTileThreads) {
    const int64_t jn = j + kTileThreads;
    load_point(pa, 3, jn, jn < end, cn);
    if (vals) vn = pr.values[jn < end ? jn : 0];
    float z[3];
    int off;
    const uint32_t p = atomicAdd(&place[fold_point<true>(c, pr.g, 3, z, off)], 1u);
    pr.out.r[p] = make_float4(z[0], z[1], z[2], __int_as_float(off));
    if (vals) {
      pr.out.v[p] = v;
      mx = fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y)));
    }
    if (pr.out.i) pr.out.i[p] = (uint32_t)j;
#pragma unroll
    for (int a = 0; a < 3; ++a) c[a] = cn[a];
    v = vn;
  }
  if (vals) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x < 64) value_max(threadIdx.x < kTileThreads / 64 ? wmax[threadIdx.x] : 0.f, pr.cls.vmax);
  }
}

// ---- class list of the matrix-core kernels ----------------------------------
// Their 16-row windows take the points of one y-offset class of a tile, and a
// window slides along y from class to class.  The tile binning stays coarse
// (its per-chunk counts grow with the tile count, and classes as tiles of
// their own would be 3 to 16 times as many), and the classes are listed inside
// each subproblem of the tile list: one block per subproblem (at most
// kClassSub points) ranks every point among those of its class and x offset
// (LDS atomics) and writes the sorted positions in that order (perm) and the
// classes' starts.  The x order lets the kernels leave out the x cells no
// point of a group reaches.
constexpr int kClsThreads = 256;
constexpr int kClsSteps = kClassSub / kClsThreads;
constexpr int kClsKeys = kClsThreads;  // (class, x offset) pairs at most

// The problem of this block: the one passed by value (no table), or the last
// table entry whose first block is at most blockIdx.x.
__device__ __forceinline__ const BinProblem &piece_problem(const BinProblem &one,
                                                            const BinProblem *table, int nprob,
                                                            uint32_t &local) {
  local = blockIdx.x;
  if (!table) return one;
  int lo = 0, hi = nprob - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (table[mid].piece0 <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  local = blockIdx.x - table[lo].piece0;
  return table[lo];
}

__global__ __launch_bounds__(kClsThreads) void class_sort_kernel(BinProblem one,
                                                                 const BinProblem *table,
                                                                 int nprob) {
  __shared__ uint32_t cnt[kClsKeys];  // points of each key, then its first place
  __shared__ uint32_t sh[kClsThreads / 64];
  uint32_t piece;
  const BinProblem &pr = piece_problem(one, table, nprob, piece);
  if (piece >= pr.nsub[0]) return;
  const ClassBuffers &cb = pr.cls;
  const int ncls = cb.ncls, binx = pr.g.bin[0], nkeys = ncls * binx;
  const int4 sub = pr.subs[piece];
  const int n = sub.z;
  const float *ofs = (const float *)(pr.out.r + sub.y) + 3;  // point p's offsets: ofs[4 p]
  const float inv_cw = 1.0f / (float)cb.cw;
  int o[kClsSteps];
#pragma unroll
  for (int s = 0; s < kClsSteps; ++s) {
    const int p = threadIdx.x + s * kClsThreads;
    o[s] = p < n ? __float_as_int(ofs[4 * (int64_t)p]) : -1;
  }
  cnt[threadIdx.x] = 0u;
  __syncthreads();
  uint32_t rk[kClsSteps];
#pragma unroll
  for (int s = 0; s < kClsSteps; ++s) {
    // class (o1 - 1) / cw of the y offset o1 >= 1 (cell_div's rounding argument)
    const int c = (int)(((float)((o[s] >> 8) & 255) - 0.5f) * inv_cw);
    const int k = c * binx + (o[s] & 255);
    rk[s] = o[s] >= 0 ? atomicAdd(&cnt[k], 1u) : 0u;
    o[s] = o[s] >= 0 ? k : -1;
  }
  __syncthreads();
  uint32_t all;
  const int k = threadIdx.x;
  const uint32_t at = block_scan_waves<kClsThreads>(cnt[k], sh, all);
  if (k < nkeys && k % binx == 0) cb.start[(int64_t)piece * ncls + k / binx] = (uint16_t)at;
  cnt[k] = at;
  __syncthreads();
  uint32_t *perm = cb.perm + (int64_t)sub.y;
#pragma unroll
  for (int s = 0; s < kClsSteps; ++s)
    if (o[s] >= 0) perm[cnt[o[s]] + rk[s]] = (uint32_t)(sub.y + (int)threadIdx.x + s * kClsThreads);
}

// Subproblems of a list at most.
int class_pieces(int64_t n, int nbins, int max_sub) {
  return (int)(std::min<int64_t>(nbins, n) + (n + max_sub - 1) / max_sub);
}
// The whole binning of at most kSmallPoints points by one workgroup: counts of
// (tile, class, x offset) keys in LDS, their scan, the subproblem list, the
// class starts, and the records at once in their final order (the class list
// is the identity).  The launch's other workgroups zero pr.zero.  In place of
// four launches that each wait for the one before (2000 points on 32^3 cells:
// fill, count, scatter and class list 19 us, this kernel 11; a Type-1 call 51
// and 46).
constexpr int kSmallPer = 4;
constexpr int kSmallPoints = kSmallPer * kTileThreads;
constexpr size_t kSmallLds = 148 * 1024;
static int small_keys(const Geom &g, int nbins, int ncls) { return nbins * ncls * g.bin[0]; }
// LDS: key counts (then places), tile starts, the list's.
static size_t small_lds(int nkeys, int nbins) {
  return sizeof(uint32_t) * (((size_t)nkeys + 4) & ~(size_t)3) +
         sizeof(uint32_t) * (((size_t)nbins + 4) & ~(size_t)3) + sizeof(TileSubLds);
}

__global__ __launch_bounds__(kTileThreads) void small_binning_kernel(BinProblem pr) {
  extern __shared__ uint4 tile_lds[];
  __shared__ uint32_t sh[kTileThreads / 64];
  __shared__ float wmax[kTileThreads / 64];
  if (blockIdx.x > 0) {
    const int64_t st = (int64_t)(gridDim.x - 1) * kTileThreads;
    for (int64_t i = (int64_t)(blockIdx.x - 1) * kTileThreads + threadIdx.x; i < pr.zero_n; i += st)
      pr.zero[i] = make_float2(0.f, 0.f);
    return;
  }
  const PointArgs &pa = pr.pa;
  const ClassBuffers &cb = pr.cls;
  const int nbins = pr.nbins, ncls = cb.ncls, binx = pr.g.bin[0], tk = ncls * binx, nkeys = nbins * tk;
  const int n = (int)pa.num_points;
  uint32_t *cnt = (uint32_t *)tile_lds, *starts = cnt + ((nkeys + 4) & ~3);
  const bool vals = pr.out.v != nullptr;
  float c[kSmallPer][3];
  float2 v[kSmallPer];
#pragma unroll
  for (int s = 0; s < kSmallPer; ++s) {
    const int j = (int)threadIdx.x + s * kTileThreads;
    load_point(pa, 3, j, j < n, c[s]);
    v[s] = vals ? pr.values[j < n ? j : 0] : make_float2(0.f, 0.f);
  }
  for (int d = threadIdx.x; d < nkeys; d += kTileThreads) cnt[d] = 0u;
  __syncthreads();
  const float inv_cw = 1.0f / (float)cb.cw;
  float z[kSmallPer][3], mx = 0.f;
  int off[kSmallPer];
  uint32_t key[kSmallPer], rk[kSmallPer];
#pragma unroll
  for (int s = 0; s < kSmallPer; ++s) {
    const uint32_t tile = fold_point<true>(c[s], pr.g, 3, z[s], off[s]);
    const int cls = (int)(((float)((off[s] >> 8) & 255) - 0.5f) * inv_cw);  // as class_sort_kernel
    key[s] = tile * (uint32_t)tk + (uint32_t)(cls * binx + (off[s] & 255));
    rk[s] = 0u;
    if ((int)threadIdx.x + s * kTileThreads < n) {
      rk[s] = atomicAdd(&cnt[key[s]], 1u);
      mx = fmaxf(mx, fmaxf(fabsf(v[s].x), fabsf(v[s].y)));
    }
  }
  __syncthreads();
  {
    // first place of each key: exclusive scan, a run of keys per thread
    const int per = (nkeys + kTileThreads - 1) / kTileThreads;
    const int d0 = min(nkeys, (int)threadIdx.x * per), d1 = min(nkeys, d0 + per);
    uint32_t sum = 0, total;
    for (int d = d0; d < d1; ++d) sum += cnt[d];
    uint32_t at = block_scan_waves<kTileThreads>(sum, sh, total);
    for (int d = d0; d < d1; ++d) {
      const uint32_t k = cnt[d];
      cnt[d] = at;
      at += k;
    }
  }
  __syncthreads();
  // the records, in their final order
#pragma unroll
  for (int s = 0; s < kSmallPer; ++s) {
    const int j = (int)threadIdx.x + s * kTileThreads;
    if (j >= n) continue;
    const uint32_t p = cnt[key[s]] + rk[s];
    pr.out.r[p] = make_float4(z[s][0], z[s][1], z[s][2], __int_as_float(off[s]));
    if (vals) pr.out.v[p] = v[s];
    if (pr.out.i) pr.out.i[p] = (uint32_t)j;
    cb.perm[j] = (uint32_t)j;
  }
  for (int d = threadIdx.x; d <= nbins; d += kTileThreads) starts[d] = d < nbins ? cnt[d * tk] : (uint32_t)n;
  if (vals) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (vals && threadIdx.x < kMaxSlots) {  // (one block: one slot, the others zero)
    float m = 0.f;
    for (int w = 0; w < kTileThreads / 64; ++w) m = fmaxf(m, wmax[w]);
    cb.vmax[threadIdx.x * kMaxStride] = threadIdx.x == 0 ? __float_as_uint(m) : 0u;
  }
  subproblems_body<kTileThreads, 1>(*(TileSubLds *)(starts + ((nbins + 4) & ~3)), starts, nullptr, 0, nbins,
                                    make_int3(pr.g.nbin[0], pr.g.nbin[1], pr.g.nbin[2]), pr.along_x,
                                    pr.max_sub, pr.sub_work, pr.nsub, pr.subs);
  __syncthreads();
  // classes of the subproblems: a tile's class starts, cut to the subproblem
  const int nsub = (int)pr.nsub[0];
  for (int i = threadIdx.x; i < nsub * ncls; i += kTileThreads) {
    const int piece = i / ncls, k = i - piece * ncls;
    const int4 sub = pr.subs[piece];
    const int first = (int)cnt[sub.x * tk + k * binx] - sub.y;
    cb.start[i] = (uint16_t)max(0, min(sub.z, first));
  }
}

// descriptors per table-fill launch (kernarg size)
constexpr int kBinTableChunk = 8;
struct BinTableChunk {
  int first, count;
  BinProblem probs[kBinTableChunk];
};
__global__ void bin_table_kernel(BinTableChunk chunk, BinProblem *table) {
  const int i = threadIdx.x;
  if (i < chunk.count) table[chunk.first + i] = chunk.probs[i];
}

int key_bits(int nbins) {
  int bits = 0;
  while ((1 << bits) < nbins) ++bits;
  return bits;
}

hipError_t set_lds(const void *fn, size_t lds) {
  if (lds <= 65536) return hipSuccess;
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

// Points of a chunk: two chunks a CU on 256 CUs, in steps of a block (twice
// and four times as many: 479, 522 and 593 us at 16e6 points, as their counts
// grow; 75 and 97 at 2e6); up to 4096 points one chunk, whose totals need no
// scan launch (5 us) for a few steps of a block (1 us each).
constexpr int kTileChunks = 512;
int tile_chunk(int64_t n) {
  if (n <= 4 * kTileThreads) return 4 * kTileThreads;
  return (int)(((n + kTileChunks - 1) / kTileChunks + kTileThreads - 1) / kTileThreads) * kTileThreads;
}
int tile_chunks(int64_t n) { return (int)((n + tile_chunk(n) - 1) / tile_chunk(n)); }

// (pr.zero: 16-byte aligned, as workspaces are laid out)
// The tile binning's launches over `chunks` chunks, `scans` scan blocks and
// `pieces` subproblems at most, of one problem or a table.
hipError_t launch_tile_binning(const BinProblem &one, const BinProblem *table, int nprob,
                               int max_bins, uint32_t chunks, uint32_t scans, uint32_t pieces,
                               hipStream_t s) {
  const size_t hist = sizeof(uint32_t) * (size_t)max_bins, lds = tile_scatter_lds(max_bins);
  const void *scatter = table ? (const void *)tile_scatter_kernel<true> : (const void *)tile_scatter_kernel<false>;
  hipError_t e = set_lds(scatter, lds);
  if (e != hipSuccess) return e;
  const dim3 nt(kTileThreads), ns(kScanDigits * kChunkScanSegs), lists(chunks + (uint32_t)nprob);
  if (table) {
    if (chunks > 0) hipLaunchKernelGGL(tile_count_kernel<true>, dim3(chunks), nt, hist, s, one, table, nprob);
    hipLaunchKernelGGL(tile_scan_kernel<true>, dim3(scans), ns, 0, s, one, table, nprob);
    hipLaunchKernelGGL(tile_scatter_kernel<true>, lists, nt, lds, s, one, table, nprob);
  } else {
    const uint32_t fill = (uint32_t)std::min<int64_t>((one.zero_n + 8 * kTileThreads - 1) / (8 * kTileThreads), 2048);
    hipLaunchKernelGGL(tile_count_kernel<false>, dim3(chunks + fill), nt, hist, s, one, table, nprob);
    if (scans > 0) hipLaunchKernelGGL(tile_scan_kernel<false>, dim3(scans), ns, 0, s, one, table, nprob);
    hipLaunchKernelGGL(tile_scatter_kernel<false>, lists, nt, lds, s, one, table, nprob);
  }
  if (pieces > 0)
    hipLaunchKernelGGL(class_sort_kernel, dim3(pieces), dim3(kClsThreads), 0, s, one, table, nprob);
  return hipGetLastError();
}

} // namespace

bool sort_one_pass(int nbins) { return nbins <= kOneMaxBins; }
// (4 bytes of LDS a tile)
bool tile_binning(int nbins) { return nbins <= kTileMaxBins; }

size_t radix_count_entries(int64_t num_points) {
  const int64_t M = std::max<int64_t>(num_points, 1);
  return (size_t)(kRadix * ((M + kSortChunk - 1) / kSortChunk));
}
// The chunks at most of up to num_points points (tile_chunks falls where the
// chunks grow by a step, from 512 at 524288 points to 257 at one more), so that
// a workspace for many points serves fewer.
size_t tile_count_entries(int64_t num_points, int nbins) {
  if (!tile_binning(nbins)) return 0;
  const int64_t chunks = num_points <= 4 * kTileThreads
                             ? 1 : std::min<int64_t>((num_points + kTileThreads - 1) / kTileThreads, kTileChunks);
  return (size_t)nbins * (size_t)chunks;
}
size_t one_pass_count_entries(int64_t num_points, int nbins) {
  const int64_t M = std::max<int64_t>(num_points, 1);
  return sort_one_pass(nbins) ? (size_t)nbins * (size_t)((M + kOneChunk - 1) / kOneChunk) : 0;
}

static BinProblem bin_problem(const PointArgs &pa, const Geom &g, int dim, const SortBuffers &sb,
                              const RecordOut *rec) {
  BinProblem pr{};
  pr.pa = pa;
  pr.g = g;
  pr.cnt = sb.cnt;
  pr.tot = sb.scan_tmp;
  pr.bin_start = sb.bin_start;
  pr.nsub = sb.sub_ofs + sb.nbins;
  pr.subs = sb.subs;
  if (rec) {
    pr.out = rec->out;
    pr.values = rec->values;
    pr.cls = sb.cls;
  } else {
    pr.keys_out = sb.keys[sb.passes & 1];
    pr.idx_out = sb.idx[sb.passes & 1];
  }
  pr.dim = dim;
  pr.nbins = sb.nbins;
  pr.bits = key_bits(sb.nbins);
  pr.max_sub = sb.max_sub;
  pr.sub_work = sb.sub_work;
  pr.along_x = sb.along_x;
  pr.zero = sb.zero;
  pr.zero_n = sb.zero_n;
  return pr;
}

// One-pass binning: see the comment above chunk_count_kernel.
static hipError_t sort_points_one_pass(const PointArgs &pa, const Geom &g, int dim,
                                       const SortBuffers &sb, hipStream_t s,
                                       const RecordOut *rec) {
  const int64_t n = pa.num_points;
  const int nbins = sb.nbins;
  BinProblem pr = bin_problem(pa, g, dim, sb, rec);
  pr.nchunks = (int)((n + kOneChunk - 1) / kOneChunk);
  const int nch = pr.nchunks;
  // with the tile starts in LDS beside the count rows, the scatter launch
  // also writes the list (one more block)
  pr.fused = n > 0 && nbins <= kFusedMaxBins;
  if (n > 0) {
    hipLaunchKernelGGL(chunk_count_kernel, dim3(nch), dim3(kCountThreads), sizeof(uint32_t) * nbins, s,
                       pr);
    hipLaunchKernelGGL(chunk_scan_kernel, dim3((nbins + kScanDigits - 1) / kScanDigits),
                       dim3(kScanDigits * kChunkScanSegs), 0, s, pr);
  }
  if (!pr.fused) {
    // tile starts and the subproblem list need only the counts
    const int3 nb = dim == 3 ? make_int3(g.nbin[0], g.nbin[1], g.nbin[2]) : make_int3(1, 1, 1);
    hipLaunchKernelGGL(subproblems_kernel, dim3(1), dim3(kSubThreads), 0, s, sb.bin_start,
                       n > 0 ? (const uint32_t *)sb.scan_tmp : (const uint32_t *)nullptr, 1,
                       sb.nbins, nb, sb.along_x, sb.max_sub, sb.sub_work, sb.sub_ofs + sb.nbins, sb.subs);
  }
  if (n > 0) {
    size_t lds = sizeof(uint16_t) * (size_t)kOneWaves * nbins;
    if (pr.fused) lds = std::max(lds + sizeof(uint32_t) * nbins, sizeof(SubLds<kOneThreads>));
    hipError_t e = set_lds(rec ? (const void *)chunk_scatter_kernel<true>
                               : (const void *)chunk_scatter_kernel<false>, lds);
    if (e != hipSuccess) return e;
    const int blocks = nch + (pr.fused ? 1 : 0);
    if (rec)
      hipLaunchKernelGGL(chunk_scatter_kernel<true>, dim3(blocks), dim3(kOneThreads), lds, s, pr);
    else
      hipLaunchKernelGGL(chunk_scatter_kernel<false>, dim3(blocks), dim3(kOneThreads), lds, s, pr);
  }
  return hipGetLastError();
}

hipError_t sort_points_batched(BinProblem *probs, int nprob, BinProblem *table, hipStream_t s) {
  if (nprob <= 0) return hipSuccess;
  uint32_t chunks = 0, scans = 0, pieces = 0;
  int max_bins = 1;
  for (int i = 0; i < nprob; ++i) {
    BinProblem &pr = probs[i];
    if (!tile_binning(pr.nbins) || pr.cls.ncls == 0 || pr.cls.ncls * pr.g.bin[0] > kClsKeys)
      return hipErrorInvalidValue;
    pr.chunk = tile_chunk(pr.pa.num_points);
    pr.nchunks = tile_chunks(pr.pa.num_points);
    pr.chunk0 = chunks;
    pr.scan0 = scans;
    pr.piece0 = pieces;
    pieces += (uint32_t)class_pieces(pr.pa.num_points, pr.nbins, pr.max_sub);
    chunks += (uint32_t)pr.nchunks;
    scans += (uint32_t)((pr.nbins + kScanDigits - 1) / kScanDigits);
    max_bins = std::max(max_bins, pr.nbins);
  }
  for (int first = 0; first < nprob; first += kBinTableChunk) {
    BinTableChunk chunk{};
    chunk.first = first;
    chunk.count = std::min(kBinTableChunk, nprob - first);
    for (int i = 0; i < chunk.count; ++i) chunk.probs[i] = probs[first + i];
    hipLaunchKernelGGL(bin_table_kernel, dim3(1), dim3(64), 0, s, chunk, table);
  }
  return launch_tile_binning(BinProblem{}, table, nprob, max_bins, chunks, scans, pieces, s);
}

hipError_t sort_points(const PointArgs &pa, const Geom &g, int dim, const SortBuffers &sb,
                       hipStream_t s, const RecordOut *rec) {
  const int64_t n = pa.num_points;
  if (sb.cls.ncls * g.bin[0] > kClsKeys) return hipErrorInvalidValue;
  if (rec && sb.cls.ncls > 0 && n > 0 && tile_binning(sb.nbins)) {
    BinProblem pr = bin_problem(pa, g, dim, sb, rec);
    const int nkeys = small_keys(g, sb.nbins, sb.cls.ncls);
    const size_t lds = small_lds(nkeys, sb.nbins);
    if (n <= kSmallPoints && lds <= kSmallLds) {
      hipError_t e = set_lds((const void *)small_binning_kernel, lds);
      if (e != hipSuccess) return e;
      const int fill = (int)std::min<int64_t>((pr.zero_n + 4 * kTileThreads - 1) / (4 * kTileThreads), 1024);
      hipLaunchKernelGGL(small_binning_kernel, dim3(1 + fill), dim3(kTileThreads), lds, s, pr);
      return hipGetLastError();
    }
    pr.chunk = tile_chunk(n);
    pr.nchunks = tile_chunks(n);
    // the totals of a single chunk are its counts
    uint32_t scans = (uint32_t)((sb.nbins + kScanDigits - 1) / kScanDigits);
    if (pr.nchunks == 1) pr.tot = pr.cnt, scans = 0;
    return launch_tile_binning(pr, nullptr, 1, sb.nbins, (uint32_t)pr.nchunks, scans,
                               (uint32_t)class_pieces(n, sb.nbins, sb.max_sub), s);
  }
  if (sb.zero_n > 0) {
    const hipError_t e = launch_fill(sb.zero, sb.zero_n, s);
    if (e != hipSuccess) return e;
  }
  if (sort_one_pass(sb.nbins)) return sort_points_one_pass(pa, g, dim, sb, s, rec);
  // with records, the last pass writes rec->out; earlier ones alternate with tmp
  auto dst = [&](int q) { return ((sb.passes - 1 - q) & 1) == 0 ? rec->out : rec->tmp; };
  if (n > 0) {
    hipLaunchKernelGGL(keys_kernel, dim3(sb.nchunks), dim3(kSortThreads), 0, s, pa, g, dim,
                       sb.keys[0], sb.cnt, sb.nchunks, sb.cls.ncls > 0 ? sb.cls.vmax : nullptr);
    for (int p = 0; p < sb.passes; ++p) {
      if (p > 0) {
        const KeySrc ks{sb.keys[p & 1], rec ? dst(p - 1).r : nullptr};
        hipLaunchKernelGGL(hist_kernel, dim3(sb.nchunks), dim3(kSortThreads), 0, s, ks, n,
                           p * kRadixBits, sb.cnt, sb.nchunks);
      }
      hipLaunchKernelGGL(scan_rows_kernel, dim3(kRadix), dim3(kScanThreads), 0, s, sb.cnt,
                         sb.nchunks, sb.scan_tmp);
      RecMove rm{};
      if (rec) {
        rm.out = dst(p);
        if (p > 0) rm.in = dst(p - 1);
        rm.values = rec->values;
        rm.pa = pa;
        rm.g = g;
        rm.first = p == 0;
        rm.last = p == sb.passes - 1;
        rm.vmax = p == 0 && rec->values && sb.cls.ncls > 0 ? sb.cls.vmax : nullptr;
        hipLaunchKernelGGL(scatter_kernel<true>, dim3(sb.nchunks), dim3(kSortThreads), 0, s,
                           sb.keys[0], (const uint32_t *)nullptr, sb.keys[1],
                           (uint32_t *)nullptr, n, p * kRadixBits, sb.cnt, sb.scan_tmp,
                           sb.nchunks, rm);
      } else {
        hipLaunchKernelGGL(scatter_kernel<false>, dim3(sb.nchunks), dim3(kSortThreads), 0, s,
                           sb.keys[p & 1], p == 0 ? (const uint32_t *)nullptr : sb.idx[p & 1],
                           sb.keys[(p + 1) & 1], sb.idx[(p + 1) & 1], n, p * kRadixBits, sb.cnt,
                           sb.scan_tmp, sb.nchunks, rm);
      }
    }
  }
  const KeySrc sorted{rec ? sb.keys[1] : sb.keys[sb.passes & 1], nullptr};
  int nb1 = sb.nbins + 1;
  const int3 nb = dim == 3 ? make_int3(g.nbin[0], g.nbin[1], g.nbin[2]) : make_int3(1, 1, 1);
  hipLaunchKernelGGL(bounds_kernel, dim3((nb1 + 255) / 256), dim3(256), 0, s, sorted, n,
                     sb.bin_start, sb.nbins);
  hipLaunchKernelGGL(subproblems_kernel, dim3(1), dim3(kSubThreads), 0, s, sb.bin_start,
                     (const uint32_t *)nullptr, 0, sb.nbins, nb, sb.along_x, sb.max_sub, sb.sub_work,
                     sb.sub_ofs + sb.nbins, sb.subs);
  if (n > 0 && rec && sb.cls.ncls > 0)
    hipLaunchKernelGGL(class_sort_kernel, dim3(class_pieces(n, sb.nbins, sb.max_sub)), dim3(kClsThreads),
                       0, s, bin_problem(pa, g, dim, sb, rec), (const BinProblem *)nullptr, 1);
  return hipGetLastError();
}

} // namespace anufft
