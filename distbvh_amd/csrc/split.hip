// split.hip -- the geom_axis / ml_geom_axis element splitters on gfx950.
//
// Replaces split_permutations and split_permutations_ml with split::mean and
// axis::longest (split/split.hpp:121-323, split/mean.hpp:47-81,
// split/axis.hpp:42-49) as set_entity_data_geom_axis / _ml_geom_axis call
// them (collision_object.hpp:133-162): a permutation of the elements (the
// reference order) and 2^depth - 1 split offsets, depth = log2(od).
//
// The reference recursion works range by range; here every range of one
// level is handled at once:
//  * ml_geom_axis: level l has 2^l ranges.  Per range: the union of its
//    element k-DOPs gives the longest axis; the mean of the centroid
//    projections on that axis is the split point; a two-pointer partition
//    (libstdc++ std::partition) moves the elements; fewer than two elements
//    give offset 0, an empty side gives size / 2.
//  * geom_axis: the reference takes the axis and the split point over all
//    elements at every level (its element span is never narrowed), so only
//    level 0 partitions; every deeper range is all on one side of that split
//    point and is split at its middle without moving anything.
//
// Exact split points.  The reference sums the projections in element order
// (std::accumulate; Kokkos::Serial parallel_reduce), and that rounded sum
// decides which side an element whose projection is close to the mean goes
// to.  Here the sum and the sum of magnitudes are accumulated in any order,
// which bounds both that sum and the reference's (recursive summation:
// |error| <= gamma(m) * sum |x|).  Every element whose projection lies outside
// the resulting interval is on a known side; only if some projection lies
// inside it is the sum recomputed as the reference rounds it
// (k_split_maps, k_split_exact).
//
// The two-pointer partition pairs, in order, the misplaced elements of the
// left part (those that fail the test, from the left) with the misplaced
// elements of the right part (those that pass, from the right) and swaps
// each pair.  With P the exclusive scan of the test bits, the k-th
// misplaced element from the left and from the right are found by rank, so
// a level is a scan and two scatter / gather passes.
#include "device.hpp"
#include "kernels.hpp"

namespace dbvh {

__constant__ double c_split_normals[kAxes][3] = {
    {1., 0., 0.}, {0., 1., 0.}, {0., 0., 1.},
    {DBVH_R3, DBVH_R3, DBVH_R3}, {DBVH_R3, -DBVH_R3, DBVH_R3},
    {DBVH_R3, DBVH_R3, -DBVH_R3}, {DBVH_R3, -DBVH_R3, -DBVH_R3},
    {DBVH_R2, DBVH_R2, 0.0}, {DBVH_R2, 0.0, DBVH_R2}, {0.0, DBVH_R2, DBVH_R2},
    {DBVH_R2, -DBVH_R2, 0.0}, {DBVH_R2, 0.0, -DBVH_R2}, {0.0, DBVH_R2, -DBVH_R2}};

// project(v, axis) with a run-time axis: the operations of project<A>
// (x * 1.0 is exactly x, the zero and +-R terms are the same products)
__device__ __forceinline__ double project_rt(const double* c, int a) {
  return c[0] * c_split_normals[a][0] + c[1] * c_split_normals[a][1] + c[2] * c_split_normals[a][2];
}

__device__ __forceinline__ void split_centroid(const SplitInput& si, uint32_t e, double* c) {
  if (si.cplanes) {
    c[0] = si.cplanes[e];
    c[1] = si.cplanes[si.n + e];
    c[2] = si.cplanes[2 * si.n + e];
  } else {
    c[0] = si.caos[3 * (uint64_t)e];
    c[1] = si.caos[3 * (uint64_t)e + 1];
    c[2] = si.caos[3 * (uint64_t)e + 2];
  }
}

// the range of position i: the last range whose begin is <= i (empty ranges
// come before the non-empty one with the same begin)
__device__ __forceinline__ uint32_t find_seg(const uint32_t* begin, uint32_t nseg, uint32_t i) {
  uint32_t lo = 0, hi = nseg;  // answer in [lo, hi)
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (begin[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// v of another lane of the wave: DPP control CTRL on the rows of ROWS (the
// other rows keep v), 64 bits
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned long long dpp_u64(unsigned long long v) {
  const int lo = (int)(uint32_t)v, hi = (int)(uint32_t)(v >> 32);
  const uint32_t l = (uint32_t)__builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xF, false);
  const uint32_t h = (uint32_t)__builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xF, false);
  return ((unsigned long long)h << 32) | l;
}

// Minimum / maximum over the wave (every lane active), the same in every
// lane: DPP within each row of 16 lanes (quad_perm [1,0,3,2], [2,3,0,1],
// row_ror 4, 8), then row_bcast 15 and 31 carry the rows' results to lane 63.
template <bool MAX>
__device__ __forceinline__ unsigned long long wave_reduce_u64(unsigned long long v) {
  auto op = [](unsigned long long x, unsigned long long y) { return MAX ? (y > x ? y : x) : (y < x ? y : x); };
  v = op(v, dpp_u64<0xB1, 0xF>(v));
  v = op(v, dpp_u64<0x4E, 0xF>(v));
  v = op(v, dpp_u64<0x124, 0xF>(v));
  v = op(v, dpp_u64<0x128, 0xF>(v));
  v = op(v, dpp_u64<0x142, 0xA>(v));
  v = op(v, dpp_u64<0x143, 0xC>(v));
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)v, 63);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(v >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// in-order index of range s of level l in the complete binary recursion of
// `depth` levels (the order in which the reference pushes the splits)
__device__ __forceinline__ uint32_t inorder(uint32_t l, uint32_t s, uint32_t depth) {
  return ((2u * s + 1u) << (depth - 1u - l)) - 1u;
}

// what a range's level accumulates into, before its first use: the empty
// k-DOP, zero sums, no undecided element
__device__ __forceinline__ void clear_range(const SplitBufs& sb, uint64_t s, uint32_t slab) {
  sb.seg_k64[s * kSlabs + slab] = (slab & 1) ? 0ull : ~0ull;
  if (slab < 2) sb.seg_acc[5 * s + slab] = 0.0;
  if (slab == 2) sb.seg_flag[s] = 0;
}

// level 0: one range of every element, in input order
__global__ __launch_bounds__(256) void k_split_start(SplitBufs sb, uint64_t n, uint64_t od) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) sb.rp[i] = (uint32_t)i;
  if (i < kSlabs) clear_range(sb, 0, (uint32_t)i);
  if (i == 0) {
    sb.seg[0] = 0;
    sb.seg[od] = (uint32_t)n;
  }
}

constexpr uint32_t kSplitItems = 2;  // positions per thread of the union and sum passes
constexpr uint32_t kSplitTile = 256 * kSplitItems;

// The wave's positions still to do (todo, range s each): the lanes of the
// first of them's range s0, which it takes off; false when there is none.
// Ranges of fewer than kSplitRunMin lanes are added to `alone`.
constexpr uint32_t kSplitRuns = 4;
constexpr uint32_t kSplitRunMin = 12;
__device__ __forceinline__ bool next_run(bool& todo, uint32_t s, uint32_t& s0, bool& mine, bool& alone) {
  const uint64_t m = __ballot(todo);
  if (m == 0) return false;
  s0 = __builtin_amdgcn_readlane(s, __ffsll((long long)m) - 1);
  mine = todo && s == s0;
  const bool few = (uint32_t)__popcll(__ballot(mine)) < kSplitRunMin;
  alone = alone || (mine && few);
  todo = todo && s != s0;
  mine = mine && !few;
  return true;
}

// Union of the element k-DOPs per range (ordered-u64 min / max).  A block
// takes kSplitTile consecutive positions: when they lie in one range, each
// thread folds its positions, the block folds its waves in LDS, and 26 lanes
// issue one atomic each.  (One set of 26 atomics per wave, one lane after
// the other, serialised on the range's 26 words: 162 us for 131,072 triangles
// per level, 15.5 us on average over the levels now.)
template <int KIND, int NV>
__global__ __launch_bounds__(256) void k_split_union(ElemInput in, SplitBufs sb, uint32_t nseg) {
  __shared__ unsigned long long part[256 / kWave][kSlabs];
  const uint64_t n = in.n, base = (uint64_t)blockIdx.x * kSplitTile;
  const uint32_t t = threadIdx.x;
  const uint64_t last = base + kSplitTile < n ? base + kSplitTile - 1 : n - 1;
  const uint32_t s0 = find_seg(sb.seg, nseg, (uint32_t)base), s1 = find_seg(sb.seg, nseg, (uint32_t)last);
  if (s0 == s1) {
    unsigned long long acc[kSlabs];
#pragma unroll
    for (int a = 0; a < kSlabs; ++a) acc[a] = (a & 1) ? 0ull : ~0ull;
#pragma unroll 1
    for (uint32_t j = 0; j < kSplitItems; ++j) {
      const uint64_t i = base + j * 256 + t;
      if (i >= n) break;
      double kd[kSlabs];
      element_kdop<KIND, NV>(in, sb.rp[i], kd);
#pragma unroll
      for (int a = 0; a < kSlabs; ++a) {
        const unsigned long long v = ordered_u64(kd[a]);
        acc[a] = (a & 1) ? (v > acc[a] ? v : acc[a]) : (v < acc[a] ? v : acc[a]);
      }
    }
#pragma unroll
    for (int a = 0; a < kSlabs; ++a) {
      const unsigned long long r = (a & 1) ? wave_reduce_u64<true>(acc[a]) : wave_reduce_u64<false>(acc[a]);
      if (lane_id() == (uint32_t)a) part[t / kWave][a] = r;
    }
    __syncthreads();
    if (t < kSlabs) {
      unsigned long long r = part[0][t];
      for (uint32_t w = 1; w < 256 / kWave; ++w) {
        const unsigned long long v = part[w][t];
        r = (t & 1) ? (v > r ? v : r) : (v < r ? v : r);
      }
      unsigned long long* d = sb.seg_k64 + (uint64_t)s0 * kSlabs + t;
      if (t & 1) atomicMax(d, r);
      else atomicMin(d, r);
    }
    return;
  }
  // Several ranges: each wave folds the long runs of one range among its 64
  // positions (at most kSplitRuns of them) and issues one set of atomics per
  // run; the elements of short runs issue their own (few to a range).
#pragma unroll 1
  for (uint32_t j = 0; j < kSplitItems; ++j) {
    const uint64_t i = base + j * 256 + t;
    const bool act = i < n;
    const uint32_t s = act ? find_seg(sb.seg, nseg, (uint32_t)i) : kEnd;
    unsigned long long v[kSlabs];
    if (act) {
      double kd[kSlabs];
      element_kdop<KIND, NV>(in, sb.rp[i], kd);
#pragma unroll
      for (int a = 0; a < kSlabs; ++a) v[a] = ordered_u64(kd[a]);
    }
    bool todo = act, alone = false, mine;
    uint32_t sr;
    for (uint32_t r = 0; r < kSplitRuns && next_run(todo, s, sr, mine, alone); ++r) {
      if (__ballot(mine) == 0) continue;
      unsigned long long mx = 0;
#pragma unroll
      for (int a = 0; a < kSlabs; ++a) {
        const unsigned long long f = (a & 1) ? wave_reduce_u64<true>(mine ? v[a] : 0ull) : wave_reduce_u64<false>(mine ? v[a] : ~0ull);
        if (lane_id() == (uint32_t)a) mx = f;
      }
      if (lane_id() < kSlabs) {
        unsigned long long* d = sb.seg_k64 + (uint64_t)sr * kSlabs + lane_id();
        if (lane_id() & 1) atomicMax(d, mx);
        else atomicMin(d, mx);
      }
    }
    if (todo || alone) {
      unsigned long long* d = sb.seg_k64 + (uint64_t)s * kSlabs;
#pragma unroll
      for (int a = 0; a < kSlabs; ++a) {
        if (a & 1) atomicMax(d + a, v[a]);
        else atomicMin(d + a, v[a]);
      }
    }
  }
}

// axis::longest of a range's union: the first maximum slab width
// (kdop.hpp:354-362, std::max_element with length() <)
__device__ __forceinline__ int longest_axis(const SplitBufs& sb, uint32_t s) {
  const unsigned long long* k = sb.seg_k64 + (uint64_t)s * kSlabs;
  int best = 0;
  double bl = from_ordered_u64(k[1]) - from_ordered_u64(k[0]);
  for (int a = 1; a < kAxes; ++a) {
    const double l = from_ordered_u64(k[2 * a + 1]) - from_ordered_u64(k[2 * a]);
    if (bl < l) {
      best = a;
      bl = l;
    }
  }
  return best;
}

// sum and sum of magnitudes of the centroid projections per range (any
// order: a block whose positions lie in one range adds once), and the
// range's axis, written where the range begins
__global__ __launch_bounds__(256) void k_split_sum(SplitInput si, SplitBufs sb, uint32_t nseg) {
  __shared__ double part[2][256 / kWave];
  const uint64_t n = si.n, base = (uint64_t)blockIdx.x * kSplitTile;
  const uint32_t t = threadIdx.x;
  const uint64_t last = base + kSplitTile < n ? base + kSplitTile - 1 : n - 1;
  const uint32_t s0 = find_seg(sb.seg, nseg, (uint32_t)base), s1 = find_seg(sb.seg, nseg, (uint32_t)last);
  const bool one = s0 == s1;
  const int axis0 = longest_axis(sb, s0);
  double sum = 0.0, mag = 0.0;
#pragma unroll
  for (uint32_t j = 0; j < kSplitItems; ++j) {
    const uint64_t i = base + j * 256 + t;
    const bool act = i < n;
    uint32_t s = s0;
    double x = 0.0;
    if (act) {
      if (!one) s = find_seg(sb.seg, nseg, (uint32_t)i);
      const int axis = s == s0 ? axis0 : longest_axis(sb, s);
      if (sb.seg[s] == (uint32_t)i) sb.seg_axis[s] = axis;
      double c[3];
      split_centroid(si, sb.rp[i], c);
      x = project_rt(c, axis);
    }
    if (one) {
      sum += x;
      mag += __builtin_fabs(x);
    } else {
      bool todo = act, alone = false, mine;
      uint32_t sr;
      for (uint32_t r = 0; r < kSplitRuns && next_run(todo, s, sr, mine, alone); ++r) {
        if (__ballot(mine) == 0) continue;
        const double fs = wave_sum(mine ? x : 0.0), fm = wave_sum(mine ? __builtin_fabs(x) : 0.0);
        if (lane_id() == 0) {
          atomicAdd(sb.seg_acc + 5 * (uint64_t)sr, fs);
          atomicAdd(sb.seg_acc + 5 * (uint64_t)sr + 1, fm);
        }
      }
      if (todo || alone) {
        atomicAdd(sb.seg_acc + 5 * (uint64_t)s, x);
        atomicAdd(sb.seg_acc + 5 * (uint64_t)s + 1, __builtin_fabs(x));
      }
    }
  }
  if (!one) return;
  sum = wave_sum(sum);
  mag = wave_sum(mag);
  if (lane_id() == 0) {
    part[0][t / kWave] = sum;
    part[1][t / kWave] = mag;
  }
  __syncthreads();
  if (t < 2) atomicAdd(sb.seg_acc + 5 * (uint64_t)s0 + t, (part[t][0] + part[t][1]) + (part[t][2] + part[t][3]));
}

// an interval [lo, hi] that contains the reference's split point sum / m of a
// range, whatever order the sum was rounded in
__device__ __forceinline__ void split_interval(const SplitBufs& sb, uint32_t s, uint64_t od, double& lo, double& hi) {
  const double m = (double)(sb.seg[od + s] - sb.seg[s]);
  const double u = 0x1p-53;
  const double S = sb.seg_acc[5 * (uint64_t)s], A = sb.seg_acc[5 * (uint64_t)s + 1];
  // gamma(m) = m u / (1 - m u) bounds recursive summation in any order; once
  // for the reference's order, once for the order used here
  const double g = m * u / (1.0 - m * u);
  const double E = 2.0 * g * A;
  const double W = (__builtin_fabs(S) + E) / m;
  const double slack = 8.0 * u * W + 0x1p-1000;  // rounding of these lines and of the division
  lo = S / m - E / m - slack;
  hi = S / m + E / m + slack;
}

// Per position its projection (xbuf, range order) and its test bit: 1 below
// the interval, 0 above, 2 undecided (and the range flagged for the exact
// split point).  A wave takes one kExactBlock of positions; when they lie in
// one range, it leaves their sums for k_split_maps.  Also clears the words of
// the scan that follows.
__global__ __launch_bounds__(256) void k_split_pred(SplitInput si, SplitBufs sb, uint32_t nseg, uint64_t od,
                                                    uint64_t scan_words) {
  const uint64_t n = si.n, gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (uint64_t k = gid; k < scan_words; k += (uint64_t)gridDim.x * blockDim.x) ((uint32_t*)sb.scan_lb)[k] = 0;
  if (gid == 0) {
    *sb.scan_ctr = 0;
    sb.scan[n] = 0;
  }
  const uint64_t blk = gid / kWave, base = blk * kExactBlock;
  if (base >= n) return;  // uniform per wave
  const uint64_t last = base + kExactBlock < n ? base + kExactBlock - 1 : n - 1;
  const uint32_t s0 = find_seg(sb.seg, nseg, (uint32_t)base), s1 = find_seg(sb.seg, nseg, (uint32_t)last);
  const bool one = s0 == s1;
  double lo0, hi0;
  split_interval(sb, s0, od, lo0, hi0);
  const int axis0 = sb.seg_axis[s0];
  double sum = 0.0, mag = 0.0;
  bool open = false;
#pragma unroll
  for (uint32_t j = 0; j < kExactBlock / kWave; ++j) {
    const uint64_t i = base + j * kWave + lane_id();
    if (i >= n) break;
    double lo = lo0, hi = hi0;
    int axis = axis0;
    uint32_t s = s0;
    if (!one) {
      s = find_seg(sb.seg, nseg, (uint32_t)i);
      split_interval(sb, s, od, lo, hi);
      axis = sb.seg_axis[s];
    }
    double c[3];
    split_centroid(si, sb.rp[i], c);
    const double x = project_rt(c, axis);
    uint32_t p;
    if (x < lo) p = 1;
    else if (x > hi) p = 0;
    else p = 2;  // also NaN x, lo or hi
    sb.scan[i] = p;
    sb.xbuf[i] = x;
    if (p == 2 && !one) atomicOr(sb.seg_flag + s, 1u);
    open = open | (p == 2);
    sum += x;
    mag += __builtin_fabs(x);
  }
  if (one) {
    if (__ballot(open) != 0 && lane_id() == 0) atomicOr(sb.seg_flag + s0, 1u);
    sum = wave_sum(sum);
    mag = wave_sum(mag);
    if (lane_id() == 0) {
      sb.blk[blk].sum = sum;
      sb.blk[blk].mag = mag;
    }
  }
}

// The reference's split point of a flagged range is s / m with s the sum
// rounded after every element, fl(... fl(fl(0 + x0) + x1) ...): a serial chain
// of fp64 adds.  But while s stays in one binade [2^E, 2^(E+1))
// every sum is a multiple of u = 2^(E-52), and fl(s + x) = s + rint(x / u) u
// unless x / u lies halfway between two integers, where the rule (ties to
// even) depends on the parity of s / u alone.  So the effect of a run of
// elements is a map from that parity to an integer, such maps compose
// associatively, and runs are evaluated in parallel, exactly.
//
// k_split_maps: a wave per kExactBlock of positions (those that lie in one
// flagged range).  The approximate sum before the block and the block's sums
// of positive and negative elements bound every partial sum in it, margin
// included; if those bounds lie strictly in one binade the wave leaves the
// block's map there, else the block is left for serial adds (the blocks in
// which the sum crosses a power of two or zero).  Negative sums mirror.
__device__ __forceinline__ void map_then(long long& a0, long long& a1, long long b0, long long b1) {
  a0 += (a0 & 1) ? b1 : b0;
  a1 += ((a1 + 1) & 1) ? b1 : b0;
}

__global__ __launch_bounds__(256) void k_split_maps(SplitBufs sb, uint64_t n, uint32_t nseg, uint64_t od) {
  const uint64_t blk = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave, base = blk * kExactBlock;
  if (base + kExactBlock > n) return;  // uniform per wave, as every branch below
  const uint32_t s = find_seg(sb.seg, nseg, (uint32_t)base);
  const uint32_t b = sb.seg[s], e = sb.seg[od + s];
  if (sb.seg_flag[s] == 0 || base + kExactBlock > e) return;
  const uint32_t lane = lane_id();
  // the sum before the block: the range's head up to its first whole block,
  // then whole blocks
  const uint64_t j0 = (b + kExactBlock - 1) / kExactBlock;
  double P = 0.0;
  for (uint64_t i = b + lane; i < j0 * kExactBlock; i += kWave) P += sb.xbuf[i];
  for (uint64_t j = j0 + lane; j < blk; j += kWave) P += sb.blk[j].sum;
  P = wave_sum(P);
  const double A = sb.seg_acc[5 * (uint64_t)s + 1], sum = sb.blk[blk].sum, mag = sb.blk[blk].mag;
  const double m = (double)(e - b);
  // rounding of the reference's partial sums and of these (each within
  // gamma(m) A of the exact ones), with room to spare
  const double M = 4.0 * m * 0x1p-53 * A;
  const double lo = P - (0.5 * (mag - sum) * (1.0 + 0x1p-30) + M), hi = P + (0.5 * (mag + sum) * (1.0 + 0x1p-30) + M);
  int E = kExactNone, neg = 0;
  if (lo > 0.0 && hi < 0x1p900 && lo > 0x1p-900) {
    const int el = ilogb(lo);
    if (el == ilogb(hi)) E = el;
  } else if (hi < 0.0 && lo > -0x1p900 && hi < -0x1p-900) {
    const int el = ilogb(lo);
    if (el == ilogb(hi)) E = el;
    neg = 1;
  }
  if (E != kExactNone) {
    constexpr uint32_t kPer = kExactBlock / kWave;
    long long a0 = 0, a1 = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
      const double x = sb.xbuf[base + lane * kPer + k];
      const double y = __builtin_ldexp(neg ? -x : x, 52 - E);
      const double r = __builtin_rint(y);
      const double f = y - r;  // exact
      const long long d0 = (long long)r;
      const long long d1 = __builtin_fabs(f) == 0.5 ? d0 + (f > 0.0 ? 1 : -1) : d0;
      map_then(a0, a1, d0, d1);
    }
    for (int o = 1; o < kWave; o <<= 1) {
      const long long b0 = __shfl_down(a0, o, kWave), b1 = __shfl_down(a1, o, kWave);
      map_then(a0, a1, b0, b1);  // (lane 0 folds the lanes in order; the others' values are not used)
    }
    if (lane == 0) {
      sb.blk[blk].d0 = a0;
      sb.blk[blk].d1 = a1;
    }
  }
  if (lane == 0) sb.blk[blk].key = E == kExactNone ? kExactNone : 2 * E + neg;
}

// The exact split points of the flagged ranges, one wave per range: whole
// blocks of one binade by their maps, 64 blocks at a time, the others (the
// range's head and tail, and the blocks left open) by lane 0's serial adds from
// LDS.  131,072 elements took about 800 us as one
// serial chain, 40 to 55 us so (and 5 us for k_split_maps).
__global__ __launch_bounds__(64) void k_split_exact(SplitBufs sb, uint32_t nseg, uint64_t od) {
  __shared__ double buf[kExactBlock];
  const uint32_t s = blockIdx.x;
  if (s >= nseg || sb.seg_flag[s] == 0) return;
  const uint64_t b = sb.seg[s], e = sb.seg[od + s];
  const uint32_t lane = threadIdx.x;
  double S = 0.0;
  auto serial = [&](uint64_t from, uint64_t to) {
    for (uint64_t at = from; at < to; at += kExactBlock) {
      const uint32_t cnt = (uint32_t)(to - at < kExactBlock ? to - at : kExactBlock);
#pragma unroll
      for (uint32_t k = 0; k < kExactBlock / kWave; ++k) {
        const uint32_t j = k * kWave + lane;
        if (j < cnt) buf[j] = sb.xbuf[at + j];
      }
      __syncthreads();
      if (lane == 0) S = ordered_sum(buf, cnt, S);
      S = __shfl(S, 0, kWave);
      __syncthreads();
    }
  };
  const uint64_t j0 = (b + kExactBlock - 1) / kExactBlock, j1 = e / kExactBlock;
  if (j0 >= j1) {
    serial(b, e);
  } else {
    serial(b, j0 * kExactBlock);
    for (uint64_t j = j0; j < j1; j += kWave) {
      const uint32_t cnt = (uint32_t)(j1 - j < kWave ? j1 - j : kWave);
      const bool in = lane < cnt;
      const int32_t key = in ? sb.blk[j + lane].key : kExactNone;
      const long long d0 = in && key != kExactNone ? sb.blk[j + lane].d0 : 0;
      const long long d1 = in && key != kExactNone ? sb.blk[j + lane].d1 : 0;
      for (uint32_t k = 0; k < cnt;) {
        const int32_t kk = __builtin_amdgcn_readlane(key, k);
        bool done = false;
        if (kk != kExactNone) {
          // the run of blocks from k on in this binade
          const uint64_t other = __ballot(key != kk || !in) >> k;
          const uint32_t run = other ? (uint32_t)__builtin_ctzll(other) : kWave - k;
          const bool mine = lane >= k && lane < k + run;
          long long a0 = mine ? d0 : 0, a1 = mine ? d1 : 0;  // (0, 0): the identity
          for (int o = 1; o < kWave; o <<= 1) {
            const long long b0 = __shfl_down(a0, o, kWave), b1 = __shfl_down(a1, o, kWave);
            map_then(a0, a1, b0, b1);
          }
          a0 = __shfl(a0, 0, kWave);
          a1 = __shfl(a1, 0, kWave);
          const int neg = kk & 1, E = (kk - neg) / 2;
          const double y = __builtin_ldexp(neg ? -S : S, 52 - E);
          if (y >= 0x1p52 && y < 0x1p53) {  // (as the bounds promise)
            const long long N = (long long)y;
            const long long N2 = N + ((N & 1) ? a1 : a0);
            if (N2 >= (1ll << 52) && N2 <= (1ll << 53)) {
              S = __builtin_ldexp((double)N2, E - 52);
              S = neg ? -S : S;
              k += run;
              done = true;
            }
          }
        }
        if (!done) {
          serial((j + k) * kExactBlock, (j + k + 1) * kExactBlock);
          ++k;
        }
      }
    }
    serial(j1 * kExactBlock, e);
  }
  if (lane == 0) sb.seg_acc[5 * (uint64_t)s + 4] = S / (double)(e - b);
}

// the undecided elements against the exact split points
__global__ __launch_bounds__(256) void k_split_fix(SplitBufs sb, uint64_t n, uint32_t nseg) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || sb.scan[i] != 2) return;
  const uint32_t s = find_seg(sb.seg, nseg, (uint32_t)i);
  sb.scan[i] = sb.xbuf[i] < sb.seg_acc[5 * (uint64_t)s + 4] ? 1u : 0u;
}

// range s of this level: its bounds, and the partition point L if it moves
// (else kEnd); m / 2 splits a range whose elements all lie on one side
struct SplitRange {
  uint32_t b, e, L, split;
};
__device__ __forceinline__ SplitRange split_range(const SplitBufs& sb, uint32_t s, uint64_t od, int ml) {
  SplitRange r;
  r.b = sb.seg[s];
  r.e = sb.seg[od + s];
  const uint32_t m = r.e - r.b, L = sb.scan[r.e] - sb.scan[r.b];
  const bool part = !(ml && m < 2);
  r.split = r.b + (part ? ((L == 0 || L == m) ? m / 2 : L) : 0u);
  r.L = (part && L > 0 && L < m) ? L : kEnd;
  return r;
}

// The two-pointer swaps by rank: the k-th failing element left of the
// partition point and the k-th passing element right of it (counted from the
// right end) trade places.  Also, per range, its split offset (in the
// reference's push order) and the next level's two ranges, cleared.
__global__ __launch_bounds__(256) void k_split_scatter(SplitBufs sb, uint64_t n, uint32_t nseg, uint64_t od,
                                                       uint32_t level, uint32_t depth, int ml, uint32_t* splits) {
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t s = gid; s < nseg; s += stride) {
    const SplitRange r = split_range(sb, (uint32_t)s, od, ml);
    splits[inorder(level, (uint32_t)s, depth)] = r.split;
    sb.seg_next[2 * s] = r.b;
    sb.seg_next[od + 2 * s] = r.split;
    sb.seg_next[2 * s + 1] = r.split;
    sb.seg_next[od + 2 * s + 1] = r.e;
  }
  if (level + 1 < depth)
    for (uint64_t k = gid; k < 2ull * nseg * kSlabs; k += stride)
      clear_range(sb, k / kSlabs, (uint32_t)(k % kSlabs));
  if (gid >= n) return;
  const uint32_t i = (uint32_t)gid, s = find_seg(sb.seg, nseg, i);
  const SplitRange r = split_range(sb, s, od, ml);
  if (r.L == kEnd) return;
  const uint32_t* P = sb.scan;
  const uint32_t pv = P[i + 1] - P[i];
  if (i < r.b + r.L && pv == 0) {
    const uint32_t k = (i - r.b) - (P[i] - P[r.b]);
    sb.tmpf[r.b + k] = sb.rp[i];
  } else if (i >= r.b + r.L && pv == 1) {
    const uint32_t k = P[r.e] - P[i + 1];
    sb.tmpt[r.b + k] = sb.rp[i];
  }
}

__global__ __launch_bounds__(256) void k_split_gather(SplitBufs sb, uint64_t n, uint32_t nseg, uint64_t od, int ml) {
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= n) return;
  const uint32_t i = (uint32_t)gid;
  const SplitRange r = split_range(sb, find_seg(sb.seg, nseg, i), od, ml);
  uint32_t v = sb.rp[i];
  if (r.L != kEnd) {
    const uint32_t* P = sb.scan;
    const uint32_t pv = P[i + 1] - P[i];
    if (i < r.b + r.L && pv == 0) v = sb.tmpt[r.b + (i - r.b) - (P[i] - P[r.b])];
    else if (i >= r.b + r.L && pv == 1) v = sb.tmpf[r.b + P[r.e] - P[i + 1]];
  }
  sb.rp_b[i] = v;
}

// geom_axis below level 0: every range is split at its middle (one thread;
// at most od - 1 splits)
__global__ void k_split_midpoints(SplitBufs sb, uint64_t od, uint32_t depth, uint32_t* splits) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  uint32_t* cur = sb.seg;
  uint32_t* nxt = sb.seg_next;
  for (uint32_t l = 1; l < depth; ++l) {
    const uint32_t nseg = 1u << l;
    for (uint32_t s = 0; s < nseg; ++s) {
      const uint32_t b = cur[s], e = cur[od + s];
      const uint32_t sp = b + (e - b) / 2;
      splits[inorder(l, s, depth)] = sp;
      nxt[2 * s] = b;
      nxt[od + 2 * s] = sp;
      nxt[2 * s + 1] = sp;
      nxt[od + 2 * s + 1] = e;
    }
    uint32_t* t = cur;
    cur = nxt;
    nxt = t;
  }
}

// patch of every input element: the number of split offsets <= its position
__global__ __launch_bounds__(256) void k_split_patch_key(SplitBufs sb, uint64_t n, const uint32_t* splits,
                                                         uint32_t nsplits, uint32_t* patch_key) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t lo = 0, hi = nsplits;  // count of splits <= i
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (splits[mid] <= (uint32_t)i) lo = mid + 1;
    else hi = mid;
  }
  patch_key[sb.rp[i]] = lo;
}

// keys[i] = src[idx[i]]
template <typename T>
__global__ __launch_bounds__(256) void k_gather_by(const T* __restrict__ src, const uint32_t* __restrict__ idx, uint64_t n,
                                                   T* __restrict__ dst) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[idx[i]];
}

template <typename T>
hipError_t launch_gather_by(const T* src, const uint32_t* idx, uint64_t n, T* dst, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_by<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, idx, n, dst);
  return hipGetLastError();
}
template hipError_t launch_gather_by<uint32_t>(const uint32_t*, const uint32_t*, uint64_t, uint32_t*, hipStream_t);
template hipError_t launch_gather_by<uint64_t>(const uint64_t*, const uint32_t*, uint64_t, uint64_t*, hipStream_t);

// Patches given by the caller: patch k holds input indices [given[k-1],
// given[k]) (given[-1] = 0, given[od-1] = n); the reference order is the
// input order.  given: od - 1 non-decreasing offsets (device).
hipError_t launch_given_split(SplitBufs sb, uint64_t n, uint64_t od, const uint32_t* given, uint32_t* splits,
                              uint32_t* patch_key, uint32_t** result, hipStream_t s) {
  *result = sb.rp;
  if (n == 0) return hipSuccess;
  hipError_t e = launch_iota_u32(sb.rp, n, s);
  if (e != hipSuccess) return e;
  if (od > 1) {
    e = launch_copy<uint32_t>(splits, given, od - 1, s);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_split_patch_key, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, sb, n, splits,
                     (uint32_t)(od - 1), patch_key);
  return hipGetLastError();
}

template <int KIND, int NV>
static void union_launch(unsigned g, const ElemInput& in, const SplitBufs& sb, uint32_t nseg, hipStream_t s) {
  hipLaunchKernelGGL((k_split_union<KIND, NV>), dim3(g), dim3(256), 0, s, in, sb, nseg);
}

static hipError_t launch_union(const ElemInput& in, const SplitBufs& sb, uint32_t nseg, hipStream_t s) {
  const unsigned g = (unsigned)((in.n + kSplitTile - 1) / kSplitTile);
  if (in.kind == kSphere) {
    union_launch<kSphere, 1>(g, in, sb, nseg, s);
  } else if (in.kind == kSnapshot) {
    union_launch<kSnapshot, 1>(g, in, sb, nseg, s);
  } else {
    switch (in.nv) {
      case 1: union_launch<kPoly, 1>(g, in, sb, nseg, s); break;
      case 2: union_launch<kPoly, 2>(g, in, sb, nseg, s); break;
      case 3: union_launch<kPoly, 3>(g, in, sb, nseg, s); break;
      case 4: union_launch<kPoly, 4>(g, in, sb, nseg, s); break;
      case 5: union_launch<kPoly, 5>(g, in, sb, nseg, s); break;
      case 6: union_launch<kPoly, 6>(g, in, sb, nseg, s); break;
      case 7: union_launch<kPoly, 7>(g, in, sb, nseg, s); break;
      case 8: union_launch<kPoly, 8>(g, in, sb, nseg, s); break;
      default: return hipErrorInvalidValue;
    }
  }
  return hipGetLastError();
}

hipError_t launch_split(const ElemInput& in, const SplitInput& si, SplitBufs sb, uint64_t od, int ml,
                        uint32_t* splits, uint32_t* patch_key, uint32_t** result, hipStream_t s) {
  const uint64_t n = si.n;
  *result = sb.rp;
  if (n == 0) return hipSuccess;
  if (od < 2) {
    hipError_t e = launch_iota_u32(sb.rp, n, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_split_patch_key, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, sb, n, splits, 0u,
                       patch_key);
    return hipGetLastError();
  }
  if ((od & (od - 1)) != 0 || n >= (1ull << 30) || in.n != n) return hipErrorInvalidValue;
  if (!si.cplanes && !si.caos) return hipErrorInvalidValue;
  uint32_t depth = 0;
  while ((1ull << (depth + 1)) <= od) ++depth;
  const unsigned g = (unsigned)((n + 255) / 256);
  const unsigned gt = (unsigned)((n + kSplitTile - 1) / kSplitTile);
  const uint64_t nblk = split_blocks(n);
  const unsigned gw = (unsigned)((nblk * kWave + 255) / 256);  // one wave per block of positions
  hipLaunchKernelGGL(k_split_start, dim3(g), dim3(256), 0, s, sb, n, od);
  const uint32_t levels = ml ? depth : 1u;
  for (uint32_t l = 0; l < levels; ++l) {
    const uint32_t nseg = 1u << l;
    hipError_t e = launch_union(in, sb, nseg, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_split_sum, dim3(gt), dim3(256), 0, s, si, sb, nseg);
    hipLaunchKernelGGL(k_split_pred, dim3(gw), dim3(256), 0, s, si, sb, nseg, od, 2 * sort_tiles(n + 1));
    hipLaunchKernelGGL(k_split_maps, dim3(gw), dim3(256), 0, s, sb, n, nseg, od);
    hipLaunchKernelGGL(k_split_exact, dim3(nseg), dim3(64), 0, s, sb, nseg, od);
    hipLaunchKernelGGL(k_split_fix, dim3(g), dim3(256), 0, s, sb, n, nseg);
    e = launch_scan_u32(sb.scan, n + 1, sb.scan_lb, sb.scan_ctr, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_split_scatter, dim3(g), dim3(256), 0, s, sb, n, nseg, od, l, depth, ml, splits);
    hipLaunchKernelGGL(k_split_gather, dim3(g), dim3(256), 0, s, sb, n, nseg, od, ml);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    uint32_t* t = sb.rp;
    sb.rp = sb.rp_b;
    sb.rp_b = t;
    t = sb.seg;
    sb.seg = sb.seg_next;
    sb.seg_next = t;
  }
  if (!ml) hipLaunchKernelGGL(k_split_midpoints, dim3(1), dim3(64), 0, s, sb, od, depth, splits);
  hipLaunchKernelGGL(k_split_patch_key, dim3(g), dim3(256), 0, s, sb, n, splits, (uint32_t)(od - 1), patch_key);
  *result = sb.rp;
  return hipGetLastError();
}

}  // namespace dbvh
