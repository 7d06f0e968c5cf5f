// sweep.hip -- sort-and-sweep between the elements of two patches.
//
// Replaces sort_and_sweep_local and max_variant_axis (narrowphase/kokkos.hpp:
// 119-248).  The axis with the largest variance of the two patches'
// centroids; then B's slab minima on that axis, scaled to [0, UINT32_MAX]
// over the union of the two patches' slabs and truncated, are sorted (stable
// LSD radix sort); every element a of A visits the sorted B from the start,
// skips b while b's scaled maximum (fp64) lies below a's truncated minimum,
// stops at the first b whose truncated minimum exceeds a's truncated maximum,
// and reports (a, b) when the two 26-DOPs overlap.
//
// The stop is the first sorted position whose minimum exceeds a's maximum,
// i.e. an upper bound, searched 64 ways by the wave that sweeps a.  The range
// before it is walked in tiles of 64 positions, in order, so each a's pairs
// come out in B's sorted order, as the reference's callback sees them; a tile
// whose largest scaled maximum lies below a's minimum holds only skipped b, and
// one ballot finds the others among 64 tiles (of 8,192 x 8,192 sheet elements
// six are left where 64 of the 128 were walked: 73 + 70 us for the two passes
// instead of 120 + 102).  What a walked tile costs is its reads: the sorted k-DOPs
// are planes, and x, y, z are tested first (35 + 34 us).  A count pass
// and a write pass at per-a offsets (exclusive scan) make the output order
// (a ascending, then sorted b) independent of scheduling.
#include "device.hpp"
#include "kernels.hpp"

namespace dbvh {

namespace {
constexpr int kMomentBlock = 256;
constexpr uint32_t kMomentBlocks = 256;
}  // namespace

// Per-block sums of (x, y, z, x^2, y^2, z^2) over A's centroids then B's
// (the concatenation of kokkos.hpp:127-136), in a fixed order: a thread sums
// its strided elements, the block folds its threads pairwise.
__global__ __launch_bounds__(kMomentBlock) void k_moments(const double* __restrict__ ca, uint64_t na,
                                                          const double* __restrict__ cb, uint64_t nb,
                                                          double* __restrict__ part) {
  __shared__ double s[6][kMomentBlock];
  const uint64_t n = na + nb;
  double acc[6] = {0, 0, 0, 0, 0, 0};
  for (uint64_t i = (uint64_t)blockIdx.x * kMomentBlock + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * kMomentBlock) {
    const double* c = i < na ? ca + 3 * i : cb + 3 * (i - na);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double x = c[j];
      acc[j] = acc[j] + x;
      acc[3 + j] = acc[3 + j] + x * x;
    }
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) s[k][threadIdx.x] = acc[k];
  __syncthreads();
  for (int h = kMomentBlock / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h)
#pragma unroll
      for (int k = 0; k < 6; ++k) s[k][threadIdx.x] = s[k][threadIdx.x] + s[k][threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x < 6) part[(uint64_t)blockIdx.x * 6 + threadIdx.x] = s[threadIdx.x][0];
}

// The block sums folded in block order, then var = s2 - s * s / n per axis
// and the first axis of largest variance (kokkos.hpp:144-158).
__global__ __launch_bounds__(256) void k_variant_axis(const double* __restrict__ part, uint32_t nblocks, uint64_t n,
                                                      int32_t* __restrict__ axis) {
  // the partials through LDS, then a lane per sum, in block order (one thread
  // that loaded as it added took 15 us)
  __shared__ double sp[kMomentBlocks * 6];
  __shared__ double s[6];
  for (uint32_t i = threadIdx.x; i < nblocks * 6; i += 256) sp[i] = part[i];
  __syncthreads();
  if (threadIdx.x < 6) {
    double x = 0;
#pragma unroll 8
    for (uint32_t b = 0; b < nblocks; ++b) x = x + sp[b * 6 + threadIdx.x];
    s[threadIdx.x] = x;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double var[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) var[i] = s[3 + i] - s[i] * s[i] / (double)n;
  int ax = 0;
  if (var[1] > var[0]) ax = 1;
  if (var[2] > var[ax]) ax = 2;
  *axis = ax;
}

// B's truncated minima on the axis and the identity payload (kokkos.hpp:
// 183-193); the casts are the reference's double -> uint32 conversions.
__global__ __launch_bounds__(256) void k_sweep_quantize(const double* __restrict__ kb, uint64_t nb, int axis,
                                                        double gmin, double conv, uint32_t* __restrict__ bq,
                                                        uint32_t* __restrict__ bidx) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nb) return;
  bq[i] = (uint32_t)float_to_uint((kb[i * 26 + 2 * axis] - gmin) * conv);
  bidx[i] = (uint32_t)i;
}

// B's k-DOPs in sorted order, as 26 planes, and their scaled maxima; and the
// largest scaled maximum of every 64 sorted positions.  A block per 64: its
// rows come in through LDS and leave as plane segments, so that both sides are
// whole lines.
__global__ __launch_bounds__(256) void k_sweep_gather(const double* __restrict__ kb, const uint32_t* __restrict__ bidx,
                                                      uint64_t nb, int axis, double gmin, double conv,
                                                      double* __restrict__ kbs, double* __restrict__ bmax,
                                                      double* __restrict__ tmax) {
  __shared__ double s[64][kSlabs + 1];
  const uint64_t j0 = (uint64_t)blockIdx.x * 64;
  const uint32_t cnt = nb - j0 < 64 ? (uint32_t)(nb - j0) : 64u;
  for (uint32_t t = threadIdx.x; t < cnt * kSlabs; t += 256) {
    const uint32_t j = t / kSlabs, k = t - j * kSlabs;
    s[j][k] = kb[(uint64_t)bidx[j0 + j] * kSlabs + k];
  }
  __syncthreads();
  const uint32_t j = threadIdx.x & 63;
  if (j < cnt)
    for (uint32_t k = threadIdx.x >> 6; k < kSlabs; k += 4) kbs[(uint64_t)k * nb + j0 + j] = s[j][k];
  if (threadIdx.x < 64) {
    double v = -__builtin_inf();
    if (j < cnt) {
      v = (s[j][2 * axis + 1] - gmin) * conv;
      bmax[j0 + j] = v;
    }
    if (!(v == v)) v = __builtin_inf();  // a NaN is below nothing: its tile is walked
    for (int o = 32; o > 0; o >>= 1) {
      const double x = __shfl_xor(v, o, 64);
      v = x > v ? x : v;
    }
    if (j == 0) tmax[blockIdx.x] = v;
  }
}

// The 64-bit sum of the counts: one addition a block, where one a wave of the
// sweep queued for the word.
__global__ __launch_bounds__(256) void k_sweep_total(const uint32_t* __restrict__ count, uint64_t na,
                                                     unsigned long long* __restrict__ total) {
  __shared__ unsigned long long s[4];
  unsigned long long c = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < na; i += (uint64_t)gridDim.x * 256) c += count[i];
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if (lane_id() == 0) s[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    c = s[0] + s[1] + s[2] + s[3];
    if (c) atomicAdd(total, c);
  }
}

// Strict overlap on axes [A0, A1) of a's k-DOP with the k-DOP in planes of nb.
template <int A0, int A1>
__device__ __forceinline__ bool sweep_axes(const double* ak, const double* kb, uint64_t nb) {
  bool o = true;
#pragma unroll
  for (int x = A0; x < A1; ++x)
    o = o & (ak[2 * x] < kb[(uint64_t)(2 * x + 1) * nb]) & (kb[(uint64_t)(2 * x) * nb] < ak[2 * x + 1]);
  return o;
}

// The sweep of one element a of A by one wave: COUNT writes a's pair count;
// WRITE writes the pairs at a's exclusive offset.
template <bool WRITE>
__device__ __forceinline__ void sweep_one(const SweepArgs& a, uint64_t ai, int lane) {
  const double* ak = a.ka + ai * 26;
  const uint32_t amin = (uint32_t)float_to_uint((ak[2 * a.axis] - a.gmin) * a.conv);
  const uint32_t amax = (uint32_t)float_to_uint((ak[2 * a.axis + 1] - a.gmin) * a.conv);
  // the first sorted position whose minimum exceeds amax: the sweep's stop
  // (64 probes a round: those at or below amax are the first c of them)
  uint64_t lo = 0, hi = a.nb;
  while (lo < hi) {
    const uint64_t step = (hi - lo + 63) / 64, at = lo + (uint64_t)lane * step;
    const uint64_t c = (uint64_t)__popcll(__ballot(at < hi && a.bq[at < hi ? at : lo] <= amax));
    if (c == 0) break;  // position lo is above
    if (lo + c * step < hi) hi = lo + c * step;
    lo += (c - 1) * step + 1;
  }
  const uint64_t ub = lo;
  uint32_t cnt = 0;
  uint64_t base = 0;
  uint64_t gid_a = 0;
  if constexpr (WRITE) {
    base = a.count[ai];
    gid_a = a.ga ? a.ga[ai] : ai;
  }
  uint64_t t0 = 0, tiles = 0;  // tiles to walk among the 64 from t0 - 64 on
  for (;;) {
    while (tiles == 0 && t0 * 64 < ub) {
      const uint64_t t = t0 + lane;
      tiles = __ballot(t * 64 < ub && !(a.tmax[t * 64 < ub ? t : t0] < (double)amin));
      t0 += 64;
    }
    if (tiles == 0) break;
    const uint64_t j = (t0 - 64 + (uint64_t)__builtin_ctzll(tiles)) * 64 + lane;
    tiles &= tiles - 1;
    bool hit = false;
    if (j < ub) {
      // skipped while b lies below a (bmax < amin, fp64 against the integer)
      hit = !(a.bmax[j] < (double)amin);
      // x, y and z first: the other axes are read if these leave a lane
      hit = hit & sweep_axes<0, 3>(ak, a.kbs + j, a.nb);
    }
    if (__ballot(hit) == 0) continue;
    if (j < ub) hit = hit & sweep_axes<3, kAxes>(ak, a.kbs + j, a.nb);
    const uint64_t m = __ballot(hit);
    if constexpr (WRITE) {
      if (hit) {
        const uint64_t pos = base + cnt + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                     __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        const uint32_t bj = a.bidx[j];
        a.out[2 * pos] = gid_a;
        a.out[2 * pos + 1] = a.gb ? a.gb[bj] : bj;
      }
    }
    cnt += (uint32_t)__popcll(m);
  }
  if constexpr (!WRITE) {
    if (lane == 0) a.count[ai] = cnt;
  }
}

// One wave per element a of A, striding over A.
template <bool WRITE>
__global__ __launch_bounds__(256) void k_sweep(SweepArgs a) {
  const int lane = threadIdx.x & 63;
  // a is uniform across the wave: every wave leaves the loop together
  for (uint64_t ai = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6); ai < a.na; ai += (uint64_t)gridDim.x * 4)
    sweep_one<WRITE>(a, ai, lane);
}

// kdop::from_vertices for a batch of polytopes (kdop.hpp:238-264): element
// e's 26-DOP (n x 26) with the build's own projections, for callers that
// sweep elements outside an object.
template <int NV>
__global__ __launch_bounds__(256) void k_element_kdops(ElemInput in, double* __restrict__ out) {
  const uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= in.n) return;
  double kd[kSlabs];
  element_kdop<kPoly, NV>(in, (uint32_t)e, kd);
#pragma unroll
  for (int i = 0; i < kSlabs; ++i) out[e * kSlabs + i] = kd[i];
}

hipError_t launch_element_kdops(const ElemInput& in, double* out, hipStream_t s) {
  if (in.n == 0) return hipSuccess;
  const dim3 g((uint32_t)((in.n + 255) / 256)), b(256);
  switch (in.nv) {
    case 1: hipLaunchKernelGGL(k_element_kdops<1>, g, b, 0, s, in, out); break;
    case 2: hipLaunchKernelGGL(k_element_kdops<2>, g, b, 0, s, in, out); break;
    case 3: hipLaunchKernelGGL(k_element_kdops<3>, g, b, 0, s, in, out); break;
    case 4: hipLaunchKernelGGL(k_element_kdops<4>, g, b, 0, s, in, out); break;
    case 5: hipLaunchKernelGGL(k_element_kdops<5>, g, b, 0, s, in, out); break;
    case 6: hipLaunchKernelGGL(k_element_kdops<6>, g, b, 0, s, in, out); break;
    case 7: hipLaunchKernelGGL(k_element_kdops<7>, g, b, 0, s, in, out); break;
    case 8: hipLaunchKernelGGL(k_element_kdops<8>, g, b, 0, s, in, out); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_variant_axis(const double* ca, uint64_t na, const double* cb, uint64_t nb, double* part,
                               int32_t* axis, hipStream_t s) {
  const uint64_t n = na + nb;
  uint64_t blocks = (n + kMomentBlock - 1) / kMomentBlock;
  if (blocks > kMomentBlocks) blocks = kMomentBlocks;
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(k_moments, dim3((uint32_t)blocks), dim3(kMomentBlock), 0, s, ca, na, cb, nb, part);
  hipLaunchKernelGGL(k_variant_axis, dim3(1), dim3(256), 0, s, part, (uint32_t)blocks, n, axis);
  return hipGetLastError();
}

uint32_t variant_axis_partials() { return kMomentBlocks; }

hipError_t launch_sweep_prepare(const double* kb, uint64_t nb, int axis, double gmin, double conv, uint32_t* bq,
                                uint32_t* bidx, hipStream_t s) {
  if (nb == 0) return hipSuccess;
  hipLaunchKernelGGL(k_sweep_quantize, dim3((uint32_t)((nb + 255) / 256)), dim3(256), 0, s, kb, nb, axis, gmin, conv,
                     bq, bidx);
  return hipGetLastError();
}

hipError_t launch_sweep_gather(const double* kb, const uint32_t* bidx, uint64_t nb, int axis, double gmin,
                               double conv, double* kbs, double* bmax, double* tmax, hipStream_t s) {
  if (nb == 0) return hipSuccess;
  hipLaunchKernelGGL(k_sweep_gather, dim3((uint32_t)((nb + 63) / 64)), dim3(256), 0, s, kb, bidx, nb, axis, gmin,
                     conv, kbs, bmax, tmax);
  return hipGetLastError();
}

hipError_t launch_sweep(const SweepArgs& a, bool write, hipStream_t s) {
  if (a.na == 0) return hipSuccess;
  uint64_t blocks = (a.na + 3) / 4;
  if (blocks > 65536) blocks = 65536;
  if (write) {
    hipLaunchKernelGGL(k_sweep<true>, dim3((uint32_t)blocks), dim3(256), 0, s, a);
  } else {
    hipLaunchKernelGGL(k_sweep<false>, dim3((uint32_t)blocks), dim3(256), 0, s, a);
    uint64_t sum = (a.na + 2047) / 2048;
    if (sum > 64) sum = 64;
    hipLaunchKernelGGL(k_sweep_total, dim3((uint32_t)sum), dim3(256), 0, s, (const uint32_t*)a.count, a.na, a.total);
  }
  return hipGetLastError();
}

}  // namespace dbvh
