// sort.hip -- stable LSD radix sort for gfx950 (8-bit digits, one kernel per
// digit pass, decoupled look-back across tiles).
//
// Replaces radix_sorter<T, I> (util/sort.hpp:75-144), which runs one 1-bit
// split pass (3 dispatches) per key bit.  The result is the same stable
// permutation: keys ascending, ties in input order.
//
// Per pass, a workgroup takes a tile of 4,096 or 8,192 keys (tile ids come
// from an atomic counter, so a tile only ever waits on tiles already running):
//  * keys are read coalesced (a wave's items are consecutive runs of 64) and
//    ranked per wave with 8 ballots per item (the lanes holding the same
//    digit) plus per-wave LDS digit counters;
//  * the tile's 256 digit counts are published as an aggregate, then each
//    thread (= digit) walks back over earlier tiles until it meets an
//    inclusive prefix (flag and count packed in one 32-bit word, agent-scope
//    atomics);
//  * keys and payloads are reordered by digit in LDS and written out in digit
//    runs, so consecutive lanes write consecutive addresses.
// Digit histograms for all passes come from one read of the keys (fused into
// the Morton kernel for the object build).  A pass whose digit is the same
// for every key is skipped on the device.
#include "device.hpp"
#include "kernels.hpp"
#include "sort_block.hpp"

namespace dbvh {

// The two shapes of a pass.  Narrow: 1,024 threads x 4 keys, keys and payloads
// in LDS together; its tile's latency is the shortest (4 serial ranking steps
// a wave), which is what bounds a sort of few tiles.  Wide: 512 threads x 16
// keys, payloads after the keys through the same LDS, so that two workgroups
// share a CU (72 KB each) and one's ranking hides the other's memory time,
// and the digit runs written are twice as long.  Per 8-bit pass of u64 keys
// with payloads, narrow / wide: 54,612 keys 9.1 / 13.8 us, 524,288 13.7 / 17.3,
// 2,097,152 25.0 / 23.4, 12,000,017 104.9 / 81.3 (one shape of 256 threads x
// 16 keys: 13.3, 18.0, 28.8, 118.7).  The line is where whole sorts cross, for
// both key widths, with and without payload (narrow / wide, us): u64 pairs 202 /
// 214 at 1,048,576 keys, 226 / 227 at 1,500,000, 242 / 228 at 1,650,000; u64 keys
// 187 / 193, 215 / 216, 228 / 218; u32 pairs 118 / 127, 133 / 136, 141 / 137; u32
// keys 110 / 116, 123 / 124, 133 / 127.
template <bool WIDE>
struct SortShape {
  static constexpr int block = WIDE ? 512 : 1024;
  static constexpr int items = WIDE ? 16 : 4;
  static constexpr int tile = block * items;
};
constexpr uint64_t kSortWideMin = 3ull << 19;  // 1,572,864 keys
constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagInc = 2u << 30;
constexpr uint32_t kValMask = (1u << 30) - 1u;
constexpr int kScanItems = 16;
constexpr int kScanTile = 256 * kScanItems;
constexpr int kLookWindow = 4;  // predecessors read per look-back round trip

__device__ __forceinline__ uint32_t lb_load(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void lb_store(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive scan of one value per thread over a 256-thread block.
__device__ __forceinline__ uint32_t block_excl_scan256(uint32_t v, uint32_t* s_tmp /*4*/) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_tmp[w] = x;
  __syncthreads();
  uint32_t wp = 0;
  for (int i = 0; i < w; ++i) wp += s_tmp[i];
  __syncthreads();
  return wp + x - v;
}

// Histograms of all digit passes of `keys` (grid-stride), and the sort's
// look-back words cleared.  What bounds it is adds to one address: lanes of a
// wave that share a digit serialise in LDS, and the blocks' sums on a digit's
// word in memory.  So the LDS histograms are kept twice (lane mod 2,
// interleaved over the banks; four copies cost a workgroup a place on the CU
// and took 109 us where two take 85), a wave whose lanes all share a digit
// adds once, and the blocks' sums go to kHistCopies copies (block b to copy b
// mod kHistCopies) that the plan sums.  With one LDS histogram a block, a
// block per 256 keys and one copy in memory it took 320 us on the 27 M pair
// keys of a sphere cloud and 36 us on 420,000; now 110 and 10.
constexpr unsigned kHistBlocks = 2048;
constexpr int kHistLds = 2;
constexpr uint64_t kHistKeys = 4;  // keys per thread and round, their loads together
template <typename K>
__global__ __launch_bounds__(256) void k_sort_histogram(const K* __restrict__ keys, uint64_t n,
                                                        uint32_t* __restrict__ hist, uint32_t* __restrict__ lookback,
                                                        uint64_t lb_words) {
  constexpr int kPasses = sizeof(K);
  __shared__ uint32_t sh[kPasses * 256 * kHistLds];
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
  for (int i = threadIdx.x; i < kPasses * 256 * kHistLds; i += 256) sh[i] = 0;
  for (uint64_t i = gid; i < lb_words; i += stride) lookback[i] = 0;
  __syncthreads();
  const uint32_t copy = threadIdx.x % kHistLds;
  for (uint64_t i0 = gid; i0 - threadIdx.x % 64 < n; i0 += kHistKeys * stride) {  // uniform per wave
    K k[kHistKeys];
#pragma unroll
    for (uint64_t u = 0; u < kHistKeys; ++u) k[u] = i0 + u * stride < n ? keys[i0 + u * stride] : (K)0;
#pragma unroll
    for (uint64_t u = 0; u < kHistKeys; ++u) {
      const bool valid = i0 + u * stride < n;
      const uint64_t active = __ballot(valid);
      if (active == 0) break;
      const uint32_t leader = (uint32_t)(__ffsll((long long)active) - 1);
#pragma unroll
      for (int p = 0; p < kPasses; ++p) {
        const uint32_t d = (uint32_t)(k[u] >> (8 * p)) & 255u;
        const uint32_t d0 = __builtin_amdgcn_readlane(d, leader);
        if (__ballot(valid & (d != d0)) == 0) {
          if (lane_id() == leader) atomicAdd(&sh[(p * 256 + d0) * kHistLds], (uint32_t)__popcll(active));
        } else if (valid) {
          atomicAdd(&sh[(p * 256 + d) * kHistLds + copy], 1u);
        }
      }
    }
  }
  __syncthreads();
  uint32_t* h = hist + (blockIdx.x % kHistCopies) * kSortHistWords;
  for (int i = threadIdx.x; i < kPasses * 256; i += 256) {
    const uint32_t c = sh[kHistLds * i] + sh[kHistLds * i + 1];
    if (c) atomicAdd(&h[i], c);
  }
}

// One block: digit offsets (exclusive scan per pass), pass activity and the
// ping-pong buffer selectors: the last active pass writes buffer A, or the
// result buffer with out_sel0 = kSelOut.  That buffer may be the input, so at
// least two passes are then active (one more moves every key to its own
// place): no pass reads what it writes.
constexpr uint32_t kSelOut = 3;
__global__ __launch_bounds__(256) void k_sort_plan(const uint32_t* __restrict__ hist, uint64_t n, int npass,
                                                   SortCtl* __restrict__ ctl, int copies, uint32_t copy_stride,
                                                   uint32_t out_sel0) {
  __shared__ uint32_t s_wtot[8][4];
  __shared__ uint32_t s_active[8];
  const int t = threadIdx.x;
  // every pass's count of digit t, summed over the copies (all loads issued
  // before any is used)
  // (every load is made, at a clamped address, and the unwanted ones count
  // zero: no branch separates them)
  uint32_t hv[8][8];
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    const int pp = p < npass ? p : 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int cc = c < copies ? c : 0;
      hv[p][c] = hist[(uint64_t)cc * copy_stride + pp * 256 + t];
    }
  }
  uint32_t hs[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    hs[p] = 0;
#pragma unroll
    for (int c = 0; c < 8; ++c) hs[p] += (p < npass && c < copies) ? hv[p][c] : 0u;
  }
  // the exclusive scans of all passes side by side (wave scans, then the
  // four wave totals of each pass through LDS: two barriers for all passes);
  // a pass is needed unless one bin holds every key
  const int lane = t & 63, w = t >> 6;
  uint32_t xs[8];
#pragma unroll
  for (int p = 0; p < 8; ++p) xs[p] = hs[p];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const uint32_t y = __shfl_up(xs[p], o, 64);
      if (lane >= o) xs[p] += y;
    }
  }
  if (t < 8) s_active[t] = 1u;
  __syncthreads();
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    if (lane == 63) s_wtot[p][w] = xs[p];
    if (p < npass && (uint64_t)hs[p] == n) s_active[p] = 0u;
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < 8; ++p) {
    if (p >= npass) break;  // (uniform)
    uint32_t wp = 0;
    for (int i = 0; i < w; ++i) wp += s_wtot[p][i];
    ctl->offsets[p * 256 + t] = wp + xs[p] - hs[p];
  }
  if (t == 0) {
    int nact = 0;
    for (int p = 0; p < npass; ++p) nact += s_active[p];
    const int need = out_sel0 == kSelOut ? 2 : 1;
    for (int p = 0; p < npass && nact < need; ++p)
      if (!s_active[p]) {
        s_active[p] = 1;
        ++nact;
      }
    // walk backwards: last active pass -> the result, previous -> A or B in turn
    uint32_t out_sel[8];
    uint32_t cur = out_sel0;
    for (int p = npass - 1; p >= 0; --p) {
      if (s_active[p]) {
        out_sel[p] = cur;
        cur = (cur == 1) ? 2 : 1;
      } else {
        out_sel[p] = 0;
      }
    }
    uint32_t prev_out = 0;  // input of the first active pass is the caller's buffer (0)
    for (int p = 0; p < npass; ++p) {
      SortPassInfo pi;
      pi.active = s_active[p];
      pi.in_sel = prev_out;
      pi.out_sel = out_sel[p];
      pi.first = (prev_out == 0) ? 1u : 0u;
      ctl->pass[p] = pi;
      if (s_active[p]) prev_out = out_sel[p];
      ctl->tile_counter[p] = 0;
    }
    for (int p = npass; p < 8; ++p) {
      ctl->pass[p].active = 0;
      ctl->tile_counter[p] = 0;
    }
  }
}

// One digit pass over one tile.  Bound by the VALU work of the ranking (about
// 45 instructions a key) beside the memory time of 24 bytes a key.
template <typename K, bool WIDE>
__global__ __launch_bounds__(SortShape<WIDE>::block) void k_sort_pass(SortArgs<K> a, int pass) {
  constexpr int kBlock = SortShape<WIDE>::block, kItems = SortShape<WIDE>::items, kTile = SortShape<WIDE>::tile;
  constexpr int kWaves = kBlock / 64;
  const SortPassInfo pi = a.ctl->pass[pass];
  if (!pi.active) return;
  const K* __restrict__ kin = pi.in_sel == 0 ? a.k0 : (pi.in_sel == 1 ? a.ka : a.kb);
  K* __restrict__ kout = pi.out_sel == 1 ? a.ka : (pi.out_sel == 2 ? a.kb : a.kout);
  const uint32_t* __restrict__ vin = pi.in_sel == 0 ? a.v0 : (pi.in_sel == 1 ? a.va : a.vb);
  uint32_t* __restrict__ vout = pi.out_sel == 1 ? a.va : (pi.out_sel == 2 ? a.vb : a.vout);
  const bool has_vals = a.va != nullptr;
  const int shift = 8 * pass;
  const uint64_t n = a.n;

  __shared__ uint32_t s_tile;
  __shared__ __align__(4) uint16_t s_wcount[kWaves][256];  // (a tile's counts fit 16 bits)
  __shared__ uint32_t s_texcl[256];
  __shared__ uint32_t s_gbase[256];
  __shared__ uint32_t s_tmp[4];
  __shared__ uint32_t s_hist[256];
  __shared__ __align__(16) unsigned char s_buf[kTile * (WIDE ? sizeof(K) : sizeof(K) + 4)];
  K* s_keys = (K*)s_buf;
  uint32_t* s_vals = (uint32_t*)(WIDE ? s_buf : s_buf + kTile * sizeof(K));

  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  if (tid == 0) s_tile = atomicAdd(&a.ctl->tile_counter[pass], 1u);
  for (int i = tid; i < kWaves * 128; i += kBlock) ((uint32_t*)&s_wcount[0][0])[i] = 0;
  if (tid < 256) s_hist[tid] = 0;
  __syncthreads();
  const uint32_t tile = s_tile;
  if (tile >= a.ntiles) return;  // uniform per block; no tile waits on it
  const uint64_t base = (uint64_t)tile * kTile;
  const uint32_t cnt = (uint32_t)(n - base < (uint64_t)kTile ? n - base : (uint64_t)kTile);

  // this thread's keys: tile positions p0 + 64 j
  const uint32_t p0 = (uint32_t)(w * (kItems * 64) + lane);
  K key[kItems];
  uint32_t val[kItems];
  uint32_t rank[kItems];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const uint64_t pos = base + (p0 + j * 64);
    const bool valid = pos < n;
    key[j] = valid ? kin[pos] : (K)0;
    if (has_vals) val[j] = valid ? (vin ? vin[pos] : (uint32_t)pos) : 0u;
  }
  auto valid = [&](int j) { return p0 + j * 64 < cnt; };
  auto digit = [&](K k) { return (uint32_t)(k >> shift) & 255u; };
  // the tile's digit counts first, published as its aggregate before the
  // ranking, so that later tiles' look-backs find it sooner
#pragma unroll
  for (int j = 0; j < kItems; ++j)
    if (valid(j)) atomicAdd(&s_hist[digit(key[j])], 1u);
  __syncthreads();
  uint32_t* lb = a.lookback + ((uint64_t)pass * a.ntiles + tile) * 256;
  uint32_t total = 0;
  if (tid < 256) {
    total = s_hist[tid];
    lb_store(&lb[tid], (tile == 0 ? kFlagInc : kFlagAgg) | total);
  }
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const uint32_t d = digit(key[j]);
    const bool ok = valid(j);
    const uint64_t m = __ballot(ok);
    uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
#pragma unroll
    for (int b = 0; b < 8; ++b) match_bit(d, b, lo, hi);
    const uint32_t before = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    const uint32_t same = (uint32_t)(__popc(lo) + __popc(hi));
    uint32_t old = 0;
    if (ok) old = s_wcount[w][d];
    rank[j] = old + before;
    __builtin_amdgcn_wave_barrier();
    if (ok && before == 0) s_wcount[w][d] = (uint16_t)(old + same);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();

  // thread t < 256 owns digit t: exclusive scans over the waves and the digits
  uint32_t x = total;
  if (tid < 256) {
    uint32_t run = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) {
      const uint32_t c = s_wcount[v][tid];
      s_wcount[v][tid] = (uint16_t)run;
      run += c;
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_tmp[w] = x;
  }
  __syncthreads();
  if (tid < 256) {
    uint32_t texcl = x - total;
    for (int i = 0; i < w; ++i) texcl += s_tmp[i];
    s_texcl[tid] = texcl;
    uint32_t excl = 0;
    if (tile > 0) {
      // decoupled look-back over a window of kLookWindow predecessors whose
      // words are loaded together (one round trip per window, not per tile):
      // their aggregates are added in order up to the first inclusive prefix;
      // a word not yet published is polled until it is (tile 0 publishes an
      // inclusive prefix, so the walk ends by it)
      const uint32_t* lb0 = a.lookback + (uint64_t)pass * a.ntiles * 256 + tid;
      int64_t prev = (int64_t)tile - 1;
      bool done = false;
      while (!done) {
        uint32_t v[kLookWindow];
#pragma unroll
        for (int k = 0; k < kLookWindow; ++k) v[k] = prev - k >= 0 ? lb_load(lb0 + (uint64_t)(prev - k) * 256) : 0u;
#pragma unroll
        for (int k = 0; k < kLookWindow; ++k) {
          if (done || prev - k < 0) break;
          uint32_t y = v[k];
          while ((y & ~kValMask) == 0) {
            __builtin_amdgcn_s_sleep(1);
            y = lb_load(lb0 + (uint64_t)(prev - k) * 256);
          }
          excl += y & kValMask;
          done = (y & ~kValMask) == kFlagInc;
        }
        prev -= kLookWindow;
      }
      lb_store(&lb[tid], kFlagInc | (excl + total));
    }
    s_gbase[tid] = a.ctl->offsets[pass * 256 + tid] + excl - texcl;  // + tile-local place = output position
  }
  __syncthreads();

#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const uint32_t d = digit(key[j]);
    rank[j] += s_texcl[d] + s_wcount[w][d];  // now the place in the tile's output
    if (valid(j)) {
      s_keys[rank[j]] = key[j];
      if (!WIDE && has_vals) s_vals[rank[j]] = val[j];
    }
  }
  __syncthreads();
  uint32_t op[kItems];
#pragma unroll
  for (int j = 0; j < kItems; ++j) {
    const uint32_t i = j * kBlock + tid;
    op[j] = kEnd;
    if (i < cnt) {
      const K k = s_keys[i];
      op[j] = s_gbase[digit(k)] + i;
      if (op[j] < n) {
        kout[op[j]] = k;
        if (!WIDE && has_vals) vout[op[j]] = s_vals[i];
      }
    }
  }
  if (WIDE && has_vals) {
    __syncthreads();  // the keys in LDS have been read
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (valid(j)) s_vals[rank[j]] = val[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j)
      if (op[j] < n) vout[op[j]] = s_vals[j * kBlock + tid];
  }
}

// A whole sort of at most kSmallBlock * ITEMS keys in one workgroup: the keys
// and payloads stay in registers between passes and change places through LDS,
// digits that all keys share are skipped, and nothing is cleared or planned
// beforehand.  Bound by its barriers and LDS latency: 1.5 us a pass of 512
// pairs, 6 us of 8,192.  A whole sort of 512 / 4,096 / 8,192 pairs takes 13 /
// 30 / 48 us so, 51 / 63 / 72 as passes of their own; at 16,384 keys the one
// CU's work would pass the launches' 75 us.
template <typename K, int ITEMS>
__global__ __launch_bounds__(kSmallBlock) void k_sort_small(SortArgs<K> a, int npass) {
  __shared__ SortBlockLds<K, ITEMS> L;
  const uint32_t n = (uint32_t)a.n;
  const K* k0 = a.k0;
  const uint32_t* v0 = a.v0;
  K* kout = a.kout ? a.kout : a.ka;  // (may be the input)
  uint32_t* vout = a.kout ? a.vout : a.va;
  const bool has_vals = a.va != nullptr;
  K key[ITEMS];
  uint32_t val[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t pos = small_pos<ITEMS>(j);
    key[j] = pos < n ? k0[pos] : (K)0;
    val[j] = has_vals && pos < n ? (v0 ? v0[pos] : pos) : 0u;
  }
  sort_block<K, ITEMS>(L, key, val, has_vals, n, npass);
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t pos = small_pos<ITEMS>(j);
    if (pos < n) {
      kout[pos] = key[j];
      if (has_vals) vout[pos] = val[j];
    }
  }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

__global__ void k_iota_u32(uint32_t* __restrict__ p, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = (uint32_t)i;
}

template <typename T>
__global__ void k_copy(T* __restrict__ dst, const T* __restrict__ src, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// ---- host launchers ----------------------------------------------------------------
// tiles of the narrow shape and of the scan: what callers size look-back
// words by (the wide shape has fewer)
uint64_t sort_tiles(uint64_t n) { return (n + kScanTile - 1) / kScanTile; }

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_iota_u32(uint32_t* p, uint64_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_iota_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_copy(T* dst, const T* src, uint64_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_copy<T>, dim3((unsigned)blocks), dim3(256), 0, s, dst, src, n);
  return hipGetLastError();
}
template hipError_t launch_copy<uint64_t>(uint64_t*, const uint64_t*, uint64_t, hipStream_t);
template hipError_t launch_copy<uint32_t>(uint32_t*, const uint32_t*, uint64_t, hipStream_t);
template hipError_t launch_copy<double>(double*, const double*, uint64_t, hipStream_t);

template <typename K>
static hipError_t launch_sort_histogram(const SortArgs<K>& a, uint32_t* hist, hipStream_t s) {
  uint64_t blocks = (a.n + 2047) / 2048;
  if (blocks > kHistBlocks) blocks = kHistBlocks;
  hipLaunchKernelGGL(k_sort_histogram<K>, dim3((unsigned)blocks), dim3(256), 0, s, a.k0, a.n, hist, a.lookback,
                     sizeof(K) * sort_tiles(a.n) * 256);
  return hipGetLastError();
}

// Sort after the histograms are in `hist` (npass * 256 counters) and the
// look-back words are zero.  Result in a.ka (and a.va).
template <typename K>
hipError_t launch_sort_plan(const SortArgs<K>& a, int npass, const uint32_t* hist, hipStream_t s, int copies,
                            uint32_t copy_stride) {
  if (a.n == 0) return hipSuccess;
  if (npass < 1 || npass > 8 || copies < 1 || copies > 8) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_sort_plan, dim3(1), dim3(256), 0, s, hist, a.n, npass, a.ctl, copies, copy_stride,
                     a.kout ? kSelOut : 1u);
  return hipGetLastError();
}

template <typename K>
hipError_t launch_sort_pass(const SortArgs<K>& a, int p, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  SortArgs<K> b = a;
  if (a.n >= kSortWideMin) {
    using S = SortShape<true>;
    b.ntiles = (a.n + S::tile - 1) / S::tile;
    hipLaunchKernelGGL((k_sort_pass<K, true>), dim3((unsigned)b.ntiles), dim3(S::block), 0, s, b, p);
  } else {
    using S = SortShape<false>;
    b.ntiles = (a.n + S::tile - 1) / S::tile;
    hipLaunchKernelGGL((k_sort_pass<K, false>), dim3((unsigned)b.ntiles), dim3(S::block), 0, s, b, p);
  }
  return hipGetLastError();
}

constexpr uint64_t kSortSmallMax = 8 * kSmallBlock;
bool sort_is_small(uint64_t n) { return n <= kSortSmallMax; }

template <typename K>
hipError_t launch_sort_small(const SortArgs<K>& a, int npass, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (!sort_is_small(a.n) || npass < 1 || npass > (int)sizeof(K)) return hipErrorInvalidValue;
  const dim3 g(1), b(kSmallBlock);
  if (a.n <= 1 * kSmallBlock) hipLaunchKernelGGL((k_sort_small<K, 1>), g, b, 0, s, a, npass);
  else if (a.n <= 2 * kSmallBlock) hipLaunchKernelGGL((k_sort_small<K, 2>), g, b, 0, s, a, npass);
  else if (a.n <= 4 * kSmallBlock) hipLaunchKernelGGL((k_sort_small<K, 4>), g, b, 0, s, a, npass);
  else hipLaunchKernelGGL((k_sort_small<K, 8>), g, b, 0, s, a, npass);
  return hipGetLastError();
}
template hipError_t launch_sort_small<uint64_t>(const SortArgs<uint64_t>&, int, hipStream_t);
template hipError_t launch_sort_small<uint32_t>(const SortArgs<uint32_t>&, int, hipStream_t);

template <typename K>
hipError_t launch_sort(const SortArgs<K>& a, int npass, uint32_t* hist, hipStream_t s) {
  if (a.n == 0) return hipSuccess;
  if (sort_is_small(a.n)) return launch_sort_small<K>(a, npass, s);
  hipError_t e = launch_fill_u32(hist, (uint64_t)kHistCopies * kSortHistWords, 0u, s);
  if (e == hipSuccess) e = launch_sort_histogram<K>(a, hist, s);
  if (e == hipSuccess) e = launch_sort_plan<K>(a, npass, hist, s, kHistCopies, kSortHistWords);
  for (int p = 0; p < npass && e == hipSuccess; ++p) e = launch_sort_pass<K>(a, p, s);
  return e;
}
template hipError_t launch_sort_plan<uint64_t>(const SortArgs<uint64_t>&, int, const uint32_t*, hipStream_t, int,
                                              uint32_t);
template hipError_t launch_sort_plan<uint32_t>(const SortArgs<uint32_t>&, int, const uint32_t*, hipStream_t, int,
                                              uint32_t);
template hipError_t launch_sort_pass<uint64_t>(const SortArgs<uint64_t>&, int, hipStream_t);
template hipError_t launch_sort_pass<uint32_t>(const SortArgs<uint32_t>&, int, hipStream_t);
template hipError_t launch_sort<uint64_t>(const SortArgs<uint64_t>&, int, uint32_t*, hipStream_t);
template hipError_t launch_sort<uint32_t>(const SortArgs<uint32_t>&, int, uint32_t*, hipStream_t);


// ---- exclusive scan (prefix_sum, util/prefix_sum.hpp:41-54) ---------------------------
// Single pass: 256 threads x 16 values per tile, decoupled look-back with the
// flag in the top two bits of a 64-bit word.  Values wrap modulo 2^32 as the
// reference's uint32 scan does.
constexpr uint64_t kScanAgg = 1ull << 62;
constexpr uint64_t kScanInc = 2ull << 62;
constexpr uint64_t kScanMask = (1ull << 62) - 1;

__global__ __launch_bounds__(256) void k_scan_u32(uint32_t* __restrict__ v, uint64_t n, uint64_t* __restrict__ lb,
                                                  uint32_t* __restrict__ counter) {
  __shared__ uint32_t s_tile;
  __shared__ uint32_t s_tmp[4];
  __shared__ uint64_t s_excl;
  const int tid = threadIdx.x;
  if (tid == 0) s_tile = atomicAdd(counter, 1u);
  __syncthreads();
  const uint32_t tile = s_tile;
  if ((uint64_t)tile * kScanTile >= n) return;
  const uint64_t base = (uint64_t)tile * kScanTile + (uint64_t)tid * kScanItems;
  uint32_t x[kScanItems];
  uint32_t sum = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    const uint64_t i = base + j;
    x[j] = i < n ? v[i] : 0u;
    sum += x[j];
  }
  const uint32_t texcl = block_excl_scan256(sum, s_tmp);
  if (tid == 255) {
    const uint64_t total = (uint64_t)(texcl + sum);
    uint64_t excl = 0;
    if (tile == 0) {
      __hip_atomic_store(&lb[0], kScanInc | (total & kScanMask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
      __hip_atomic_store(&lb[tile], kScanAgg | (total & kScanMask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      int64_t prev = (int64_t)tile - 1;
      for (;;) {
        uint64_t w = __hip_atomic_load(&lb[prev], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        while ((w & ~kScanMask) == 0) {
          __builtin_amdgcn_s_sleep(1);
          w = __hip_atomic_load(&lb[prev], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        excl += w & kScanMask;
        if ((w & ~kScanMask) == kScanInc) break;
        --prev;
      }
      __hip_atomic_store(&lb[tile], kScanInc | ((excl + total) & kScanMask), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    s_excl = excl;
  }
  __syncthreads();
  uint32_t run = (uint32_t)s_excl + texcl;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    const uint64_t i = base + j;
    if (i < n) v[i] = run;
    run += x[j];
  }
}

hipError_t launch_scan_u32(uint32_t* v, uint64_t n, uint64_t* lb, uint32_t* counter, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_scan_u32, dim3((unsigned)sort_tiles(n)), dim3(256), 0, s, v, n, lb, counter);
  return hipGetLastError();
}

}  // namespace dbvh
