// sort_block.hpp -- the radix sort of few keys inside one workgroup.
#pragma once
#include "device.hpp"

namespace dbvh {

// Keeps in (lo, hi), a lane mask, the lanes whose bit b of d equals this
// lane's: m & ~(ballot ^ own bit), one three-input operation per half.
__device__ __forceinline__ void match_bit(uint32_t d, int b, uint32_t& lo, uint32_t& hi) {
  const int own = (int)(d << (31 - b)) >> 31;
  const uint64_t bb = __ballot(own != 0);
  lo = (uint32_t)__builtin_amdgcn_bitop3_b32((int)lo, (int)(uint32_t)bb, own, 0x90);
  hi = (uint32_t)__builtin_amdgcn_bitop3_b32((int)hi, (int)(uint32_t)(bb >> 32), own, 0x90);
}

constexpr int kSmallBlock = 1024;

template <typename K, int ITEMS>
struct SortBlockLds {
  K keys[kSmallBlock * ITEMS];
  uint32_t vals[kSmallBlock * ITEMS];
  alignas(4) uint16_t wcount[kSmallBlock / 64][256];
  uint32_t texcl[256];
  uint32_t tmp[4];
  uint32_t diff[2];
  K first;
};

// position of item j of this thread: a wave's items are consecutive runs of 64
template <int ITEMS>
__device__ __forceinline__ uint32_t small_pos(int j) {
  return (threadIdx.x >> 6) * (ITEMS * 64) + (threadIdx.x & 63) + j * 64;
}

// Stable sort of the block's n keys (position small_pos(j) in key[j]) by
// their lowest npass bytes, in place, with payloads if has_vals.  Called by
// all kSmallBlock threads; L is free again after the next barrier.
template <typename K, int ITEMS>
__device__ __forceinline__ void sort_block(SortBlockLds<K, ITEMS>& L, K (&key)[ITEMS], uint32_t (&val)[ITEMS],
                                           bool has_vals, uint32_t n, int npass) {
  constexpr int kWaves = kSmallBlock / 64;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  auto valid = [&](int j) { return small_pos<ITEMS>(j) < n; };
  if (tid < 2) L.diff[tid] = 0;
  if (tid == 0) L.first = key[0];
  for (int i = lane; i < 128; i += 64) ((uint32_t*)&L.wcount[w][0])[i] = 0;
  __syncthreads();
  {  // the bits in which some key differs from the first
    const K f = L.first;
    K x = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
      if (valid(j)) x |= key[j] ^ f;
    uint32_t lo = (uint32_t)x, hi = sizeof(K) == 8 ? (uint32_t)((uint64_t)x >> 32) : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo |= __shfl_xor(lo, o, 64);
      if (sizeof(K) == 8) hi |= __shfl_xor(hi, o, 64);
    }
    if (lane == 0) {
      if (lo) atomicOr(&L.diff[0], lo);
      if (hi) atomicOr(&L.diff[1], hi);
    }
  }
  __syncthreads();
  const uint64_t diff = ((uint64_t)L.diff[1] << 32) | L.diff[0];
  for (int p = 0; p < npass; ++p) {
    const int shift = 8 * p;
    if (((diff >> shift) & 255u) == 0) continue;  // uniform
    uint32_t rank[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      const uint32_t d = (uint32_t)(key[j] >> shift) & 255u;
      const bool ok = valid(j);
      const uint64_t m = __ballot(ok);
      uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
#pragma unroll
      for (int b = 0; b < 8; ++b) match_bit(d, b, lo, hi);
      const uint32_t before = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
      const uint32_t same = (uint32_t)(__popc(lo) + __popc(hi));
      uint32_t old = 0;
      if (ok) old = L.wcount[w][d];
      rank[j] = old + before;
      __builtin_amdgcn_wave_barrier();
      if (ok && before == 0) L.wcount[w][d] = (uint16_t)(old + same);
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    uint32_t run = 0, x = 0;
    if (tid < 256) {
#pragma unroll
      for (int v = 0; v < kWaves; ++v) {
        const uint32_t c = L.wcount[v][tid];
        L.wcount[v][tid] = (uint16_t)run;
        run += c;
      }
      x = run;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
      }
      if (lane == 63) L.tmp[w] = x;
    }
    __syncthreads();
    if (tid < 256) {
      uint32_t texcl = x - run;
      for (int i = 0; i < w; ++i) texcl += L.tmp[i];
      L.texcl[tid] = texcl;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (valid(j)) {
        const uint32_t d = (uint32_t)(key[j] >> shift) & 255u;
        const uint32_t at = L.texcl[d] + L.wcount[w][d] + rank[j];
        L.keys[at] = key[j];
        if (has_vals) L.vals[at] = val[j];
      }
    }
    for (int i = lane; i < 128; i += 64) ((uint32_t*)&L.wcount[w][0])[i] = 0;  // (the wave's own counters)
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
      if (valid(j)) {
        key[j] = L.keys[small_pos<ITEMS>(j)];
        if (has_vals) val[j] = L.vals[small_pos<ITEMS>(j)];
      }
    }
    // (the next pass writes keys and vals after two barriers)
  }
}

}  // namespace dbvh
