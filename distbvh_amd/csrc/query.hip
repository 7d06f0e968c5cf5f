// query.hip -- broadphase and narrowphase traversal on gfx950.
//
//  * k_narrow64s / k_narrow64 / k_narrow32: one lane per query element (the
//    query object's leaves in its sorted order, so a wave holds 64 spatially
//    adjacent elements).  The wave walks the other object's tree with a
//    wave-uniform node: each internal node's record holds both children's
//    slabs, so one memory round trip tests two nodes; leaf children are
//    tested at once and internal children that some lane overlaps go on a
//    per-wave LDS stack.  Records arrive in scalar registers (k_narrow32,
//    k_narrow64s) or, K at a time, staged in LDS (k_narrow64).
//    Hits are staged per wave in LDS and appended with one atomic per flush.
//    Replaces query_tree / query_node_impl (collision_query.hpp:166-213) as
//    used by a narrowphase functor per patch pair, and self_collision_set
//    (collision_query.hpp:331-368) in self mode (each unordered pair once).
//  * k_patch_pairs: one lane per pair of patches, testing the two patch
//    k-DOPs (start_broadphase, collision_object/broadphase.cpp:68-119, which
//    walks the other object's patch-level tree to the same set).
#include "device.hpp"
#include "kernels.hpp"

namespace dbvh {

__device__ __forceinline__ void emit(const PairOut& out, bool pred, uint64_t key) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const int leader = __ffsll((long long)m) - 1;
  unsigned long long base = 0;
  if ((int)lane_id() == leader) base = atomicAdd(out.count, (unsigned long long)__popcll(m));
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)base, leader);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(base >> 32), leader);
  base = ((unsigned long long)hi << 32) | lo;
  if (pred) {
    const unsigned long long idx = base + (unsigned long long)__popcll(m & lanemask_lt());
    if (idx < out.cap) out.pairs[idx] = key;
  }
}

__device__ __forceinline__ uint64_t pair_key(uint32_t a, uint32_t b, bool self) {
  if (self && b < a) {
    const uint32_t t = a;
    a = b;
    b = t;
  }
  return ((uint64_t)a << 32) | b;
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ void empty_slabs(double* k) {
#pragma unroll
  for (int a = 0; a < kAxes; ++a) {
    k[2 * a] = __builtin_inf();
    k[2 * a + 1] = -__builtin_inf();
  }
}

// Per-wave pair staging in LDS: hits are appended with a ballot (all lanes of
// the wave are converged in the uniform traversal loop) and written to
// global memory in coalesced runs with one atomic per flush.
constexpr uint32_t kWaveBuf = 512;

__device__ __forceinline__ void wave_flush(uint64_t* buf, uint32_t& fill, const PairOut& out) {
  if (fill == 0) return;
  __builtin_amdgcn_wave_barrier();
  unsigned long long base = 0;
  if (lane_id() == 0) base = atomicAdd(out.count, (unsigned long long)fill);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
  base = ((unsigned long long)hi << 32) | lo;
  for (uint32_t i = lane_id(); i < fill; i += kWave)
    if (base + i < out.cap) out.pairs[base + i] = buf[i];
  __builtin_amdgcn_wave_barrier();
  fill = 0;
}

// End of a kernel whose waves all reach this point together (every thread of
// the block calls it): the block's waves append their staged pairs with one
// atomic for the whole block (the pair counter is one address; its atomics
// are serialized, about 12 ns each).
__device__ __forceinline__ void block_flush(uint64_t* buf, uint32_t fill, const PairOut& out) {
  __shared__ uint32_t s_fill[256 / kWave];
  __shared__ unsigned long long s_base;
  const uint32_t wv = threadIdx.x / kWave, nw = blockDim.x / kWave;
  if (lane_id() == 0) s_fill[wv] = fill;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (uint32_t v = 0; v < nw; ++v) tot += s_fill[v];
    s_base = tot ? atomicAdd(out.count, (unsigned long long)tot) : 0ull;
  }
  __syncthreads();
  unsigned long long base = s_base;
  for (uint32_t v = 0; v < wv; ++v) base += s_fill[v];
  for (uint32_t i = lane_id(); i < fill; i += kWave)
    if (base + i < out.cap) out.pairs[base + i] = buf[i];
}

__device__ __forceinline__ void wave_emit(uint64_t* buf, uint32_t& fill, const PairOut& out, bool pred,
                                          uint64_t key) {
  const uint64_t m = __ballot(pred);
  if (m == 0) return;
  const uint32_t cnt = (uint32_t)__popcll(m);
  if (fill + cnt > kWaveBuf) wave_flush(buf, fill, out);
  if (pred) buf[fill + (uint32_t)__popcll(m & lanemask_lt())] = key;
  fill += cnt;
}

// fp32-outward form.  Node slabs are fp32 in the frame of their object's
// origin P, rounded outward, so an fp32 miss proves an fp64 miss: with q, t the exact slabs and f(.) the rounded ones,
// q_lo < t_hi implies f(q_lo) <= q_lo - P < t_hi - P <= f(t_hi).  The query's
// slabs are its own fp32 leaf slabs.
//
// A leaf that passes the fp32 test is a candidate.  The rounding is also
// bounded from the inside: a leaf slab f = next_down(rn(fl64(x - P))) has
// x - P < next_up(next_up(f)) (rn moves by at most half an ulp and fl64 by far
// less), and likewise for upper slabs.  The records hold the ordered-integer
// images ord32() of the fp32 slabs, where next_up adds one and integer
// compares order like float compares, so ord(f(t_hi)) - ord(f(q_lo)) > 6 on
// a slab pair proves q_lo < t_hi in fp64, and both the overlap test and this
// bound are integer compares against scalar registers.  Candidates proven on every
// slab are emitted; the rest go to a re-check list whose pairs are tested on
// fp64 k-DOPs recomputed from element data (k_recheck).  The pairs are
// exactly those of the fp64 form.
//
// The tree is stored as child-pair records: visiting an internal node loads
// both children's slabs with one round of scalar loads, tests both, handles
// leaf children at once and pushes the internal children some lane overlaps
// on a per-wave LDS stack (left on top: depth-first order).
typedef __attribute__((address_space(4))) const Rec32 CRec32;
typedef __attribute__((address_space(4))) const int32_t CInt;

constexpr int32_t kInnerUlps = 6;

// stack entries per wave: above the height of any radix tree over the
// augmented keys (14 patch bits + 63 code bits + 30 position bits)
constexpr uint32_t kStack = 128;

// A walk of the fp32 records over a tree of 2..kFrontierMax patches starts at
// the patch roots whose slabs overlap the union of the wave's query slabs
// (one 26-compare test per patch, each lane testing every 64th patch) instead
// of at the root: the visits above the patch roots are saved (on 2 x 2M
// triangles in 256 patches, 32 of 200 per wave).  A wave's
// queries are 64 consecutive positions of their own tree, so the union is
// small and overlaps few patches.
constexpr uint32_t kFrontierMax = 256;
constexpr uint32_t kFrontierWords = kFrontierMax / kWave;
constexpr uint32_t kFrontierPush = 32;

// Minimum / maximum of v over the wave (every lane active), in a scalar
// register: DPP within each row of 16 lanes (quad_perm [1,0,3,2], [2,3,0,1],
// row_ror 4, 8), then row_bcast 15 and 31 carry the rows' results to lane 63.
template <bool MAX>
__device__ __forceinline__ int32_t wave_reduce_i32(int32_t v) {
  auto op = [](int32_t x, int32_t y) { return MAX ? max(x, y) : min(x, y); };
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x124, 0xF, 0xF, false));
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x128, 0xF, 0xF, false));
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xA, 0xF, false));
  v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xC, 0xF, false));
  return __builtin_amdgcn_readlane(v, 63);
}


// Smallest gap over the 13 slab pairs between query q and box b, in ordered
// fp32 images: min(b_hi - q_lo, q_hi - b_lo) with saturating subtraction
// (which keeps every sign).  The boxes overlap strictly iff the gap is > 0,
// and the fp64 overlap of the exact slabs is proven iff it is > kInnerUlps.
template <typename P>
__device__ __forceinline__ int32_t min_gap(const int32_t* q, P b) {
  int32_t m = 0x7fffffff;
#pragma unroll
  for (int a = 0; a < kAxes; ++a) {
    const int32_t d1 = __builtin_elementwise_sub_sat(b[2 * a + 1], q[2 * a]);
    const int32_t d2 = __builtin_elementwise_sub_sat(q[2 * a + 1], b[2 * a]);
    m = min(m, min(d1, d2));
  }
  return m;
}

// The same v_cmpx chain on ordered fp32 images (int32 compares): the strict
// overlap of the lane's query slabs with one wave-uniform box, for internal
// children of the fp32 walk (a leaf child needs the gap, min_gap).  Returns
// the mask of the lanes that hit (EXEC after the chain; every lane of the
// wave is active in the walk), which stays in scalar registers: an internal
// child only needs to know whether any lane hits it.  Every second box is missed
// by all lanes, mostly on x, y or z: the chain ends there if no lane is left
// (walk of 2 x 2M triangles 1,149 -> 1,086 us; leaving after one axis, or at more
// places, gains less or nothing).
__device__ __forceinline__ uint64_t box_mask32(const int32_t* q, const int32_t* b) {
  unsigned long long res, save, m;
  asm volatile(
      "s_mov_b64 %[save], exec\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q0], %[b1]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b0], %[q1]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q2], %[b3]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b2], %[q3]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q4], %[b5]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b4], %[q5]\n\t"
      "s_nop 4\n\t"
      "s_cbranch_execz .Lmiss%=\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q6], %[b7]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b6], %[q7]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q8], %[b9]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b8], %[q9]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q10], %[b11]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b10], %[q11]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q12], %[b13]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b12], %[q13]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q14], %[b15]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b14], %[q15]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q16], %[b17]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b16], %[q17]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q18], %[b19]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b18], %[q19]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q20], %[b21]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b20], %[q21]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q22], %[b23]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b22], %[q23]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[q24], %[b25]\n\t"
      "v_cmpx_lt_i32_e64 %[m], %[b24], %[q25]\n\t"
      "s_nop 4\n"
      ".Lmiss%=:\n\t"
      "s_mov_b64 %[res], exec\n\t"
      "s_mov_b64 exec, %[save]\n\t"
      : [res] "=&s"(res), [save] "=&s"(save), [m] "=&s"(m)
      : [q0] "v"(q[0]), [q1] "v"(q[1]), [q2] "v"(q[2]), [q3] "v"(q[3]), [q4] "v"(q[4]), [q5] "v"(q[5]), [q6] "v"(q[6]), [q7] "v"(q[7]), [q8] "v"(q[8]), [q9] "v"(q[9]), [q10] "v"(q[10]), [q11] "v"(q[11]), [q12] "v"(q[12]), [q13] "v"(q[13]), [q14] "v"(q[14]), [q15] "v"(q[15]), [q16] "v"(q[16]), [q17] "v"(q[17]), [q18] "v"(q[18]), [q19] "v"(q[19]), [q20] "v"(q[20]), [q21] "v"(q[21]), [q22] "v"(q[22]), [q23] "v"(q[23]), [q24] "v"(q[24]), [q25] "v"(q[25]),
        [b0] "s"(b[0]), [b1] "s"(b[1]), [b2] "s"(b[2]), [b3] "s"(b[3]), [b4] "s"(b[4]), [b5] "s"(b[5]), [b6] "s"(b[6]), [b7] "s"(b[7]), [b8] "s"(b[8]), [b9] "s"(b[9]), [b10] "s"(b[10]), [b11] "s"(b[11]), [b12] "s"(b[12]), [b13] "s"(b[13]), [b14] "s"(b[14]), [b15] "s"(b[15]), [b16] "s"(b[16]), [b17] "s"(b[17]), [b18] "s"(b[18]), [b19] "s"(b[19]), [b20] "s"(b[20]), [b21] "s"(b[21]), [b22] "s"(b[22]), [b23] "s"(b[23]), [b24] "s"(b[24]), [b25] "s"(b[25]));
  return res;
}

// Per-wave LDS staging of the candidates queued for the fp64 re-check: one
// atomic on the wave's stripe counter per flush (mesh self collision queues
// every pair of elements that share a vertex, so these are many).
constexpr uint32_t kRecheckBuf = 128;

__device__ __forceinline__ void recheck_flush(uint64_t* buf, uint32_t& fill, const PairOut& out, uint32_t stripe) {
  if (fill == 0) return;
  __builtin_amdgcn_wave_barrier();
  unsigned long long base = 0;
  if (lane_id() == 0) base = atomicAdd(out.rcount + (uint64_t)stripe * kRecheckStride, (unsigned long long)fill);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
  base = ((unsigned long long)hi << 32) | lo;
  uint64_t* list = out.recheck + (uint64_t)stripe * out.rcap;
  for (uint32_t i = lane_id(); i < fill; i += kWave)
    if (base + i < out.rcap) list[base + i] = buf[i];
  __builtin_amdgcn_wave_barrier();
  fill = 0;
}

// Queries in a row per XCD.  One eighth of them for each XCD left some XCDs
// idle while others still walked: work differs between parts of a scene, and
// the start of a self walk meets more than its end.  With 1,024 queries in turn
// the 2 x 2M walk takes 933 us instead of 1,038 (931 / 947 with 4,096 / 16,384 in
// a row), the 512-mesh walk 1,215 instead of 1,259 (1,256 / 1,310), the 2 x 524k
// walk over fp64 records 433 instead of 474; tiles that share lines still run on
// one XCD.
constexpr uint32_t kXcdQueries = 1024;

// The self walks take CROSS = true for cross-patch self collision: a lane
// skips every child whose position range lies inside its own patch's range
// [pb, pe) (patches are contiguous position ranges of the tree order), so
// pairs within one patch are neither tested nor emitted.
__device__ __forceinline__ void own_patch_range(const TreeView& q, uint32_t qa, bool valid, uint32_t n, uint32_t& pb,
                                                uint32_t& pe) {
  pb = 0;
  pe = 0;
  if (!valid) return;
  const uint32_t k = q.patch_of_input[qa];
  pb = k == 0 ? 0u : q.splits[k - 1];
  pe = (uint64_t)k + 1 >= q.od ? n : q.splits[k];
}

// A lane's query: the slabs (ord32 images, in the frame of the tree t), input
// index and position of position p of the query object's order.
struct Query32 {
  int32_t s[kSlabs];
  uint32_t elem, pos;  // (0 for a lane without a query, which hits nothing)
  bool valid;
};
template <bool SELF>
__device__ __forceinline__ void load_query32(const TreeView& q, const TreeView& t, uint64_t p, bool valid,
                                             Query32& r) {
  r.valid = valid;
  r.elem = 0;
  r.pos = valid ? (uint32_t)p : 0u;  // positions fit 32 bits
  if (valid) {
    // this leaf's slabs: its half of its parent's record (the root's array if n = 1)
    const int32_t* src = q.rootbox32;
    if (q.n > 1) {
      uint32_t parent;
      int side;
      leaf_slot(q.delta, q.n, p, parent, side);
      src = q.rec32[parent].h[side].box;
    }
#pragma unroll
    for (int a = 0; a < kAxes; ++a) {
      const int2 v = ((const int2*)src)[a];
      r.s[2 * a] = v.x;
      r.s[2 * a + 1] = v.y;
    }
    r.elem = q.perm[p];
    // another object's tree has its own frame: the slabs moved to it, still
    // outward (their fp32 rounding then bounds nothing from the inside, so
    // every candidate of such a query is decided in fp64)
    if (!SELF && q.origin != t.origin)
      reframe32(r.s, q.origin[0], q.origin[1], q.origin[2], t.origin[0], t.origin[1], t.origin[2]);
  } else {
#pragma unroll
    for (int a = 0; a < kAxes; ++a) {  // the empty box overlaps nothing
      r.s[2 * a] = 0x7fffffff;
      r.s[2 * a + 1] = (int32_t)0x80000000;
    }
  }
}

// What a wave does with its queries: the whole walk; the walk's top, leaving
// subtrees of at most kItemLeaves leaves to a second launch as items of the
// split list ((wave << 32) | subtree root) once it has made kItemBudget visits;
// or a run of such items.  The cross-patch walk is split: where meshes of
// uneven sizes meet, a coarse element overlaps thousands of a fine mesh's, and
// its wave alone (7,700 visits among 213 on average over 512 meshes of
// lognormal size) held the launch for 4,577 us.  Split, it took 1,465 + 1,092
// (and takes 1,215 + 1,020 by the order of the waves and the early out);
// with 128 or 64 visits before the split, or 32 or 128 leaves an item, 2,536 to
// 2,661 us.  Evenly loaded walks lose by it (contact of 2 x 2M triangles 1,158
// -> 1,271 us: the split's registers cost every visit) and stay whole.
constexpr int kWalkWhole = 0, kWalkTop = 1, kWalkItems = 2;
constexpr uint32_t kItemBuf = 32;  // staged items per wave
constexpr uint32_t kItemBudget = 256;
constexpr uint32_t kItemLeaves = 64;
constexpr unsigned kItemBlocks = 4 * 1792;  // seven waves a SIMD

// Appends the wave's n staged subtree roots to the split list; returns how
// many found room (the list is sized by the queries, not by the data: the wave
// walks the others itself).
__device__ __forceinline__ uint32_t items_flush(const uint32_t* ibuf, uint32_t n, uint32_t wave, const PairOut& out) {
  if (n == 0) return 0;
  __builtin_amdgcn_wave_barrier();
  unsigned long long base = 0;
  if (lane_id() == 0) base = atomicAdd(out.icount, (unsigned long long)n);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
  base = ((unsigned long long)hi << 32) | lo;
  const uint32_t room = base >= out.icap ? 0u : (uint32_t)(out.icap - base < n ? out.icap - base : n);
  if (lane_id() < room) out.items[base + lane_id()] = ((uint64_t)wave << 32) | ibuf[lane_id()];
  __builtin_amdgcn_wave_barrier();
  return room;
}

// The fp32-outward record walk of one wave (the body of k_narrow32 and of its
// batched and item forms): the qper queries from position wave * qper on, one
// lane each, or, as kWalkItems, the items [i0, i1) of the split list; buf /
// rbuf / stk / ibuf are the wave's LDS pair staging, re-check staging, stack
// and item staging.  Leaf candidates with a gap above `inner` are emitted, the
// rest queued for the fp64 re-check, in stripe rstripe (items: that of the wave
// they come from, so that a stripe's length is the same in every run, whoever
// walks an item and in whatever order the list was filled).
template <bool SELF, bool CROSS, int MODE>
__device__ __forceinline__ void walk32(const TreeView& q, const TreeView& t, uint32_t wave, uint32_t qper, uint64_t i0,
                                       uint64_t i1, const PairOut& out, int32_t inner, uint64_t* buf, uint64_t* rbuf,
                                       uint32_t* stk, uint32_t* ibuf, uint32_t rstripe) {
  uint32_t fill = 0, rfill = 0;
  if (!SELF && q.origin != t.origin) inner = 0x7fffffff;
  uint64_t item = MODE == kWalkItems ? out.items[i0] : 0;
  if (MODE == kWalkItems) {
    wave = uniform((uint32_t)(item >> 32));
    rstripe = wave % kRecheckStripes;
  }
  Query32 Q;
  uint64_t p0 = (uint64_t)wave * qper + lane_id();
  load_query32<SELF>(q, t, p0, lane_id() < qper && p0 < q.n, Q);
  const uint32_t n = (uint32_t)t.n;
  const uint32_t tleaf0 = n - 1;
  const uint32_t lane = lane_id();
  uint32_t pb = 0, pe = 0;
  if (CROSS) own_patch_range(q, Q.elem, Q.valid, n, pb, pe);
  CRec32* recs = (CRec32*)t.rec32;
  uint32_t sink = 0, pf = 0;  // record prefetch (below)
  uint32_t steps = 0, total = 0;
  uint32_t ncand = 0;
  // fp32 candidates at one (wave-uniform) leaf, gap g per lane: emit what
  // the inner bound proves, queue the rest for the fp64 re-check
  auto leaf_check = [&](int32_t g, uint32_t elem, bool h) {
    const uint64_t m = __ballot(h);
    if (m == 0) return;
    ncand += (uint32_t)__popcll(m);
    const bool sure = h & (g > inner);
    const uint64_t key = pair_key(Q.elem, elem, SELF);
    wave_emit(buf, fill, out, sure, key);
    const bool unsure = h & !sure;
    const uint64_t mu = __ballot(unsure);
    if (mu != 0) {
      const uint32_t cnt = (uint32_t)__popcll(mu);
      if (rfill + cnt > kRecheckBuf) recheck_flush(rbuf, rfill, out, rstripe);
      if (unsure) rbuf[rfill + (uint32_t)__popcll(mu & lanemask_lt())] = key;
      rfill += cnt;
    }
  };
  // the node to visit next (kEnd: pop the stack)
  uint32_t x = kEnd;
  uint32_t sp = 0;
  const uint32_t od = (uint32_t)t.od;
  bool from_root = true;
  // (not in the cross-patch self walk: its workloads have many patches, and
  // the start's registers would cost that kernel a wave per SIMD)
  if (MODE != kWalkItems && !CROSS && t.patch_box32 != nullptr && n > 1 && od > 1 && od <= kFrontierMax) {
    // self: patches that end at or before the wave's first position hold no
    // pair of it
    const uint32_t pmin = __builtin_amdgcn_readlane(Q.pos, 0);
    // lane l tests patches l, l + 64, ... (clamped to the last patch, with
    // the test off); the union is reduced one axis at a time, so that it
    // takes two scalar registers and each axis's loads go out together
    uint32_t kk[kFrontierWords];
    bool h[kFrontierWords];
#pragma unroll
    for (uint32_t w = 0; w < kFrontierWords; ++w) {
      const uint32_t k = w * kWave + lane;
      kk[w] = (k < od ? k : od - 1) & (kFrontierMax - 1);  // (the mask: a 32-bit load offset)
      h[w] = (k < od) & (t.patch_root[kk[w]] != kEnd);
      if (SELF) h[w] = h[w] & ((kk[w] + 1 >= od ? n : t.splits[kk[w]]) > pmin + 1);
    }
#pragma unroll
    for (int a = 0; a < kAxes; ++a) {
      const int32_t ulo = wave_reduce_i32<false>(Q.s[2 * a]), uhi = wave_reduce_i32<true>(Q.s[2 * a + 1]);
      const int32_t* plo = t.patch_box32 + (uint64_t)(2 * a) * od;  // this axis's slabs of every patch
      const int32_t* phi = plo + od;
#pragma unroll
      for (uint32_t w = 0; w < kFrontierWords; ++w) {
        if (w * kWave >= od) break;
        h[w] = h[w] & (ulo < phi[kk[w]]) & (plo[kk[w]] < uhi);
      }
    }
    uint32_t cnt = 0;
#pragma unroll
    for (uint32_t w = 0; w < kFrontierWords; ++w) cnt += (uint32_t)__popcll(__ballot(h[w]));
    // the patch roots hit go on the stack; within one patch's subtree the
    // walk stacks fewer than 96 entries (its height is below the 93 key bits
    // under the patch bits), so kFrontierPush roots leave the stack room; a
    // wave hitting more patches starts at the root
    if (cnt <= kFrontierPush) {
      from_root = false;
      uint32_t leafm = 0;  // bit w: this lane's patch of round w is one element, hit
#pragma unroll
      for (uint32_t w = 0; w < kFrontierWords; ++w) {
        const uint32_t r = h[w] ? t.patch_root[kk[w]] : kEnd;
        const bool in = h[w] & (r < tleaf0);
        const uint64_t mi = __ballot(in);
        if (in) stk[sp + (uint32_t)__popcll(mi & lanemask_lt())] = r;
        sp += (uint32_t)__popcll(mi);
        leafm |= (uint32_t)(h[w] & (r >= tleaf0)) << w;
      }
      // a patch of one element: its leaf is tested here
      uint64_t lm = __ballot(leafm != 0);
      while (lm != 0) {
        const uint32_t j = (uint32_t)__builtin_ctzll(lm);
        lm &= lm - 1;
        uint32_t bits = __builtin_amdgcn_readlane(leafm, j);
        while (bits != 0) {
          const uint32_t k = (uint32_t)__builtin_ctz(bits) * kWave + j;
          bits &= bits - 1;
          const uint32_t pos = uniform(t.patch_root[k]) - tleaf0;
          if (pos >= n) {
            if (lane == 0) atomicOr(t.status, kErrTraverse);
            continue;
          }
          int32_t bx[kSlabs];
#pragma unroll
          for (int a = 0; a < kSlabs; ++a) bx[a] = t.patch_box32[(uint64_t)a * od + k];
          const int32_t g = min_gap(Q.s, bx);
          bool hit = g > 0;
          if (SELF) hit = hit & (pos > Q.pos);
          leaf_check(g, uniform(t.perm[pos]), hit);
        }
      }
    }
  }
  if (MODE == kWalkItems) {
    x = uniform((uint32_t)item);
  } else if (from_root) {
    const int32_t g = min_gap(Q.s, (CInt*)t.rootbox32);
    bool h = g > 0;
    if (SELF) h = h & ((n - 1) > Q.pos);  // the root's last position
    if (n == 1) {
      if (!SELF) leaf_check(g, uniform(t.perm[0]), h);
    } else if (__ballot(h) != 0) {
      x = uniform(*t.root);
    }
  }
  // kWalkTop: staged items; once the list is full, the first of them left to
  // this wave (else kEnd: still splitting)
  uint32_t nitem = 0, kept = kEnd;
  for (;;) {
    if (x == kEnd) {
      if (sp != 0) {
        x = uniform(stk[--sp]);
      } else if (MODE == kWalkItems) {
        if (++i0 >= i1) break;
        item = out.items[i0];
        if (uniform((uint32_t)(item >> 32)) != wave) {  // another wave's queries
          recheck_flush(rbuf, rfill, out, rstripe);
          wave = uniform((uint32_t)(item >> 32));
          rstripe = wave % kRecheckStripes;
          p0 = (uint64_t)wave * qper + lane;
          load_query32<SELF>(q, t, p0, lane < qper && p0 < q.n, Q);
          if (CROSS) own_patch_range(q, Q.elem, Q.valid, n, pb, pe);
        }
        x = uniform((uint32_t)item);
        steps = 0;  // (visits of earlier items: total)
      } else if (MODE == kWalkTop && nitem != 0) {
        if (kept == kEnd) {  // the walk is done but for its staged items
          kept = items_flush(ibuf, nitem, wave, out);
        }
        if (kept >= nitem) break;
        x = uniform(ibuf[kept++]);
      } else {
        break;
      }
    }
    if (MODE == kWalkItems) ++total;
    if (x >= tleaf0 || ++steps > n) {
      if (lane == 0) atomicOr(t.status, kErrTraverse);
      break;
    }
    // both halves' slabs, child ids and leaf elements (the first 112 bytes of
    // each 128-byte half) and `last`: every scalar load issued before any is
    // used, one memory round trip per visit
    CInt* rp = (CInt*)(recs + x);
    int32_t rw[56];
#pragma unroll
    for (int k = 0; k < 28; ++k) rw[k] = rp[k];
#pragma unroll
    for (int k = 0; k < 28; ++k) rw[28 + k] = rp[32 + k];
    const uint32_t rlast = SELF ? recs[x].h[0].last : 0u;
    const uint32_t rfirst = CROSS ? recs[x].h[0].first : 0u;
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t cl = (uint32_t)rw[26], cr = (uint32_t)rw[54];
    const uint32_t el = (uint32_t)rw[27], er = (uint32_t)rw[55];
    // internal children: overlap only (v_cmpx chain); leaf children: the gap,
    // which also decides whether fp32 proves the fp64 overlap
    const bool leaf_l = cl >= tleaf0, leaf_r = cr >= tleaf0;
    // The next record the walk loads is one of these children's (or one it
    // pushed earlier).  The lanes load a word of each 128-byte line of both
    // children's records (lanes 4j + 0, 1: the left child, 4j + 2, 3: the
    // right; a leaf child's lanes read this record again), so the lines are
    // on their way to L2 while this record is tested; the words feed a sink
    // that nothing reads.  Every lane loads: no branch around the load.
    {
      sink += pf;
      uint32_t c = (lane & 2) ? cr : cl;
      c = c < tleaf0 ? c : x;
      pf = ((const uint32_t*)(recs + c))[(lane & 1) * 32];
    }
    // per lane, whether a child may hold its pairs at all: position bounds
    // (self) and the own patch (cross), non-short-circuit &: no branch
    bool okl = true, okr = true;
    if (SELF) {
      okl = x > Q.pos;  // the left child ends at position x
      okr = rlast > Q.pos;
    }
    if (CROSS) {  // children [rfirst, x] and [x + 1, rlast] inside the lane's own patch
      okl = okl & !((rfirst >= pb) & (x < pe));
      okr = okr & !((x + 1 >= pb) & (rlast < pe));
    }
    // the lanes hitting each child, as scalar masks (the v_cmpx chain tests
    // the same strict overlap as gap > 0); a leaf child that some lane hits
    // also gets each lane's gap for the candidate test (both gaps before
    // either test, so the record's registers are free by then)
    int32_t gl = 0, gr = 0;
    uint64_t ml = box_mask32(Q.s, rw), mr = box_mask32(Q.s, rw + 28);
    if (SELF || CROSS) {
      ml &= __ballot(okl);
      mr &= __ballot(okr);
    }
    if (leaf_l && ml != 0) gl = min_gap(Q.s, rw);
    if (leaf_r && mr != 0) gr = min_gap(Q.s, rw + 28);
    const bool any_l = ml != 0, any_r = mr != 0;
    if (any_l && leaf_l) leaf_check(gl, el, (gl > 0) & okl & (!SELF || (cl - tleaf0 > Q.pos)));
    if (any_r && leaf_r) leaf_check(gr, er, (gr > 0) & okr & (!SELF || (cr - tleaf0 > Q.pos)));
    bool go_l = any_l && !leaf_l, go_r = any_r && !leaf_r;
    if (MODE == kWalkTop && steps > kItemBudget && kept == kEnd) {
      // children of few leaves become items (this node's range: half 0)
      const uint32_t first = recs[x].h[0].first, last = recs[x].h[0].last;
      if (go_l && x - first < kItemLeaves) {
        ibuf[nitem++] = cl;
        go_l = false;
      }
      if (go_r && last - x <= kItemLeaves) {
        ibuf[nitem++] = cr;
        go_r = false;
      }
      if (nitem + 2 > kItemBuf) {
        const uint32_t room = items_flush(ibuf, nitem, wave, out);
        if (room < nitem) kept = room;
        else nitem = 0;
      }
    }
    // depth first: continue with the left child, keep the right one
    if (go_l && go_r) {
      if (sp >= kStack) {
        if (lane == 0) atomicOr(t.status, kErrTraverse);
        break;
      }
      stk[sp++] = cr;
      x = cl;
    } else {
      x = go_l ? cl : (go_r ? cr : kEnd);
    }
  }
  wave_flush(buf, fill, out);
  recheck_flush(rbuf, rfill, out, rstripe);
  sink += pf;
  asm volatile("; record prefetch sink %0" ::"v"(sink));  // keeps the prefetch loads
  // the counts go to a stripe's line, the block's (neighbours on one line queue:
  // those of items by their own wave's took the 512-mesh step from 3,345 to
  // 3,368 us), and k_recheck adds the lines up
  if (lane == 0) {
    unsigned long long* line = out.rcount + (uint64_t)(blockIdx.x % kRecheckStripes) * kRecheckStride;
    atomicAdd(line + 1, (unsigned long long)(MODE == kWalkItems ? total : steps));
    atomicAdd(line + 2, (unsigned long long)ncand);
  }
}

// One wave per block: a wave's slot is free for the next one as soon as it
// ends, not when the slowest of its block does (walk of 2 x 2M triangles
// 1,085 -> 1,040 us, of 512 meshes across patches 1,440 -> 1,260).
struct Walk32Lds {
  uint64_t buf[kWaveBuf];
  uint64_t rbuf[kRecheckBuf];
  uint32_t stack[kStack];
};

template <bool SELF, bool CROSS, int MODE = kWalkWhole>
__global__ __launch_bounds__(kWave) void k_narrow32(TreeView q, TreeView t, int xcd, uint32_t qper, PairOut out,
                                                    int32_t inner) {
  __shared__ Walk32Lds L;
  __shared__ uint32_t s_items[MODE == kWalkTop ? kItemBuf : 1];
  const uint32_t wave = xcd ? xcd_group_tile(blockIdx.x, gridDim.x, kXcdQueries / qper) : blockIdx.x;
  walk32<SELF, CROSS, MODE>(q, t, wave, qper, 0, 0, out, inner, L.buf, L.rbuf, L.stack, s_items,
                            wave % kRecheckStripes);
}

// The split list of a query: a contiguous run of items per wave (items of one
// wave's queries are neighbours, which share the loaded queries).
template <bool SELF, bool CROSS>
__global__ __launch_bounds__(kWave) void k_narrow32_items(TreeView q, TreeView t, uint32_t qper, PairOut out,
                                                          int32_t inner) {
  __shared__ Walk32Lds L;
  const unsigned long long c = *out.icount;
  const uint64_t cnt = c < out.icap ? c : out.icap;
  const uint64_t per = (cnt + gridDim.x - 1) / gridDim.x;
  const uint64_t i0 = blockIdx.x * per, i1 = i0 + per < cnt ? i0 + per : cnt;
  if (i0 >= i1) return;
  walk32<SELF, CROSS, kWalkItems>(q, t, 0, qper, i0, i1, out, inner, L.buf, L.rbuf, L.stack, nullptr, 0);
}

// Several queries (object pairs) in one launch of the fp32-outward walk: four
// waves for each of the table's blocks of 256 queries, in the order above;
// block b belongs to the query whose [block0, block0 + blocks) holds it (a
// wave-uniform binary search over the table).
__global__ __launch_bounds__(kWave) void k_narrow32_batch(const BatchQuery* __restrict__ bq, uint32_t nq,
                                                          int32_t inner) {
  __shared__ Walk32Lds L;
  const uint32_t tile = xcd_group_tile(blockIdx.x, gridDim.x, kXcdQueries / kWave), b = tile / 4;
  uint32_t lo = 0, hi = nq;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (bq[mid].block0 <= b) lo = mid;
    else hi = mid;
  }
  const BatchQuery& e = bq[lo];
  if (b - e.block0 >= e.blocks) return;
  // (the stripe by the wave's number in its query: the blocks of one query's
  // waves, 8 apart within a turn, would reach half the stripes or fewer)
  const uint32_t wave = tile - 4 * e.block0;
  walk32<false, false, kWalkWhole>(e.q, e.t, wave, kWave, 0, 0, e.out, inner, L.buf, L.rbuf, L.stack, nullptr,
                                   wave % kRecheckStripes);
}

// Strict overlap of the lane's query slabs q with one box b whose 26 slabs
// are wave-uniform (scalar registers), as the AND of 26 fp64 compares chained
// with v_cmpx: each compare clears the EXEC bit of the lanes it fails (a
// lane already cleared stays cleared), so the AND accumulates in EXEC with no
// scalar instruction per compare.  EXEC is saved first and restored last;
// the caller runs it with every lane of the wave active.  Returns the wave's
// hit mask; *hit is the lane's bit.  `touch` are loads whose only purpose is
// to bring cache lines in: they are consumed here so that they are kept.
__device__ __forceinline__ uint64_t box_hits(const double* q, const double* b, uint32_t touch0, uint32_t touch1,
                                             bool* hit) {
  unsigned long long res, save, m;
  int v;
  asm volatile(
      "s_mov_b64 %[save], exec\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q0], %[b1]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b0], %[q1]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q2], %[b3]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b2], %[q3]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q4], %[b5]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b4], %[q5]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q6], %[b7]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b6], %[q7]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q8], %[b9]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b8], %[q9]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q10], %[b11]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b10], %[q11]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q12], %[b13]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b12], %[q13]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q14], %[b15]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b14], %[q15]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q16], %[b17]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b16], %[q17]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q18], %[b19]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b18], %[q19]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q20], %[b21]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b20], %[q21]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q22], %[b23]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b22], %[q23]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q24], %[b25]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b24], %[q25]\n\t"
      "s_nop 4\n\t"
      "s_mov_b64 %[res], exec\n\t"
      "s_mov_b64 exec, %[save]\n\t"
      "v_cndmask_b32_e64 %[v], 0, 1, %[res]\n\t"
      : [res] "=&s"(res), [save] "=&s"(save), [m] "=&s"(m), [v] "=&v"(v)
      : [q0] "v"(q[0]), [q1] "v"(q[1]), [q2] "v"(q[2]), [q3] "v"(q[3]), [q4] "v"(q[4]), [q5] "v"(q[5]), [q6] "v"(q[6]), [q7] "v"(q[7]), [q8] "v"(q[8]), [q9] "v"(q[9]), [q10] "v"(q[10]), [q11] "v"(q[11]), [q12] "v"(q[12]), [q13] "v"(q[13]), [q14] "v"(q[14]), [q15] "v"(q[15]), [q16] "v"(q[16]), [q17] "v"(q[17]), [q18] "v"(q[18]), [q19] "v"(q[19]), [q20] "v"(q[20]), [q21] "v"(q[21]), [q22] "v"(q[22]), [q23] "v"(q[23]), [q24] "v"(q[24]), [q25] "v"(q[25]),
        [b0] "s"(b[0]), [b1] "s"(b[1]), [b2] "s"(b[2]), [b3] "s"(b[3]), [b4] "s"(b[4]), [b5] "s"(b[5]), [b6] "s"(b[6]), [b7] "s"(b[7]), [b8] "s"(b[8]), [b9] "s"(b[9]), [b10] "s"(b[10]), [b11] "s"(b[11]), [b12] "s"(b[12]), [b13] "s"(b[13]), [b14] "s"(b[14]), [b15] "s"(b[15]), [b16] "s"(b[16]), [b17] "s"(b[17]), [b18] "s"(b[18]), [b19] "s"(b[19]), [b20] "s"(b[20]), [b21] "s"(b[21]), [b22] "s"(b[22]), [b23] "s"(b[23]), [b24] "s"(b[24]), [b25] "s"(b[25]),
        [t0] "s"(touch0), [t1] "s"(touch1));
  *hit = v != 0;
  return res;
}

// N axes of a box in LDS against the lane's query slabs, for the lanes in
// `mask`: the v_cmpx chain of box_hits.  Returns the lanes that hit.
template <int N>
__device__ __forceinline__ uint64_t box_part64(const double* q, const double* b, uint64_t mask);
template <>
__device__ __forceinline__ uint64_t box_part64<3>(const double* q, const double* b, uint64_t mask) {
  unsigned long long save, m, res = mask;
  asm volatile(
      "s_mov_b64 %[save], exec\n\t"
      "s_mov_b64 exec, %[res]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q0], %[b1]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b0], %[q1]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q2], %[b3]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b2], %[q3]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q4], %[b5]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b4], %[q5]\n\t"
      "s_nop 4\n\t"
      "s_mov_b64 %[res], exec\n\t"
      "s_mov_b64 exec, %[save]\n\t"
      : [res] "+s"(res), [save] "=&s"(save), [m] "=&s"(m)
      : [q0] "v"(q[0]), [q1] "v"(q[1]), [q2] "v"(q[2]), [q3] "v"(q[3]), [q4] "v"(q[4]), [q5] "v"(q[5]),
        [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]), [b4] "v"(b[4]), [b5] "v"(b[5]));
  return res;
}
template <>
__device__ __forceinline__ uint64_t box_part64<5>(const double* q, const double* b, uint64_t mask) {
  unsigned long long save, m, res = mask;
  asm volatile(
      "s_mov_b64 %[save], exec\n\t"
      "s_mov_b64 exec, %[res]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q0], %[b1]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b0], %[q1]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q2], %[b3]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b2], %[q3]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q4], %[b5]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b4], %[q5]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q6], %[b7]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b6], %[q7]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[q8], %[b9]\n\t"
      "v_cmpx_lt_f64_e64 %[m], %[b8], %[q9]\n\t"
      "s_nop 4\n\t"
      "s_mov_b64 %[res], exec\n\t"
      "s_mov_b64 exec, %[save]\n\t"
      : [res] "+s"(res), [save] "=&s"(save), [m] "=&s"(m)
      : [q0] "v"(q[0]), [q1] "v"(q[1]), [q2] "v"(q[2]), [q3] "v"(q[3]), [q4] "v"(q[4]), [q5] "v"(q[5]), [q6] "v"(q[6]), [q7] "v"(q[7]), [q8] "v"(q[8]), [q9] "v"(q[9]),
        [b0] "v"(b[0]), [b1] "v"(b[1]), [b2] "v"(b[2]), [b3] "v"(b[3]), [b4] "v"(b[4]), [b5] "v"(b[5]), [b6] "v"(b[6]), [b7] "v"(b[7]), [b8] "v"(b[8]), [b9] "v"(b[9]));
  return res;
}
// Both boxes of an LDS-staged fp64 record against the lane's query slabs.
// Every second box is missed by all lanes, mostly on x, y or z, so the other
// axes are read only if these leave a lane; in parts of five axes, so that ten
// doubles of the record are in registers at a time (92 VGPRs; parts of three or
// four axes take fewer, 86, but no more waves fit).  With all 13 axes read, and
// the compares ANDed in scalar registers, the walk of 2 x 524k triangles took
// 614 us instead of 474, of 2 x 8,192 121 instead of 92.
__device__ __forceinline__ void overlap_pair(const double* qk, const Rec64& r, uint64_t& m0, uint64_t& m1) {
  m0 = box_part64<3>(qk, r.box[0], ~0ull);
  m1 = box_part64<3>(qk, r.box[1], ~0ull);
  if (m0 != 0) {
    m0 = box_part64<5>(qk + 6, r.box[0] + 6, m0);
    if (m0 != 0) m0 = box_part64<5>(qk + 16, r.box[0] + 16, m0);
  }
  if (m1 != 0) {
    m1 = box_part64<5>(qk + 6, r.box[1] + 6, m1);
    if (m1 != 0) m1 = box_part64<5>(qk + 16, r.box[1] + 16, m1);
  }
}

// fp64 form: the same record walk, K records per memory round trip.  Two
// fp64 boxes (416 B) do not fit the scalar registers, so each 448-byte record
// is loaded into LDS by a direct-to-LDS load (28 lanes x 16 bytes, no VGPR
// staging, which keeps the walk at 80 VGPRs and six waves per SIMD for K = 2)
// and every lane reads both boxes as LDS broadcasts.  Each iteration pops up to K nodes
// off the wave's stack and issues all their loads before it tests any: the
// set of visited nodes does not depend on K (a node is visited when some lane
// overlaps it and its parent was visited), only the number of dependent
// round trips does.  Leaf tests are exact, so hits are emitted directly.
// The walk of one wave's qper queries (the body of k_narrow64 and of its
// batched form k_narrow64_batch); buf / stk / R are the wave's LDS pair
// staging, stack and record slots.
template <bool SELF, int K, bool CROSS>
__device__ __forceinline__ void walk64(const TreeView& q, const TreeView& t, uint32_t wave, uint32_t qper, const PairOut& out,
                                       uint64_t* buf, uint32_t* stk, Rec64* R) {
  uint32_t fill = 0;
  const uint64_t p = (uint64_t)wave * qper + lane_id();
  const bool valid = lane_id() < qper && p < q.n;
  double qk[kSlabs];
  uint32_t qa = 0;
  if (valid) {
    // this leaf's slabs: its half of its parent's record (the root's array if n = 1)
    const double* src = q.rootbox64;
    if (q.n > 1) {
      uint32_t parent;
      int side;
      leaf_slot(q.delta, q.n, p, parent, side);
      src = q.rec64[parent].box[side];
    }
#pragma unroll
    for (int a = 0; a < kAxes; ++a) {
      const double2 v = ((const double2*)src)[a];
      qk[2 * a] = v.x;
      qk[2 * a + 1] = v.y;
    }
    qa = q.perm[p];
  } else {
    empty_slabs(qk);
  }
  const uint32_t n = (uint32_t)t.n;
  const uint32_t tleaf0 = n - 1;
  const uint32_t lane = lane_id();
  const uint32_t p32 = valid ? (uint32_t)p : 0u;  // positions fit 32 bits; invalid lanes hit nothing
  uint32_t pb = 0, pe = 0;
  if (CROSS) own_patch_range(q, qa, valid, n, pb, pe);
  uint32_t steps = 0;
  uint32_t sp = 0;
  {
    // the root's slabs through scalar loads (wave-uniform)
    const __attribute__((address_space(4))) double* rb = (const __attribute__((address_space(4))) double*)t.rootbox64;
    bool h = true;
#pragma unroll
    for (int a = 0; a < kAxes; ++a) h = h & (qk[2 * a] < rb[2 * a + 1]) & (rb[2 * a] < qk[2 * a + 1]);
    if (SELF) h = h && (uint64_t)(n - 1) > p;  // the root's last position
    if (n == 1) {
      if (!SELF) wave_emit(buf, fill, out, h, pair_key(qa, uniform(t.perm[0]), SELF));
    } else if (__ballot(h) != 0) {
      stk[0] = uniform(*t.root);
      sp = 1;
    }
  }
  while (sp != 0) {
    const uint32_t m = sp < (uint32_t)K ? sp : (uint32_t)K;
    uint32_t xs[K];
#pragma unroll
    for (int k = 0; k < K; ++k) xs[k] = (uint32_t)k < m ? uniform(stk[sp - 1 - k]) : 0u;
    sp -= m;
    steps += m;
    bool bad = steps > n;
#pragma unroll
    for (int k = 0; k < K; ++k) bad = bad || ((uint32_t)k < m && xs[k] >= tleaf0);
    if (bad) {
      if (lane == 0) atomicOr(t.status, kErrTraverse);
      break;
    }
    {
      // every record straight from memory into its LDS slot (the loads
      // write LDS directly, so no VGPRs hold them in between): lanes 0..27
      // each bring 16 bytes, which land at the slot + 16 x lane
#pragma unroll
      for (int k = 0; k < K; ++k)
        if ((uint32_t)k < m && lane < sizeof(Rec64) / 16)
          __builtin_amdgcn_global_load_lds((const void*)((const char*)(t.rec64 + xs[k]) + lane * 16),
                                           (void __attribute__((address_space(3)))*)&R[k], 16, 0, 0);
      __builtin_amdgcn_s_waitcnt(0);  // the LDS writes of those loads are done
      asm volatile("" ::: "memory");
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if ((uint32_t)k < m) {
        const Rec64& Rk = R[k];
        const uint32_t cl = uniform(Rk.child[0]), cr = uniform(Rk.child[1]);
        const uint32_t el = uniform(Rk.elem[0]), er = uniform(Rk.elem[1]);
        uint64_t ml, mr;
        overlap_pair(qk, Rk, ml, mr);
        bool okl = true, okr = true;
        if (SELF) {
          // position bounds (non-short-circuit &: no divergent branch)
          okl = xs[k] > p32;  // the left child ends at position x
          okr = uniform(Rk.last) > p32;
        }
        if (CROSS) {  // children inside the lane's own patch
          const uint32_t f = uniform(Rk.first), l = uniform(Rk.last);
          okl = okl & !((f >= pb) & (xs[k] < pe));
          okr = okr & !((xs[k] + 1 >= pb) & (l < pe));
        }
        if (SELF) {
          ml &= __ballot(okl);
          mr &= __ballot(okr);
        }
        // masks and readfirstlane values: every branch below is wave-uniform,
        // so the stack pointer and counters stay in scalar registers
        const bool any_l = ml != 0, any_r = mr != 0;
        const bool leaf_l = cl >= tleaf0, leaf_r = cr >= tleaf0;
        if (any_l && leaf_l) {
          const bool hl = (ml >> lane) & 1;
          wave_emit(buf, fill, out, SELF ? (hl & (cl - tleaf0 > p32)) : hl, pair_key(qa, el, SELF));
        }
        if (any_r && leaf_r) {
          const bool hr = (mr >> lane) & 1;
          wave_emit(buf, fill, out, SELF ? (hr & (cr - tleaf0 > p32)) : hr, pair_key(qa, er, SELF));
        }
        // the left child ends on top of the stack
        if (sp + 2 > kStack) {
          bad = true;
        } else {
          if (any_r && !leaf_r) stk[sp++] = cr;
          if (any_l && !leaf_l) stk[sp++] = cl;
        }
      }
      // one record's boxes in registers at a time
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_wave_barrier();  // every lane has read the records
    if (bad) {
      if (lane == 0) atomicOr(t.status, kErrTraverse);
      break;
    }
  }
  wave_flush(buf, fill, out);
  if (lane == 0 && out.visits) atomicAdd(out.visits, (unsigned long long)steps);
}

template <bool SELF, int K, bool CROSS = false>
__global__ __launch_bounds__(256) void k_narrow64(TreeView q, TreeView t, int xcd, uint32_t qper, PairOut out) {
  __shared__ uint64_t s_buf[256 / kWave][kWaveBuf];
  __shared__ uint32_t s_stack[256 / kWave][kStack];
  __shared__ Rec64 s_rec[256 / kWave][K];
  const uint32_t wv = threadIdx.x / kWave;
  const uint32_t group = kXcdQueries * kWave / (qper * blockDim.x);
  const uint32_t tile = xcd ? xcd_group_tile(blockIdx.x, gridDim.x, group) : blockIdx.x;
  walk64<SELF, K, CROSS>(q, t, tile * (blockDim.x / kWave) + wv, qper, out, s_buf[wv], s_stack[wv], s_rec[wv]);
}

// Several queries (object pairs) in one launch: block b walks tile
// b - block0 of the query whose [block0, block0 + tiles) holds b (a
// wave-uniform binary search over the table).
template <int K>
__global__ __launch_bounds__(256) void k_narrow64_batch(const BatchQuery* __restrict__ bq, uint32_t nq) {
  __shared__ uint64_t s_buf[256 / kWave][kWaveBuf];
  __shared__ uint32_t s_stack[256 / kWave][kStack];
  __shared__ Rec64 s_rec[256 / kWave][K];
  const uint32_t wv = threadIdx.x / kWave;
  uint32_t lo = 0, hi = nq;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (bq[mid].block0 <= blockIdx.x) lo = mid;
    else hi = mid;
  }
  const BatchQuery& e = bq[lo];
  if (blockIdx.x - e.block0 >= e.blocks) return;
  walk64<false, K, false>(e.q, e.t, (blockIdx.x - e.block0) * (256 / kWave) + wv, kWave, e.out, s_buf[wv], s_stack[wv], s_rec[wv]);
}

// fp64 form, one record per visit in scalar registers (batch 1): box 0
// with the child ids and the cache lines of box 1 in one round of scalar
// loads, then box 1 from the scalar cache; each box is tested with one
// v_cmpx chain (box_hits), so a visit issues no LDS instruction and no
// scalar instruction per compare.  The next node is kept in a register, the
// right child of a two-child visit goes on the per-wave LDS stack.
typedef __attribute__((address_space(4))) const double CDbl;

template <bool SELF, bool CROSS = false>
__global__ __launch_bounds__(256) void k_narrow64s(TreeView q, TreeView t, int xcd, uint32_t qper, PairOut out) {
  __shared__ uint64_t s_buf[256 / kWave][kWaveBuf];
  __shared__ uint32_t s_stack[256 / kWave][kStack];
  const uint32_t wv = threadIdx.x / kWave;
  uint64_t* buf = s_buf[wv];
  uint32_t* stk = s_stack[wv];
  uint32_t fill = 0;
  const uint32_t group = kXcdQueries * kWave / (qper * blockDim.x);
  const uint32_t tile = xcd ? xcd_group_tile(blockIdx.x, gridDim.x, group) : blockIdx.x;
  const uint64_t p = ((uint64_t)tile * (blockDim.x / kWave) + wv) * qper + lane_id();
  const bool valid = lane_id() < qper && p < q.n;
  double qk[kSlabs];
  uint32_t qa = 0;
  if (valid) {
    const double* src = q.rootbox64;
    if (q.n > 1) {
      uint32_t parent;
      int side;
      leaf_slot(q.delta, q.n, p, parent, side);
      src = q.rec64[parent].box[side];
    }
#pragma unroll
    for (int a = 0; a < kAxes; ++a) {
      const double2 v = ((const double2*)src)[a];
      qk[2 * a] = v.x;
      qk[2 * a + 1] = v.y;
    }
    qa = q.perm[p];
  } else {
    empty_slabs(qk);
  }
  const uint32_t n = (uint32_t)t.n;
  const uint32_t tleaf0 = n - 1;
  const uint32_t lane = lane_id();
  const uint32_t p32 = valid ? (uint32_t)p : 0u;  // positions fit 32 bits; invalid lanes hit nothing
  uint32_t pb = 0, pe = 0;
  if (CROSS) own_patch_range(q, qa, valid, n, pb, pe);
  uint32_t steps = 0;
  uint32_t sp = 0;
  uint32_t x = kEnd;  // the node to visit next (kEnd: pop the stack)
  {
    const CDbl* rb = (const CDbl*)t.rootbox64;
    bool h = true;
#pragma unroll
    for (int a = 0; a < kAxes; ++a) h = h & (qk[2 * a] < rb[2 * a + 1]) & (rb[2 * a] < qk[2 * a + 1]);
    if (SELF) h = h & ((uint32_t)(n - 1) > p32);  // the root's last position
    if (n == 1) {
      if (!SELF) wave_emit(buf, fill, out, h, pair_key(qa, uniform(t.perm[0]), SELF));
    } else if (__ballot(h) != 0) {
      x = uniform(*t.root);
    }
  }
  for (;;) {
    if (x == kEnd) {
      if (sp == 0) break;
      x = uniform(stk[--sp]);
    }
    if (x >= tleaf0 || ++steps > n) {
      if (lane == 0) atomicOr(t.status, kErrTraverse);
      break;
    }
    const CDbl* rp = (const CDbl*)(t.rec64 + x);
    const CInt* ip = (const CInt*)(t.rec64 + x);
    double bx[kSlabs];
#pragma unroll
    for (int k = 0; k < kSlabs; ++k) bx[k] = rp[k];
    // child ids, leaf elements (and `last` in self mode): dwords 104..109;
    // dwords 64 and 80 only bring box 1's cache lines into the scalar cache
    const uint32_t cl = (uint32_t)ip[104], cr = (uint32_t)ip[105];
    const uint32_t el = (uint32_t)ip[106], er = (uint32_t)ip[107];
    const uint32_t rlast = SELF ? (uint32_t)ip[109] : 0u;
    const uint32_t rfirst = CROSS ? (uint32_t)ip[108] : 0u;
    const uint32_t t0 = (uint32_t)ip[64], t1 = (uint32_t)ip[80];
    __builtin_amdgcn_sched_barrier(0);
    bool hl, hr;
    box_hits(qk, bx, t0, t1, &hl);
#pragma unroll
    for (int k = 0; k < kSlabs; ++k) bx[k] = rp[kSlabs + k];
    box_hits(qk, bx, 0u, 0u, &hr);
    if (SELF) {
      hl = hl & (x > p32);  // the left child ends at position x
      hr = hr & (rlast > p32);
    }
    if (CROSS) {  // children inside the lane's own patch
      hl = hl & !((rfirst >= pb) & (x < pe));
      hr = hr & !((x + 1 >= pb) & (rlast < pe));
    }
    const bool any_l = __ballot(hl) != 0, any_r = __ballot(hr) != 0;
    const bool leaf_l = cl >= tleaf0, leaf_r = cr >= tleaf0;
    if (any_l && leaf_l)
      wave_emit(buf, fill, out, SELF ? (hl & (cl - tleaf0 > p32)) : hl, pair_key(qa, el, SELF));
    if (any_r && leaf_r)
      wave_emit(buf, fill, out, SELF ? (hr & (cr - tleaf0 > p32)) : hr, pair_key(qa, er, SELF));
    const bool go_l = any_l && !leaf_l, go_r = any_r && !leaf_r;
    // depth first: continue with the left child, keep the right one
    if (go_l && go_r) {
      if (sp >= kStack) {
        if (lane == 0) atomicOr(t.status, kErrTraverse);
        break;
      }
      stk[sp++] = cr;
      x = cl;
    } else {
      x = go_l ? cl : (go_r ? cr : kEnd);
    }
  }
  wave_flush(buf, fill, out);
  if (lane == 0 && out.visits) atomicAdd(out.visits, (unsigned long long)steps);
}

// fp64 re-check of the fp32 candidates that the inner bound left open: both
// elements' k-DOPs recomputed from element data, the pair emitted on overlap.
// The stripe lengths are read on the device, so no host round trip separates
// the two kernels.  The grid is kRecheckStripes x (blocks per stripe); block
// b works on stripe b % kRecheckStripes.  Hits are staged per wave in LDS
// (one atomic on the pair counter per flush, not per wave that hits).  Block
// 0 also adds the stripe counts' sum and maximum to rtotal, and the stripes'
// visits and candidates to theirs, for the host.
// KIND / NV: both objects' element type (the common case, with registers
// sized for it); kGeneric: any mix, chosen at run time.
constexpr int kGeneric = -1;

// blocks per re-check stripe (512 in all): each block strides over its
// stripe's list, so a block stages many pairs per flush (12.6M candidates of a
// 2M-triangle mesh against itself: 409 us; with 32 / 16 / 6 / 4 blocks a stripe 567 /
// 522 / 508 / 506; 54,612 hexes 42 us, 51 / 46 / 52 / 65)
constexpr uint64_t kRecheckBlocksPerStripe = 8;

template <int KIND, int NV>
__global__ __launch_bounds__(256) void k_recheck(TreeView q, TreeView t, PairOut out) {
  __shared__ uint64_t s_buf[256 / kWave][kWaveBuf];
  uint64_t* buf = s_buf[threadIdx.x / kWave];
  uint32_t fill = 0;
  if (blockIdx.x == 0 && threadIdx.x < kRecheckStripes) {
    // one wave: summed in registers (an addition per lane to these neighbouring
    // words queued for 10 us, most of this kernel on short lists)
    static_assert(kRecheckStripes == kWave, "a lane per stripe");
    const unsigned long long* line = out.rcount + (uint64_t)threadIdx.x * kRecheckStride;
    unsigned long long c = line[0], mx = c, v = line[1], k = line[2];
    for (int o = kWave / 2; o > 0; o >>= 1) {
      c += __shfl_xor(c, o, kWave);
      v += __shfl_xor(v, o, kWave);
      k += __shfl_xor(k, o, kWave);
      const unsigned long long y = __shfl_xor(mx, o, kWave);
      mx = y > mx ? y : mx;
    }
    if (threadIdx.x == 0) {
      atomicAdd(out.rtotal, c);
      atomicMax(out.rtotal + 1, mx);
      if (out.visits) atomicAdd(out.visits, v);
      if (out.candidates) atomicAdd(out.candidates, k);
    }
  }
  const uint32_t stripe = blockIdx.x % kRecheckStripes;
  const uint32_t per = gridDim.x / kRecheckStripes;
  const unsigned long long cnt0 = out.rcount[(uint64_t)stripe * kRecheckStride];
  const uint64_t cnt = cnt0 < out.rcap ? cnt0 : out.rcap;
  const uint64_t* list = out.recheck + (uint64_t)stripe * out.rcap;
  const uint64_t stride = (uint64_t)per * blockDim.x;
  for (uint64_t base = (uint64_t)(blockIdx.x / kRecheckStripes) * blockDim.x; base < cnt; base += stride) {
    const uint64_t i = base + threadIdx.x;
    bool hit = false;
    uint64_t key = 0;
    if (i < cnt) {
      key = list[i];
      double ka[kSlabs];
      if constexpr (KIND == kGeneric) {
        element_kdop_any(q.elem, (uint32_t)(key >> 32), ka);
        hit = element_overlap_any(t.elem, (uint32_t)key, ka);
      } else {
        element_kdop<KIND, NV>(q.elem, (uint32_t)(key >> 32), ka);
        hit = element_overlap<KIND, NV>(t.elem, (uint32_t)key, ka);
      }
    }
    wave_emit(buf, fill, out, hit, key);
  }
  block_flush(buf, fill, out);
}

static void launch_recheck(const TreeView& q, const TreeView& t, const PairOut& out, unsigned blocks, hipStream_t s) {
  const ElemInput& a = q.elem;
  const ElemInput& b = t.elem;
  const dim3 g(blocks), th(256);
  if (a.kind == b.kind && (a.kind != kPoly || a.nv == b.nv)) {
    if (a.kind == kSphere) {
      hipLaunchKernelGGL((k_recheck<kSphere, 1>), g, th, 0, s, q, t, out);
      return;
    }
    if (a.kind == kSnapshot) {
      hipLaunchKernelGGL((k_recheck<kSnapshot, 1>), g, th, 0, s, q, t, out);
      return;
    }
    switch (a.nv) {
      case 3: hipLaunchKernelGGL((k_recheck<kPoly, 3>), g, th, 0, s, q, t, out); return;
      case 4: hipLaunchKernelGGL((k_recheck<kPoly, 4>), g, th, 0, s, q, t, out); return;
      case 8: hipLaunchKernelGGL((k_recheck<kPoly, 8>), g, th, 0, s, q, t, out); return;
      default: break;
    }
  }
  hipLaunchKernelGGL((k_recheck<kGeneric, 0>), g, th, 0, s, q, t, out);
}

// exact patch slabs (the union of the patch's element k-DOPs)
__device__ __forceinline__ void patch_slabs(const TreeView& v, uint64_t k, double* out) {
  const unsigned long long* e = v.patch_k64 + k * kSlabs;
#pragma unroll
  for (int i = 0; i < kSlabs; ++i) out[i] = from_ordered_u64(e[i]);
}

// Patch broadphase over all patch pairs: one lane per (patch of q, patch of
// t), t fastest, so a wave shares its q patch (a broadcast load) and reads 64
// consecutive t patches; both objects' patch slabs stay in L2.  Empty patches
// never overlap (broadphase.cpp:79-80).
__global__ __launch_bounds__(256) void k_patch_pairs(TreeView q, TreeView t, PairOut out) {
  const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t qp = k / t.od, tp = k - qp * t.od;
  bool hit = false;
  if (qp < q.od) {
    const uint32_t rq = q.patch_root[qp], rt = t.patch_root[tp];
    if (rq != kEnd && rq < 2 * q.n - 1 && rt != kEnd && rt < 2 * t.n - 1) {
      double qk[kSlabs], tk[kSlabs];
      patch_slabs(q, qp, qk);
      patch_slabs(t, tp, tk);
      hit = overlap(qk, tk);
    }
  }
  emit(out, hit, (qp << 32) | tp);
}

__global__ __launch_bounds__(256) void k_records(const uint64_t* __restrict__ pairs, uint64_t count,
                                                 const uint32_t* __restrict__ patch_a, const uint64_t* __restrict__ gid_a,
                                                 const uint32_t* __restrict__ patch_b, const uint64_t* __restrict__ gid_b,
                                                 uint64_t off_a, uint64_t off_b, uint64_t* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t key = pairs[i];
    const uint32_t a = (uint32_t)(key >> 32), b = (uint32_t)key;
    ulonglong4 r;
    r.x = patch_a[a] + off_a;
    r.y = gid_a ? gid_a[a] : a;
    r.z = patch_b[b] + off_b;
    r.w = gid_b ? gid_b[b] : b;
    ((ulonglong4*)out)[i] = r;
  }
}

// patch centroid = accumulate(element centroids in patch order, zeros) / size
// (patch.hpp:113-116): the sum is rounded in patch order, so each coordinate
// is one serial fp64 add chain.  What bounds it is that chain (about 8 cycles
// per element), once nothing else is in it: a block per patch stages
// kCentroidChunk centroids at a time in LDS (the permutation two chunks and
// the gathers one chunk ahead, in registers), and lanes 0..2 of its first
// wave add one coordinate each from there.  One thread per patch, each
// element's two dependent loads in the chain, took 1,703 us on 32 patches of
// 4,096 triangles on average; this takes 45 us.
constexpr uint32_t kCentroidItems = 4;
template <uint32_t BLOCK>
struct CentroidLds {
  static constexpr uint32_t chunk = BLOCK * kCentroidItems;
  double v[2][3][chunk];
};
// positions of patch k
__device__ __forceinline__ void patch_range(const uint32_t* splits, uint64_t n, uint64_t od, uint64_t k, uint32_t& b,
                                            uint32_t& e) {
  b = (k == 0) ? 0u : splits[k - 1];
  e = (k == od - 1) ? (uint32_t)n : splits[k];
}
__device__ __forceinline__ double centroid_coord(const double* planes, const double* caos, uint64_t n, uint32_t src,
                                                 uint32_t c) {
  return planes ? planes[(uint64_t)c * n + src] : caos[3 * (uint64_t)src + c];
}

// one patch of cnt > 0 elements from position b on, by the whole block
template <uint32_t BLOCK>
__device__ __forceinline__ void block_centroid(const double* __restrict__ planes, const double* __restrict__ caos,
                                               const uint32_t* __restrict__ perm, uint64_t n, uint64_t k, uint32_t b,
                                               uint32_t cnt, double* __restrict__ out, CentroidLds<BLOCK>& L) {
  constexpr uint32_t kChunk = CentroidLds<BLOCK>::chunk;
  const uint32_t t = threadIdx.x, nchunk = (cnt + kChunk - 1) / kChunk;
  uint32_t src[kCentroidItems];
  double v[kCentroidItems][3];
  auto load_src = [&](uint32_t chunk) {
#pragma unroll
    for (uint32_t j = 0; j < kCentroidItems; ++j) {
      const uint32_t i = chunk * kChunk + j * BLOCK + t;
      src[j] = i < cnt ? perm[b + i] : kEnd;
    }
  };
  auto load_val = [&]() {
#pragma unroll
    for (uint32_t j = 0; j < kCentroidItems; ++j)
#pragma unroll
      for (int c = 0; c < 3; ++c) v[j][c] = src[j] == kEnd ? 0.0 : centroid_coord(planes, caos, n, src[j], c);
  };
  load_src(0);
  load_val();
  load_src(1);
  double s = 0.0;
  for (uint32_t q = 0; q < nchunk; ++q) {
    double(*cur)[kChunk] = L.v[q & 1];
#pragma unroll
    for (uint32_t j = 0; j < kCentroidItems; ++j)
#pragma unroll
      for (int c = 0; c < 3; ++c) cur[c][j * BLOCK + t] = v[j][c];
    load_val();
    load_src(q + 2);
    // one barrier per chunk: the chunk staged next goes to the other buffer,
    // whose adds ended before every thread's arrival here
    __syncthreads();
    if (t < 3) {
      const uint32_t left = cnt - q * kChunk;
      s = ordered_sum(cur[t], left < kChunk ? left : kChunk, s);
    }
  }
  if (t < 3) out[3 * k + t] = s / (double)cnt;
}

__global__ __launch_bounds__(256) void k_patch_centroids(const double* __restrict__ planes,
                                                         const double* __restrict__ caos,
                                                         const uint32_t* __restrict__ perm,
                                                         const uint32_t* __restrict__ splits, uint64_t n,
                                                         uint64_t od, double* __restrict__ out) {
  __shared__ CentroidLds<256> L;
  const uint64_t k = blockIdx.x;
  uint32_t b, e;
  patch_range(splits, n, od, k, b, e);
  if (e <= b) {  // an empty patch
    if (threadIdx.x < 3) out[3 * k + threadIdx.x] = 0.0;
    return;
  }
  block_centroid<256>(planes, caos, perm, n, k, b, e - b, out, L);
}

// Many patches of few elements: 16 patches a wave, four lanes each, of which
// three add a coordinate straight from memory, kFewBatch loads together.  A
// patch of more than kFewElems elements is left to the wave as a whole.  The
// wave's patches are gridDim.x apart, so that large neighbours are not one
// wave's.
constexpr uint32_t kFewPatches = 16;
constexpr uint32_t kFewElems = 128;
constexpr uint32_t kFewBatch = 8;
__global__ __launch_bounds__(kWave) void k_patch_centroids_few(const double* __restrict__ planes,
                                                               const double* __restrict__ caos,
                                                               const uint32_t* __restrict__ perm,
                                                               const uint32_t* __restrict__ splits, uint64_t n,
                                                               uint64_t od, double* __restrict__ out) {
  __shared__ CentroidLds<kWave> L;
  const uint32_t c = threadIdx.x & 3;
  const uint64_t k = (uint64_t)(threadIdx.x >> 2) * gridDim.x + blockIdx.x;
  uint32_t b = 0, e = 0;
  if (k < od) patch_range(splits, n, od, k, b, e);
  const uint32_t cnt = e > b ? e - b : 0u;
  if (k < od && cnt <= kFewElems && c < 3) {
    double s = 0.0;
    for (uint32_t i = 0; i < cnt; i += kFewBatch) {
      uint32_t src[kFewBatch];
      double v[kFewBatch];
#pragma unroll
      for (uint32_t j = 0; j < kFewBatch; ++j) src[j] = i + j < cnt ? perm[b + i + j] : kEnd;
#pragma unroll
      for (uint32_t j = 0; j < kFewBatch; ++j) v[j] = src[j] == kEnd ? 0.0 : centroid_coord(planes, caos, n, src[j], c);
#pragma unroll
      for (uint32_t j = 0; j < kFewBatch; ++j)
        if (i + j < cnt) s = s + v[j];
    }
    out[3 * k + c] = cnt ? s / (double)cnt : 0.0;
  }
  uint64_t large = __ballot(c == 0 && cnt > kFewElems);
  while (large) {  // (uniform)
    const int l = __builtin_ctzll(large);
    large &= large - 1;
    block_centroid<kWave>(planes, caos, perm, n, (uint64_t)(l >> 2) * gridDim.x + blockIdx.x,
                          (uint32_t)__shfl((int)b, l, kWave), (uint32_t)__shfl((int)cnt, l, kWave), out, L);
    __syncthreads();  // L is free again
  }
}

// Order-independent digest of a pair list: the sum and the xor of two
// independent 64-bit mixes (splitmix64 finalizer) of every key.
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

__global__ __launch_bounds__(256) void k_digest(const uint64_t* __restrict__ pairs, uint64_t count,
                                                unsigned long long* out) {
  uint64_t s = 0, x = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t k = pairs[i];
    s += mix64(k);
    x ^= mix64(k ^ 0x9e3779b97f4a7c15ull);
  }
  for (int o = 32; o > 0; o >>= 1) {
    s += __shfl_xor(s, o, 64);
    x ^= __shfl_xor(x, o, 64);
  }
  // one pair of atomics per block (the two addresses serialize them)
  __shared__ uint64_t ss[256 / kWave], sx[256 / kWave];
  if (lane_id() == 0) {
    ss[threadIdx.x / kWave] = s;
    sx[threadIdx.x / kWave] = x;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t v = 1; v < blockDim.x / kWave; ++v) {
      s += ss[v];
      x ^= sx[v];
    }
    if ((s | x) != 0) {
      atomicAdd(out, (unsigned long long)s);
      atomicXor(out + 1, (unsigned long long)x);
    }
  }
}

// ---- launchers ---------------------------------------------------------------------
template <int K>
static void narrow64_dispatch(const TreeView& q, const TreeView& t, int self, int xcd, uint32_t qper, unsigned blocks, unsigned bs,
                              const PairOut& out, hipStream_t s) {
  if (self == 2) hipLaunchKernelGGL((k_narrow64<true, K, true>), dim3(blocks), dim3(bs), 0, s, q, t, xcd, qper, out);
  else if (self) hipLaunchKernelGGL((k_narrow64<true, K>), dim3(blocks), dim3(bs), 0, s, q, t, xcd, qper, out);
  else hipLaunchKernelGGL((k_narrow64<false, K>), dim3(blocks), dim3(bs), 0, s, q, t, xcd, qper, out);
}

// Queries per wave: 64, or fewer (down to 4) while the launch has less than two
// waves for each of the GPU's 1,024 SIMDs, one for a self walk.  A wave visits
// what any of its lanes overlaps, so fewer queries visit less, and a small
// object's launch, which lasts as long as its longest wave, gets shorter as long as
// idle SIMDs take the added waves.  A x B over sheets, at 64 queries a wave and
// by this rule: 2,048 queries 114 -> 46 us, 8,192 228 -> 69, 32,768 205 -> 119,
// 89,888 200 -> 160 (181,202 stay at 64: 187 us, 230 at 32); over fp64 records
// 192 -> 79, 394 -> 121, 373 -> 209, 372 -> 279.  Self walks visit half as
// much: 8,000 spheres 60 -> 27 us (fp64 records 102 -> 49), 30,000 88 -> 49
// (148 -> 91; with 2,048 waves 58 and 122), 60,000 105 -> 75 (174 -> 131).  The
// cross-patch walk keeps 64: few of its queries have work.
static uint32_t queries_per_wave(uint64_t n, int self) {
  uint32_t qper = kWave;
  while (self != 2 && qper > 4 && n / qper < (self ? 1024u : 2048u)) qper >>= 1;
  return qper;
}

hipError_t launch_narrowphase(const TreeView& q, const TreeView& t, int leaf_size, int self, int form,
                              const LaunchShape& shape, const PairOut& out, hipStream_t s) {
  (void)leaf_size;  // the record walk tests every leaf from its parent's record
  if (q.n == 0 || t.n == 0) return hipSuccess;
  const unsigned bs = shape.block;
  if (bs != 64 && bs != 128 && bs != 256) return hipErrorInvalidValue;
  if (!q.perm || !t.perm || !t.root || !t.status || !out.pairs || !out.count) return hipErrorInvalidValue;
  if (self == 2 && (!q.patch_of_input || (q.od > 1 && !q.splits))) return hipErrorInvalidValue;
  const uint32_t qper = queries_per_wave(q.n, self);
  const unsigned waves = (unsigned)((q.n + qper - 1) / qper), bw = bs / kWave;
  const unsigned blocks = (waves + bw - 1) / bw;  // of the walks over fp64 records
  const int xcd = shape.xcd_remap ? 1 : 0;
  if (form == kFormFp32 || form == kFormMixed) {
    if (!q.rec32 || !q.rootbox32 || !q.delta || !t.rec32 || !t.rootbox32 || !q.origin || !t.origin)
      return hipErrorInvalidValue;
    if (!out.recheck || !out.rcount || !out.rtotal) return hipErrorInvalidValue;
    // the fp32 walk tests leaves from their parents' records: no leaf clusters
    // one record per round trip: it arrives in scalar registers (the batch
    // applies to the fp64 walk).  Both forms keep the leaf candidates whose
    // fp32 gap proves the fp64 overlap and re-check the rest in fp64.
    const int32_t inner = kInnerUlps;
    const dim3 g(waves), bl(kWave);
    if (self == 2) {
      if ((out.icap && !out.items) || !out.icount) return hipErrorInvalidValue;
      hipLaunchKernelGGL((k_narrow32<true, true, kWalkTop>), g, bl, 0, s, q, t, xcd, qper, out, inner);
      if (out.icap)
        hipLaunchKernelGGL((k_narrow32_items<true, true>), dim3(kItemBlocks), bl, 0, s, q, t, qper, out, inner);
    } else if (self) {
      hipLaunchKernelGGL((k_narrow32<true, false>), g, bl, 0, s, q, t, xcd, qper, out, inner);
    } else {
      hipLaunchKernelGGL((k_narrow32<false, false>), g, bl, 0, s, q, t, xcd, qper, out, inner);
    }
    // in self mode both keys index the one object (q == t)
    uint64_t per = (out.rcap + 255) / 256;  // blocks per stripe
    if (per > kRecheckBlocksPerStripe) per = kRecheckBlocksPerStripe;
    if (per == 0) per = 1;
    launch_recheck(q, t, out, (unsigned)(per * kRecheckStripes), s);
    return hipGetLastError();
  }
  if (!q.rec64 || !q.rootbox64 || !q.delta || !t.rec64 || !t.rootbox64) return hipErrorInvalidValue;
  switch (shape.batch) {
    case 1:
      if (self == 2) hipLaunchKernelGGL((k_narrow64s<true, true>), dim3(blocks), dim3(bs), 0, s, q, t, xcd, qper, out);
      else if (self) hipLaunchKernelGGL(k_narrow64s<true>, dim3(blocks), dim3(bs), 0, s, q, t, xcd, qper, out);
      else hipLaunchKernelGGL(k_narrow64s<false>, dim3(blocks), dim3(bs), 0, s, q, t, xcd, qper, out);
      break;
    case 2: narrow64_dispatch<2>(q, t, self, xcd, qper, blocks, bs, out, s); break;
    case 4: narrow64_dispatch<4>(q, t, self, xcd, qper, blocks, bs, out, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Three short runs of 8-byte words (a query's counters and both objects' status
// words, a root box and its frame) in one launch, straight into pinned host
// memory: one small kernel instead of a device-to-host copy for each.
__global__ void k_readback(const unsigned long long* __restrict__ a, int na, const unsigned long long* __restrict__ b,
                           int nb, const unsigned long long* __restrict__ c, int nc,
                           unsigned long long* __restrict__ host) {
  const int i = (int)threadIdx.x;
  if (i < na) host[i] = a[i];
  else if (i < na + nb) host[i] = b[i - na];
  else if (i < na + nb + nc) host[i] = c[i - na - nb];
  __threadfence_system();  // the words are in host memory before the kernel ends
}

hipError_t launch_readback(const void* a, int na, const void* b, int nb, const void* c, int nc,
                           unsigned long long* host, hipStream_t s) {
  if (na < 0 || nb < 0 || nc < 0 || na + nb + nc > 64) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_readback, dim3(1), dim3(64), 0, s, (const unsigned long long*)a, na,
                     (const unsigned long long*)b, nb, (const unsigned long long*)c, nc, host);
  return hipGetLastError();
}

// A batch's counters, `words` of each query, set to zero (a block row per query).
__global__ __launch_bounds__(256) void k_batch_clear(const BatchQuery* __restrict__ bq, uint32_t words) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < words) bq[blockIdx.y].out.count[i] = 0;
}

// The first ncount counters of every query of a batch and its objects' status
// words, kReadbackWords words each, into pinned host memory: one launch and one
// synchronization, where three copies for each query took 30 us apiece.
__global__ void k_batch_readback(const BatchQuery* __restrict__ bq, int ncount, unsigned long long* __restrict__ host) {
  const BatchQuery& e = bq[blockIdx.x];
  const int i = (int)threadIdx.x;
  unsigned long long* h = host + (uint64_t)blockIdx.x * kReadbackWords;
  if (i < ncount) h[i] = e.out.count[i];
  else if (i < ncount + 2) h[i] = ((const unsigned long long*)e.q.status)[i - ncount];
  else if (i < ncount + 4) h[i] = ((const unsigned long long*)e.t.status)[i - ncount - 2];
  __threadfence_system();  // the words are in host memory before the kernel ends
}

hipError_t launch_batch_clear(const BatchQuery* bq, uint32_t nq, uint32_t words, hipStream_t s) {
  if (nq == 0 || words == 0) return hipSuccess;
  if (nq > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_batch_clear, dim3((words + 255) / 256, nq), dim3(256), 0, s, bq, words);
  return hipGetLastError();
}

hipError_t launch_batch_readback(const BatchQuery* bq, uint32_t nq, int ncount, unsigned long long* host,
                                 hipStream_t s) {
  if (nq == 0) return hipSuccess;
  if (ncount < 0 || (uint32_t)ncount + 4 > kReadbackWords) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_batch_readback, dim3(nq), dim3(64), 0, s, bq, ncount, host);
  return hipGetLastError();
}

hipError_t launch_narrowphase_batch(const BatchQuery* bq, uint32_t nq, uint32_t blocks, int batch, int form,
                                    hipStream_t s) {
  if (nq == 0 || blocks == 0) return hipSuccess;
  if (form == kFormFp32 || form == kFormMixed) {
    hipLaunchKernelGGL(k_narrow32_batch, dim3(4 * blocks), dim3(kWave), 0, s, bq, nq, kInnerUlps);
  } else if (batch == 4) {
    hipLaunchKernelGGL(k_narrow64_batch<4>, dim3(blocks), dim3(256), 0, s, bq, nq);
  } else {
    hipLaunchKernelGGL(k_narrow64_batch<2>, dim3(blocks), dim3(256), 0, s, bq, nq);
  }
  return hipGetLastError();
}

hipError_t launch_recheck_query(const TreeView& q, const TreeView& t, const PairOut& out, hipStream_t s) {
  if (q.n == 0 || t.n == 0) return hipSuccess;
  if (!out.recheck || !out.rcount || !out.rtotal) return hipErrorInvalidValue;
  uint64_t per = (out.rcap + 255) / 256;  // blocks per stripe
  if (per > kRecheckBlocksPerStripe) per = kRecheckBlocksPerStripe;
  if (per == 0) per = 1;
  launch_recheck(q, t, out, (unsigned)(per * kRecheckStripes), s);
  return hipGetLastError();
}

hipError_t launch_patch_broadphase(const TreeView& q, const TreeView& t, int fp32, const PairOut& out,
                                   hipStream_t s) {
  if (q.od == 0 || t.od == 0 || t.n == 0 || q.n == 0) return hipSuccess;
  if (!q.patch_k64 || !t.patch_k64) return hipErrorInvalidValue;
  (void)fp32;
  const uint64_t total = q.od * t.od;
  hipLaunchKernelGGL(k_patch_pairs, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, q, t, out);
  return hipGetLastError();
}

hipError_t launch_records(const uint64_t* pairs, uint64_t count, const uint32_t* patch_a, const uint64_t* gid_a,
                          const uint32_t* patch_b, const uint64_t* gid_b, uint64_t off_a, uint64_t off_b,
                          uint64_t* out, hipStream_t s) {
  if (count == 0) return hipSuccess;
  uint64_t blocks = (count + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_records, dim3((unsigned)blocks), dim3(256), 0, s, pairs, count, patch_a, gid_a, patch_b,
                     gid_b, off_a, off_b, out);
  return hipGetLastError();
}

hipError_t launch_digest(const uint64_t* pairs, uint64_t count, unsigned long long* out, hipStream_t s) {
  if (count == 0) return hipSuccess;
  uint64_t blocks = (count + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(k_digest, dim3((unsigned)blocks), dim3(256), 0, s, pairs, count, out);
  return hipGetLastError();
}

// Where the patches are many and small, a block each is mostly the cost of its
// launch: the whole call that packs them takes, with a block a patch / four lanes
// a patch, 63 / 26 us for 131,072 elements in 16,384 patches, 80 / 43 for a million in
// 16,384, 34 / 27 for 131,072 in 4,096 and 30 / 30 in 2,048 (an average of 64),
// but 27 / 86 in 512 and 49 / 84 for a million in 4,096.
constexpr uint64_t kFewPatchesMin = 1024;
constexpr uint64_t kFewAverage = 64;
hipError_t launch_patch_centroids(const double* planes, const double* caos, const uint32_t* perm,
                                  const uint32_t* splits, uint64_t n, uint64_t od, double* out, hipStream_t s) {
  if (od == 0) return hipSuccess;
  if (!out || (n && ((!planes && !caos) || !perm)) || (od > 1 && !splits)) return hipErrorInvalidValue;
  if (od >= kFewPatchesMin && n <= kFewAverage * od)
    hipLaunchKernelGGL(k_patch_centroids_few, dim3((unsigned)((od + kFewPatches - 1) / kFewPatches)), dim3(kWave), 0, s,
                       planes, caos, perm, splits, n, od, out);
  else
    hipLaunchKernelGGL(k_patch_centroids, dim3((unsigned)od), dim3(256), 0, s, planes, caos, perm, splits, n, od, out);
  return hipGetLastError();
}

}  // namespace dbvh
