// small.hip -- the build of an object of few elements up to its tree stage,
// in one launch of one workgroup.
//
// The stages and their results are those of build.hip and sort.hip (bounds,
// Morton codes, stable sort, cluster splits, split heights); elements,
// bounds, codes and boundaries stay in registers and LDS between them.  As
// launches of their own these stages cost an object of 512 triangles ten
// launches and their gaps, about 90 us of which 40 were the kernels; as one
// launch they take 20 us (with up to some hundred patches; what is cleared for each
// patch is below).  One CU's memory and sorting rate sets the upper end
// of the range: at 8,192 triangles the launch takes 60 us and a contact step of
// two such objects 820 us, 804 as separate launches.
#include "device.hpp"
#include "kernels.hpp"
#include "sort_block.hpp"

namespace dbvh {

namespace {
constexpr double kBig = 1.7976931348623157e308;

__device__ __forceinline__ double wave_lo(double v) {
  for (int o = 32; o > 0; o >>= 1) v = sel_min(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double wave_hi(double v) {
  for (int o = 32; o > 0; o >>= 1) v = sel_max(v, __shfl_xor(v, o, 64));
  return v;
}

// one element's cardinal slabs and centroid (the operations and order of
// k_prep in build.hip, the vertex count at run time)
__device__ __forceinline__ void element_bounds(const ElemInput& in, uint32_t e, double* lo, double* hi, double* c) {
  const uint64_t n = in.n;
  if (in.kind == kSnapshot) {
    const double* k = in.data + (uint64_t)e * kSlabs;
    for (int a = 0; a < 3; ++a) {
      lo[a] = k[2 * a];
      hi[a] = k[2 * a + 1];
      c[a] = in.centroids[3 * (uint64_t)e + a];
    }
    return;
  }
  const double x = in.data[e], y = in.data[n + e], z = in.data[2 * n + e];
  const double r = in.kind == kSphere ? in.data[3 * n + e] : in.eps;
  const double p[3] = {project<0>(x, y, z), project<1>(x, y, z), project<2>(x, y, z)};
  for (int a = 0; a < 3; ++a) {
    lo[a] = p[a] - r;
    hi[a] = p[a] + r;
  }
  if (in.kind == kSphere) {
    c[0] = x;
    c[1] = y;
    c[2] = z;
    return;
  }
  double s[3] = {0.0 + x, 0.0 + y, 0.0 + z};
  for (int j = 1; j < in.nv; ++j) {
    const double* d = in.data + (uint64_t)(3 * j) * n + e;
    const double vx = d[0], vy = d[n], vz = d[2 * n];
    const double q[3] = {project<0>(vx, vy, vz), project<1>(vx, vy, vz), project<2>(vx, vy, vz)};
    for (int a = 0; a < 3; ++a) {
      lo[a] = sel_min(lo[a], q[a] - r);
      hi[a] = sel_max(hi[a], q[a] + r);
    }
    s[0] = s[0] + vx;
    s[1] = s[1] + vy;
    s[2] = s[2] + vz;
  }
  for (int a = 0; a < 3; ++a) c[a] = s[a] / (double)in.nv;
}
}  // namespace

template <typename K, int ITEMS>
__global__ __launch_bounds__(kSmallBlock) void k_build_small(ElemInput in, BuildBufs b, int clear_k64) {
  constexpr int kWaves = kSmallBlock / 64;
  constexpr int kPasses = sizeof(K);
  __shared__ SortBlockLds<K, ITEMS> L;
  __shared__ double s_part[kWaves][6];
  __shared__ Bounds s_bounds;
  __shared__ uint32_t s_hist[256];
  __shared__ uint32_t s_cnt[kWaves][2];
  __shared__ uint32_t s_cut[2];
  const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const uint32_t n = (uint32_t)in.n, nsplits = (uint32_t)(b.od - 1);
  auto pos = [&](int j) { return small_pos<ITEMS>(j); };

  // what later stages expect cleared
  for (uint64_t i = tid; i < b.od; i += kSmallBlock) b.patch_root[i] = kEnd;
  if (clear_k64)
    for (uint64_t i = tid; i < b.od * kSlabs; i += kSmallBlock) b.patch_k64[i] = (i & 1) ? 0ull : ~0ull;
  if (tid < 4) b.status[tid] = 0;
  if (tid == 0) *b.root = kEnd;
  if (tid < 256) s_hist[tid] = 0;

  // bounds and centroids
  double cx[ITEMS], cy[ITEMS], cz[ITEMS];
  double mn[3] = {kBig, kBig, kBig}, mx[3] = {-kBig, -kBig, -kBig};
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t e = pos(j);
    cx[j] = cy[j] = cz[j] = 0.0;
    if (e < n) {
      double lo[3], hi[3], c[3];
      element_bounds(in, e, lo, hi, c);
      cx[j] = c[0];
      cy[j] = c[1];
      cz[j] = c[2];
      if (in.kind == kPoly) {
        b.centroid[e] = c[0];
        b.centroid[n + e] = c[1];
        b.centroid[2 * (uint64_t)n + e] = c[2];
      }
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        mn[a] = (lo[a] < mn[a]) ? lo[a] : mn[a];
        mx[a] = (mx[a] < hi[a]) ? hi[a] : mx[a];
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double l = wave_lo(mn[a]), h = wave_hi(mx[a]);
    if (lane == 0) {
      s_part[w][a] = l;
      s_part[w][3 + a] = h;
    }
  }
  __syncthreads();
  if (tid == 0) {
    double r[6];
    for (int a = 0; a < 6; ++a) r[a] = s_part[0][a];
    for (int v = 1; v < kWaves; ++v)
      for (int a = 0; a < 3; ++a) {
        r[a] = sel_min(r[a], s_part[v][a]);
        r[3 + a] = sel_max(r[3 + a], s_part[v][3 + a]);
      }
    Bounds bd;
    for (int a = 0; a < 3; ++a) {
      bd.min[a] = r[a];
      bd.max[a] = r[3 + a];
      const double width = r[3 + a] - r[a];
      bd.inv[a] = 1.0 / width;
    }
    bd.pad = 0.0;
    s_bounds = bd;
    *b.bounds = bd;
    if (b.origin) {  // the fp32 frame (as k_prep_final)
      double o[3];
      for (int a = 0; a < 3; ++a) {
        const double v = bd.min[a];
        o[a] = (v - v == 0.0) ? v : 0.0;
        b.origin[a] = o[a];
      }
      proj_all(o[0], o[1], o[2], b.origin + 3);
    }
  }
  __syncthreads();

  // Morton codes, sorted with their input indices
  const Bounds bd = s_bounds;
  K key[ITEMS];
  uint32_t val[ITEMS];
  K* codes0 = (K*)b.codes0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t e = pos(j);
    key[j] = 0;
    val[j] = e;
    if (e < n) {
      if constexpr (sizeof(K) == 8) key[j] = morton63(cx[j], cy[j], cz[j], bd);
      else key[j] = morton30(cx[j], cy[j], cz[j], bd);
      codes0[e] = key[j];
    }
  }
  sort_block<K, ITEMS>(L, key, val, true, n, kPasses);
  __syncthreads();
  K* codes = (K*)b.codes_a;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t p = pos(j);
    if (p < n) {
      codes[p] = key[j];
      b.perm[p] = val[j];
      L.keys[p] = key[j];
    }
  }
  __syncthreads();

  // cluster splits: the boundary depths, their histogram and its threshold
  // (k_cluster_depth, cluster_cut)
  const uint32_t m = n - 1, c = nsplits < m ? nsplits : m;
  uint32_t depth[ITEMS];
  K diff[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t i = pos(j);
    depth[j] = 0xffffffffu;
    diff[j] = 0;
    if (i < m) {
      diff[j] = key[j] ^ L.keys[i + 1];
      if constexpr (sizeof(K) == 8) depth[j] = diff[j] ? (uint32_t)__clzll((long long)diff[j]) : 255u;
      else depth[j] = diff[j] ? (uint32_t)__clz((int)diff[j]) : 255u;
      if (c) atomicAdd(&s_hist[depth[j]], 1u);
    }
  }
  __syncthreads();
  if (w == 0) {
    // four bins a lane: D is the first bin at which the running count reaches c
    uint32_t h[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      h[k] = s_hist[4 * lane + k];
      sum += h[k];
    }
    uint32_t x = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= (uint32_t)o) x += y;
    }
    const uint64_t reach = __ballot(x >= c);  // (lane 63's count is m >= c)
    if (lane == (uint32_t)__builtin_ctzll(reach)) {
      uint32_t cum = x - sum, k = 0;
      while (k < 3 && cum + h[k] < c) cum += h[k++];
      s_cut[0] = 4 * lane + k;
      s_cut[1] = c - cum;
    }
  }
  __syncthreads();
  // the taken boundaries in position order (k_cluster_emit): a position's
  // patch is the number of split values up to it
  const uint32_t D = s_cut[0], need = s_cut[1];
  uint32_t lt = 0, eq = 0;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    lt += (uint32_t)__popcll(__ballot(depth[j] < D));
    eq += (uint32_t)__popcll(__ballot(depth[j] == D));
  }
  if (lane == 0) {
    s_cnt[w][0] = lt;
    s_cnt[w][1] = eq;
  }
  __syncthreads();
  lt = eq = 0;
  for (uint32_t v = 0; v < w; ++v) {
    lt += s_cnt[v][0];
    eq += s_cnt[v][1];
  }
  uint32_t patch[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t i = pos(j);
    const bool isl = depth[j] < D, ise = depth[j] == D;
    const uint64_t ml = __ballot(isl), me = __ballot(ise);
    const uint32_t er = eq + (uint32_t)__popcll(me & lanemask_lt());
    const uint32_t slot = lt + (uint32_t)__popcll(ml & lanemask_lt()) + (er < need ? er : need);
    const bool taken = c && (isl || (ise && er < need));
    if (taken) b.splits[slot] = i;
    patch[j] = c ? slot + (taken ? 1u : 0u) : 0u;
    if (i == m) patch[j] = nsplits;  // every split value is at most n - 1
    if (i < n) L.vals[i] = patch[j];
    lt += (uint32_t)__popcll(ml);
    eq += (uint32_t)__popcll(me);
  }
  for (uint32_t i = c + tid; i < nsplits; i += kSmallBlock) b.splits[i] = m;
  __syncthreads();

  // patches, split heights and cleared arrival words (k_delta)
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const uint32_t i = pos(j);
    if (i >= n) continue;
    b.patch_of_pos[i] = patch[j];
    if (i < m) {
      b.counters[i] = 0;
      const uint32_t next = L.vals[i + 1];
      uint32_t d;
      if (next != patch[j]) {
        d = 128u + (31u - (uint32_t)__clz((int)(next ^ patch[j])));
      } else if (diff[j]) {
        d = 64u + (63u - (uint32_t)__clzll((long long)(uint64_t)diff[j]));
      } else {
        d = 31u - (uint32_t)__clz((int)(i ^ (i + 1)));
      }
      b.delta[i] = (uint8_t)d;
    }
  }
}

constexpr uint64_t kBuildSmallMax = 4 * kSmallBlock;
// Patches up to which the one workgroup also clears the patch slabs of a build
// with fp64 records (208 bytes each); above, a launch of its own does.  Build of
// one sphere, cleared here / by a launch: 64 patches 80 / 88 us, 2,048 86 / 85,
// 4,096 90 / 84, 16,384 126 / 86.
constexpr uint64_t kClearSmallMax = 2048;
bool build_is_small(uint64_t n) { return n > 0 && n <= kBuildSmallMax; }

template <typename K>
static void build_small(const ElemInput& in, const BuildBufs& b, int clear_k64, hipStream_t s) {
  const dim3 g(1), t(kSmallBlock);
  if (in.n <= 1 * kSmallBlock) hipLaunchKernelGGL((k_build_small<K, 1>), g, t, 0, s, in, b, clear_k64);
  else if (in.n <= 2 * kSmallBlock) hipLaunchKernelGGL((k_build_small<K, 2>), g, t, 0, s, in, b, clear_k64);
  else hipLaunchKernelGGL((k_build_small<K, 4>), g, t, 0, s, in, b, clear_k64);
}

hipError_t launch_build_small(const ElemInput& in, const BuildBufs& b, int bits, hipStream_t s) {
  if (!build_is_small(in.n) || in.nv < 1 || b.od < 1 || !in.data) return hipErrorInvalidValue;
  if (in.kind == kSnapshot && !in.centroids) return hipErrorInvalidValue;
  int clear_k64 = b.rec64 != nullptr;
  if (clear_k64 && b.od > kClearSmallMax) {
    const hipError_t e = launch_patch_k64_init(b.patch_k64, b.od, s);
    if (e != hipSuccess) return e;
    clear_k64 = 0;
  }
  if (bits == 63) build_small<uint64_t>(in, b, clear_k64, s);
  else build_small<uint32_t>(in, b, clear_k64, s);
  return hipGetLastError();
}

}  // namespace dbvh
