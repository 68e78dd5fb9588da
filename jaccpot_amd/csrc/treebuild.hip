// Device construction of the fixed static-radix topology: the same spec as the
// host builder in topology.cpp (the role yggdrax's build_tree, tree geometry
// and build_interactions_and_neighbors play for the reference, called from
// jaccpot/runtime/fmm_state.py:630-800 and runtime/_interaction_cache.py:523,564),
// with bit-identical output:
//
//  * bounds by exact min/max reduction; 63-bit Morton codes on the cube they
//    span (floor((x - lo) * 2^21 / extent), clamped);
//  * stable radix sort of (code, input index) -> perm;
//  * L = ceil(N/leaf) buckets, binary radix tree over the leaf keys (code of
//    the leaf's first particle, leaf index as tie-break), one thread per
//    internal node (Karras 2012);
//  * depth by the parent chain; level schedules by sorting (level, node) keys;
//  * centres of mass per leaf in slot order, internal nodes level by level
//    from their children, plain mean for a massless node; radius = exact max
//    distance from the centre to the node's particles;
//  * dual-tree walk breadth first: every frontier item (a, b) is expanded in
//    parallel exactly as the host's depth-first walk expands it (self item ->
//    three child items; MAC (r_a + r_b)^2 <= theta^2 d^2, d > 0 -> far pair in
//    both directions; two leaves -> near pair in both directions; otherwise
//    split the larger-radius non-leaf node).  The walk's set of pairs does not
//    depend on the expansion order; sorting the packed (target, source) keys
//    gives the host's CSR (targets ascending, sources ascending).
//
// Floating-point expressions are evaluated without contraction so every sum,
// product, quotient and square root rounds exactly as the host's.
//
// Buffers are the caller's; the sorts and scans take a caller-provided
// scratch (jfm_sort_scratch_bytes, jfm_scan_scratch_bytes).  The walk's steps
// read and leave their counts on the device, so many are launched without the
// host looking at them; a list that does not fit its buffer is counted on and
// reported, and the caller walks again with larger ones.

#pragma clang fp contract(off)

#include <hip/hip_runtime.h>
#include <hipcub/device/device_radix_sort.hpp>
#include <hipcub/device/device_scan.hpp>

#include <cmath>
#include <cstdint>

#include "launch.hpp"

namespace jfm {
namespace {

constexpr int kMortonBits = 21;
constexpr int kBoundBlocks = 1024;
constexpr int kMaxTreeHeight = 128;

__device__ inline uint64_t spread3_dev(uint64_t v) {
  v &= 0x1FFFFFull;
  v = (v | (v << 32)) & 0x001F00000000FFFFull;
  v = (v | (v << 16)) & 0x001F0000FF0000FFull;
  v = (v | (v << 8)) & 0x100F00F00F00F00Full;
  v = (v | (v << 4)) & 0x10C30C30C30C30C3ull;
  v = (v | (v << 2)) & 0x1249249249249249ull;
  return v;
}

// ---------------------------------------------------------------------------
// bounds and Morton codes
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) bounds_partial_kernel(const double* __restrict__ pos, int64_t n,
                                                             double* __restrict__ partial, int32_t* __restrict__ bad) {
  __shared__ double red[6][256];
  double lo[3] = {pos[0], pos[1], pos[2]}, hi[3] = {pos[0], pos[1], pos[2]};
  int nonfinite = 0;
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) {
    for (int a = 0; a < 3; ++a) {
      const double v = pos[3 * i + a];
      nonfinite |= !isfinite(v);
      lo[a] = fmin(lo[a], v);
      hi[a] = fmax(hi[a], v);
    }
  }
  if (nonfinite) atomicOr(bad, 1);
  for (int a = 0; a < 3; ++a) {
    red[a][threadIdx.x] = lo[a];
    red[3 + a][threadIdx.x] = hi[a];
  }
  __syncthreads();
  for (int w = 128; w >= 1; w >>= 1) {
    if (threadIdx.x < w)
      for (int a = 0; a < 3; ++a) {
        red[a][threadIdx.x] = fmin(red[a][threadIdx.x], red[a][threadIdx.x + w]);
        red[3 + a][threadIdx.x] = fmax(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) partial[6 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) bounds_final_kernel(const double* __restrict__ partial, int blocks,
                                                           double* __restrict__ bounds6) {
  __shared__ double red[6][256];
  for (int a = 0; a < 6; ++a) red[a][threadIdx.x] = partial[a];
  for (int b = threadIdx.x; b < blocks; b += 256)
    for (int a = 0; a < 3; ++a) {
      red[a][threadIdx.x] = fmin(red[a][threadIdx.x], partial[6 * b + a]);
      red[3 + a][threadIdx.x] = fmax(red[3 + a][threadIdx.x], partial[6 * b + 3 + a]);
    }
  __syncthreads();
  for (int w = 128; w >= 1; w >>= 1) {
    if (threadIdx.x < w)
      for (int a = 0; a < 3; ++a) {
        red[a][threadIdx.x] = fmin(red[a][threadIdx.x], red[a][threadIdx.x + w]);
        red[3 + a][threadIdx.x] = fmax(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + w]);
      }
    __syncthreads();
  }
  if (threadIdx.x < 6) bounds6[threadIdx.x] = red[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) morton_kernel(const double* __restrict__ pos, int64_t n,
                                                     const double* __restrict__ bounds6, uint64_t* __restrict__ codes,
                                                     int32_t* __restrict__ index) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const double lo[3] = {bounds6[0], bounds6[1], bounds6[2]};
  double extent = fmax(bounds6[3] - lo[0], fmax(bounds6[4] - lo[1], bounds6[5] - lo[2]));
  if (!(extent > 0.0)) extent = 1.0;
  const double scale = static_cast<double>(1 << kMortonBits) / extent;
  const double qmax = static_cast<double>((1 << kMortonBits) - 1);
  uint64_t q[3];
  for (int a = 0; a < 3; ++a) {
    double v = floor((pos[3 * i + a] - lo[a]) * scale);
    v = fmin(fmax(v, 0.0), qmax);
    q[a] = static_cast<uint64_t>(v);
  }
  codes[i] = (spread3_dev(q[0]) << 2) | (spread3_dev(q[1]) << 1) | spread3_dev(q[2]);
  index[i] = static_cast<int32_t>(i);
}

// ---------------------------------------------------------------------------
// radix tree over leaf keys
// ---------------------------------------------------------------------------

struct LeafKeys {
  const uint64_t* sorted;
  int32_t leaf, L;
  __device__ uint64_t key(int32_t l) const { return sorted[int64_t(l) * leaf]; }
  // common prefix of (code, index) keys: code bits, then index bits
  __device__ int delta(int32_t i, int32_t j) const {
    const uint64_t a = key(i), b = key(j);
    if (a != b) return __clzll(static_cast<long long>(a ^ b));
    return 64 + __clz(static_cast<int>(static_cast<uint32_t>(i ^ j)));
  }
  __device__ int delta_safe(int32_t i, int32_t j) const { return (j < 0 || j >= L) ? -1 : delta(i, j); }
};

__global__ void __launch_bounds__(256) radix_tree_kernel(LeafKeys keys, int64_t n, int32_t* __restrict__ parent,
                                                         int32_t* __restrict__ left, int32_t* __restrict__ right,
                                                         int32_t* __restrict__ range) {
  const int32_t L = keys.L, I = L - 1;
  const int32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t < L) {  // leaf: its own bucket of slots
    const int32_t node = I + t;
    range[2 * node] = static_cast<int32_t>(int64_t(t) * keys.leaf);
    range[2 * node + 1] = static_cast<int32_t>(min<int64_t>((int64_t(t) + 1) * keys.leaf, n) - 1);
  }
  if (t == 0) parent[0] = -1;
  if (t >= I) return;
  const int32_t i = t;
  int32_t first, last;
  if (i == 0) {
    first = 0;
    last = L - 1;
  } else {
    const int d = (keys.delta_safe(i, i + 1) - keys.delta_safe(i, i - 1)) > 0 ? 1 : -1;
    const int dmin = keys.delta_safe(i, i - d);
    int32_t lmax = 2;
    while (keys.delta_safe(i, i + lmax * d) > dmin) lmax *= 2;
    int32_t len = 0;
    for (int32_t s = lmax / 2; s >= 1; s /= 2)
      if (keys.delta_safe(i, i + (len + s) * d) > dmin) len += s;
    const int32_t j = i + len * d;
    first = min(i, j);
    last = max(i, j);
  }
  const int common = keys.delta(first, last);
  int32_t split = first, step = last - first;
  do {
    step = (step + 1) >> 1;
    const int32_t nw = split + step;
    if (nw < last && keys.delta(first, nw) > common) split = nw;
  } while (step > 1);
  const int32_t lc = (split == first) ? I + split : split;
  const int32_t rc = (split + 1 == last) ? I + split + 1 : split + 1;
  left[i] = lc;
  right[i] = rc;
  parent[lc] = i;
  parent[rc] = i;
  range[2 * i] = static_cast<int32_t>(int64_t(first) * keys.leaf);
  range[2 * i + 1] = static_cast<int32_t>(min<int64_t>((int64_t(last) + 1) * keys.leaf, n) - 1);
}

// depth by the parent chain; a chain longer than kMaxTreeHeight flags an error
__global__ void __launch_bounds__(256) depth_kernel(int32_t nodes, const int32_t* __restrict__ parent,
                                                    int32_t* __restrict__ depth, int32_t* __restrict__ max_depth,
                                                    int32_t* __restrict__ bad) {
  const int32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= nodes) return;
  int32_t d = 0, j = k;
  while (parent[j] >= 0 && d <= kMaxTreeHeight) {
    j = parent[j];
    ++d;
  }
  if (d > kMaxTreeHeight) atomicOr(bad, 2);
  depth[k] = d;
  atomicMax(max_depth, d);
}

// (level, node) keys: M2M order = internal nodes deepest first, L2L order =
// non-root nodes shallowest first; ascending node index within a level.
__global__ void __launch_bounds__(256) level_keys_kernel(int32_t nodes, int32_t I, const int32_t* __restrict__ depth,
                                                         const int32_t* __restrict__ max_depth,
                                                         uint64_t* __restrict__ m2m_keys,
                                                         uint64_t* __restrict__ l2l_keys) {
  const int32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k >= nodes) return;
  const int32_t D = *max_depth;
  if (k < I) m2m_keys[k] = (uint64_t(D - depth[k]) << 32) | uint32_t(k);
  if (k >= 1) l2l_keys[k - 1] = (uint64_t(depth[k] - 1) << 32) | uint32_t(k);
}

// ---------------------------------------------------------------------------
// geometry
// ---------------------------------------------------------------------------

struct Particles {
  const double* pos;   // input order [n][3]
  const double* mass;  // input order [n]
  const int32_t* perm;
  __device__ double x(int64_t slot, int a) const { return pos[3 * int64_t(perm[slot]) + a]; }
  __device__ double m(int64_t slot) const { return mass[perm[slot]]; }
};

__device__ inline void mean_of(const Particles& P, int64_t a, int64_t b, double* c) {
  double s[3] = {0, 0, 0};
  for (int64_t i = a; i <= b; ++i)
    for (int k = 0; k < 3; ++k) s[k] += P.x(i, k);
  for (int k = 0; k < 3; ++k) c[k] = s[k] / static_cast<double>(b - a + 1);
}

__global__ void __launch_bounds__(256) leaf_geometry_kernel(Particles P, int32_t L, int32_t I,
                                                            const int32_t* __restrict__ range,
                                                            double* __restrict__ mass, double* __restrict__ center) {
  const int32_t l = blockIdx.x * 256 + threadIdx.x;
  if (l >= L) return;
  const int32_t node = I + l;
  const int64_t a = range[2 * node], b = range[2 * node + 1];
  double tot = 0.0, s[3] = {0, 0, 0};
  for (int64_t i = a; i <= b; ++i) tot += P.m(i);
  for (int64_t i = a; i <= b; ++i) {
    const double mi = P.m(i);
    for (int k = 0; k < 3; ++k) s[k] += mi * P.x(i, k);
  }
  mass[node] = tot;
  if (tot > 0.0) {
    for (int k = 0; k < 3; ++k) center[3 * node + k] = s[k] / tot;
  } else {
    mean_of(P, a, b, &center[3 * node]);
  }
}

__device__ inline void internal_geometry(Particles P, int32_t node, const int32_t* __restrict__ left,
                                         const int32_t* __restrict__ right, const int32_t* __restrict__ range,
                                         double* __restrict__ mass, double* __restrict__ center) {
  const int32_t lc = left[node], rc = right[node];
  const double ml = mass[lc], mr = mass[rc];
  const double tot = ml + mr;
  mass[node] = tot;
  if (tot > 0.0) {
    for (int k = 0; k < 3; ++k) center[3 * node + k] = (ml * center[3 * lc + k] + mr * center[3 * rc + k]) / tot;
  } else {
    mean_of(P, range[2 * node], range[2 * node + 1], &center[3 * node]);
  }
}

__global__ void __launch_bounds__(256) internal_geometry_kernel(Particles P, int32_t count,
                                                                const int32_t* __restrict__ level_nodes,
                                                                const int32_t* __restrict__ left,
                                                                const int32_t* __restrict__ right,
                                                                const int32_t* __restrict__ range,
                                                                double* __restrict__ mass,
                                                                double* __restrict__ center) {
  const int32_t q = blockIdx.x * 256 + threadIdx.x;
  if (q < count) internal_geometry(P, level_nodes[q], left, right, range, mass, center);
}

// A run of small levels in one workgroup, a barrier between the levels.  The line lies
// where a level takes about as long as one more launch (256 nodes 1.7 us in a run,
// 1024 3.7; wider ones by themselves 3.5).
constexpr int kGeometrySpanThreads = 512;
constexpr int kGeometrySpanNodes = 2 * kGeometrySpanThreads;

__global__ void __launch_bounds__(kGeometrySpanThreads) internal_geometry_span_kernel(
    Particles P, LevelSpan span, const int32_t* __restrict__ level_nodes, const int32_t* __restrict__ left,
    const int32_t* __restrict__ right, const int32_t* __restrict__ range, double* __restrict__ mass,
    double* __restrict__ center) {
  for (int lev = 0; lev < span.n; ++lev) {
    for (int k = span.off[lev] + threadIdx.x; k < span.off[lev + 1]; k += kGeometrySpanThreads)
      internal_geometry(P, level_nodes[k], left, right, range, mass, center);
    __syncthreads();
  }
}

// tree-order copy of the positions, so the radius sweeps read contiguously
// (and the zeroing of the radius work counter)
__global__ void __launch_bounds__(256) sorted_positions_kernel(Particles P, int64_t n, double* __restrict__ xs,
                                                               int32_t* __restrict__ work_count) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  if (i == 0) *work_count = 0;
  for (int a = 0; a < 3; ++a) xs[3 * i + a] = P.x(i, a);
}

constexpr int kSmallRadius = 2048;  // nodes up to this many particles: one wave each
constexpr int kRadiusChunk = 4096;  // particles per work item of a larger node
constexpr int kRadiusBlocks = 2048;

__device__ inline double dist2(const double* __restrict__ xs, int64_t i, double cx, double cy, double cz) {
  const double dx = xs[3 * i] - cx, dy = xs[3 * i + 1] - cy, dz = xs[3 * i + 2] - cz;
  return dx * dx + dy * dy + dz * dz;
}

// One wave per node: a node of at most kSmallRadius particles gets its radius,
// a larger one is cut into (node, chunk) work items for radius_big_kernel, with
// its radius entry zeroed to hold the squared maximum's bits meanwhile.  One
// workgroup per large node left the root and its neighbours running alone on a
// few CUs (269 us of a 1M-body build; 40 us in chunks).
__global__ void __launch_bounds__(256) radius_small_kernel(const double* __restrict__ xs, int32_t nodes,
                                                           const int32_t* __restrict__ range,
                                                           const double* __restrict__ center,
                                                           double* __restrict__ radius, int2* __restrict__ work,
                                                           int32_t work_cap, int32_t* __restrict__ work_count) {
  const int32_t node = blockIdx.x * 4 + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (node >= nodes) return;  // whole waves leave together
  const int64_t a = range[2 * node], b = range[2 * node + 1];
  if (b - a + 1 > kSmallRadius) {
    const int chunks = static_cast<int>((b - a + kRadiusChunk) / kRadiusChunk);
    int at = 0;
    if (lane == 0) {
      radius[node] = 0.0;
      at = atomicAdd(work_count, chunks);
    }
    at = __shfl(at, 0);
    for (int c = lane; c < chunks; c += 64)
      if (at + c < work_cap) work[at + c] = make_int2(node, c);
    return;
  }
  const double cx = center[3 * node], cy = center[3 * node + 1], cz = center[3 * node + 2];
  double best = 0.0;
  for (int64_t i = a + lane; i <= b; i += 64) best = fmax(best, dist2(xs, i, cx, cy, cz));
  for (int off = 32; off >= 1; off >>= 1) best = fmax(best, __shfl_xor(best, off));
  if (lane == 0) radius[node] = sqrt(best);
}

// The larger nodes' work items, dealt to a fixed grid; the squared maxima of a
// node's items meet by an integer maximum of their bits (order preserving for
// non-negative doubles, so the result does not depend on the order).
__global__ void __launch_bounds__(256) radius_big_kernel(const double* __restrict__ xs,
                                                         const int32_t* __restrict__ range,
                                                         const double* __restrict__ center,
                                                         const int2* __restrict__ work, int32_t work_cap,
                                                         const int32_t* __restrict__ work_count,
                                                         double* __restrict__ radius) {
  const int32_t count = min(*work_count, work_cap);
  for (int32_t w = blockIdx.x * 4 + threadIdx.x / 64; w < count; w += gridDim.x * 4) {  // a wave per item
    const int2 it = work[w];
    const int64_t a = range[2 * it.x] + int64_t(it.y) * kRadiusChunk;
    const int64_t e = min(a + kRadiusChunk - 1, int64_t(range[2 * it.x + 1]));
    const double cx = center[3 * it.x], cy = center[3 * it.x + 1], cz = center[3 * it.x + 2];
    double best = 0.0;
    int64_t i = a + threadIdx.x % 64;
    for (; i + 3 * 64 <= e; i += 4 * 64) {  // four independent loads in flight
      const double d0 = dist2(xs, i, cx, cy, cz), d1 = dist2(xs, i + 64, cx, cy, cz);
      const double d2 = dist2(xs, i + 128, cx, cy, cz), d3 = dist2(xs, i + 192, cx, cy, cz);
      best = fmax(best, fmax(fmax(d0, d1), fmax(d2, d3)));
    }
    for (; i <= e; i += 64) best = fmax(best, dist2(xs, i, cx, cy, cz));
    for (int off = 32; off >= 1; off >>= 1) best = fmax(best, __shfl_xor(best, off));
    if (threadIdx.x % 64 == 0)
      atomicMax(reinterpret_cast<unsigned long long*>(radius + it.x),
                static_cast<unsigned long long>(__double_as_longlong(best)));
  }
}

__global__ void __launch_bounds__(256) radius_root_kernel(int32_t nodes, const int32_t* __restrict__ range,
                                                          double* __restrict__ radius) {
  const int32_t node = blockIdx.x * 256 + threadIdx.x;
  if (node < nodes && range[2 * node + 1] - range[2 * node] + 1 > kSmallRadius) radius[node] = sqrt(radius[node]);
}

// ---------------------------------------------------------------------------
// dual-tree walk, breadth first
// ---------------------------------------------------------------------------

// State of a walk on the device (int64 each; the three counters that every
// workgroup adds to lie in cache lines of their own).
enum WalkSlot { kFarCount = 0, kNearCount = 16, kOverflow = 32, kFrontierNeed = 33, kSteps = 48 };
// kSteps + 2 t: items of the frontier that step t reads, + 1: the buffer it lies in.
enum WalkFull : int { kFullFrontier = 1, kFullFar = 2, kFullNear = 4 };

enum WalkCode : uint32_t { kNone = 0, kSelf = 1, kFar = 2, kNear = 3, kSplitA = 4, kSplitB = 5 };

struct Walk {
  int32_t I;
  double th2;
  const double4* node;  // centre and radius
  const int32_t* left;
  const int32_t* right;
  int2* frontier[2];
  int64_t frontier_cap;
  void* far;  // packed keys (target << shift) | source, uint32 where `wide` is 0
  int64_t far_cap;
  int32_t far_shift, far_wide;
  void* near;
  int64_t near_cap;
  int32_t near_shift, near_wide;
  unsigned long long* st;
};

__global__ void __launch_bounds__(256) pack_nodes_kernel(int32_t nodes, const double* __restrict__ C,
                                                         const double* __restrict__ R, double4* __restrict__ out) {
  const int32_t k = blockIdx.x * 256 + threadIdx.x;
  if (k < nodes) out[k] = make_double4(C[3 * k], C[3 * k + 1], C[3 * k + 2], R[k]);
}

__device__ inline uint32_t walk_code(const Walk& w, int2 it) {
  const int32_t a = it.x, b = it.y;
  if (a == b) return a < w.I ? kSelf : kNone;
  const double4 A = w.node[a], B = w.node[b];
  const double dx = A.x - B.x, dy = A.y - B.y, dz = A.z - B.z;
  const double d2 = dx * dx + dy * dy + dz * dz;
  const double s = A.w + B.w;
  const bool al = a >= w.I, bl = b >= w.I;
  if (d2 > 0.0 && s * s <= w.th2 * d2) return kFar;
  if (al && bl) return kNear;
  if (bl || (!al && A.w >= B.w)) return kSplitA;
  return kSplitB;
}

__device__ inline void put_pair(void* keys, int32_t wide, int32_t shift, int64_t o, uint32_t a, uint32_t b) {
  if (wide) {
    uint64_t* k = static_cast<uint64_t*>(keys) + o;
    k[0] = (uint64_t(a) << shift) | b;
    k[1] = (uint64_t(b) << shift) | a;
  } else {
    uint32_t* k = static_cast<uint32_t*>(keys) + o;
    k[0] = (a << shift) | b;
    k[1] = (b << shift) | a;
  }
}

// One tile of THREADS * rounds frontier items (rounds <= MAXR): every thread
// classifies its items, the counts of every (round, wave) are scanned in LDS,
// `reserve(items, far, near)` returns where the tile's outputs start (or -1 where
// a list is full) and the items are written there, neighbouring lanes next to
// each other.
template <int THREADS, int MAXR, typename Reserve>
__device__ inline void walk_tile(const Walk& w, const int2* __restrict__ in, int64_t n, int64_t base, int rounds,
                                 int2* __restrict__ out, Reserve reserve) {
  constexpr int WAVES = THREADS / 64;
  constexpr int CELLS = MAXR * WAVES;
  constexpr int PER = (CELLS + 63) / 64;  // cells of a lane of the wave that scans them
  __shared__ int32_t cell[3][64 * PER];
  __shared__ int64_t start[3];
  const int tid = threadIdx.x, lane = tid % 64, wv = tid / 64;
  const uint64_t below = (uint64_t(1) << lane) - 1;
  uint64_t codes = 0;
  for (int c = 0; c < 3; ++c)
    for (int k = tid; k < 64 * PER; k += THREADS) cell[c][k] = 0;
  __syncthreads();
#pragma unroll 4
  for (int r = 0; r < rounds; ++r) {
    const int64_t t = base + int64_t(r) * THREADS + tid;
    const uint32_t c = t < n ? walk_code(w, in[t]) : uint32_t(kNone);
    codes |= uint64_t(c) << (4 * r);
    const uint64_t self = __ballot(c == kSelf), split = __ballot(c >= kSplitA);
    const uint64_t fr = __ballot(c == kFar), nr = __ballot(c == kNear);
    if (lane == 0) {
      cell[0][r * WAVES + wv] = 3 * __popcll(self) + 2 * __popcll(split);
      cell[1][r * WAVES + wv] = 2 * __popcll(fr);
      cell[2][r * WAVES + wv] = 2 * __popcll(nr);
    }
  }
  __syncthreads();
  if (wv == 0) {
    int32_t total[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      int32_t own = 0;
      for (int k = 0; k < PER; ++k) own += cell[c][lane * PER + k];
      int32_t v = own;
      for (int o = 1; o < 64; o <<= 1) {
        const int32_t u = __shfl_up(v, o);
        if (lane >= o) v += u;
      }
      int32_t at = v - own;
      for (int k = 0; k < PER; ++k) {
        const int32_t count = cell[c][lane * PER + k];
        cell[c][lane * PER + k] = at;
        at += count;
      }
      total[c] = __shfl(v, 63);
    }
    if (lane < 3) start[lane] = reserve(lane, lane == 0 ? total[0] : lane == 1 ? total[1] : total[2]);
  }
  __syncthreads();
  const int64_t s0 = start[0], s1 = start[1], s2 = start[2];
  for (int r = 0; r < rounds; ++r) {
    const uint32_t c = uint32_t(codes >> (4 * r)) & 15u;
    const uint64_t self = __ballot(c == kSelf), split = __ballot(c >= kSplitA);
    const uint64_t fr = __ballot(c == kFar), nr = __ballot(c == kNear);
    if (c == kNone) continue;
    const int2 it = in[base + int64_t(r) * THREADS + tid];
    if (c == kFar) {
      if (s1 >= 0)
        put_pair(w.far, w.far_wide, w.far_shift, s1 + cell[1][r * WAVES + wv] + 2 * __popcll(fr & below),
                 uint32_t(it.x), uint32_t(it.y));
    } else if (c == kNear) {
      if (s2 >= 0)
        put_pair(w.near, w.near_wide, w.near_shift, s2 + cell[2][r * WAVES + wv] + 2 * __popcll(nr & below),
                 uint32_t(it.x - w.I), uint32_t(it.y - w.I));
    } else if (s0 >= 0) {
      int2* o = out + s0 + cell[0][r * WAVES + wv] + 3 * __popcll(self & below) + 2 * __popcll(split & below);
      if (c == kSelf) {
        const int32_t la = w.left[it.x], ra = w.right[it.x];
        o[0] = make_int2(la, ra);
        o[1] = make_int2(ra, ra);
        o[2] = make_int2(la, la);
      } else if (c == kSplitA) {
        o[0] = make_int2(w.right[it.x], it.y);
        o[1] = make_int2(w.left[it.x], it.y);
      } else {
        o[0] = make_int2(it.x, w.right[it.y]);
        o[1] = make_int2(it.x, w.left[it.y]);
      }
    }
  }
  __syncthreads();  // cell and start are reused by the next tile
}

// One breadth-first step over a fixed grid.  Bound by the additions to the three
// shared counters, one each for a tile and one after another across the XCDs: so
// one workgroup of 1024 threads per CU, with tiles that grow with the frontier (up
// to 16384 items), instead of four of 256 (up to 4096 items): 1M Plummer bodies, leaf
// 16, 48 steps 1400 -> 1136 us; a 256k galaxy, 72 steps 787 -> 560 us; two of 512
// take 1201 and 606 us.  Loads of four rounds issued together changed nothing at 1M
// and cost 200 us in the galaxy's short steps.
constexpr int kWalkThreads = 1024;
constexpr int kWalkRounds = 16;
constexpr int kWalkBlocks = 256;

__global__ void __launch_bounds__(kWalkThreads) walk_step_kernel(Walk w, int32_t step) {
  unsigned long long* now = w.st + kSteps + 2 * step;
  const int64_t n = static_cast<int64_t>(now[0]);
  const int buf = static_cast<int>(now[1]);
  if (blockIdx.x == 0 && threadIdx.x == 0) now[3] = n > 0 ? 1 - buf : buf;
  // A frontier that did not fit shows in the count that the launch before left (the
  // unwritten entries are never read; this step leaves 0 items for the next).  The
  // overflow word would not do: other workgroups of this launch set it meanwhile, and
  // the waves of one workgroup have to leave together.
  if (n == 0 || n > w.frontier_cap) return;
  const int64_t most = int64_t(gridDim.x) * kWalkThreads;
  const int rounds = static_cast<int>(min(int64_t(kWalkRounds), (n + most - 1) / most));
  const int64_t tile = int64_t(rounds) * kWalkThreads;
  for (int64_t base = blockIdx.x * tile; base < n; base += gridDim.x * tile)
    walk_tile<kWalkThreads, kWalkRounds>(
        w, w.frontier[buf], n, base, rounds, w.frontier[1 - buf], [&](int list, int32_t count) -> int64_t {
          if (count == 0) return 0;
          unsigned long long* ctr = list == 0 ? now + 2 : list == 1 ? w.st + kFarCount : w.st + kNearCount;
          const int64_t at = static_cast<int64_t>(atomicAdd(ctr, static_cast<unsigned long long>(count)));
          const int64_t cap = list == 0 ? w.frontier_cap : list == 1 ? w.far_cap : w.near_cap;
          if (at + count <= cap) return at;
          atomicOr(w.st + kOverflow, static_cast<unsigned long long>(list == 0 ? kFullFrontier : list == 1 ? kFullFar : kFullNear));
          if (list == 0) atomicMax(w.st + kFrontierNeed, static_cast<unsigned long long>(at + count));
          return -1;
        });
}

// Steps of small frontiers (the first and last of a walk, all of a small tree's)
// in one workgroup until the frontier is empty or outgrows kWalkSmall items.
constexpr int kWalkSmallThreads = 1024;
constexpr int kWalkSmall = 2 * kWalkSmallThreads;

__global__ void __launch_bounds__(kWalkSmallThreads) walk_small_kernel(Walk w, int32_t step) {
  __shared__ int64_t next[3];  // items of the next frontier, far and near entries so far
  unsigned long long* now = w.st + kSteps + 2 * step;
  int64_t n = static_cast<int64_t>(now[0]);
  int buf = static_cast<int>(now[1]);
  bool full = n > w.frontier_cap;
  if (threadIdx.x == 0) {
    next[1] = static_cast<int64_t>(w.st[kFarCount]);
    next[2] = static_cast<int64_t>(w.st[kNearCount]);
  }
  // n items with n <= kWalkSmall make at most 3 n, and a walk is finite: every
  // step replaces an item by items of strictly smaller nodes
  while (n > 0 && n <= kWalkSmall && !full) {
    if (threadIdx.x == 0) next[0] = 0;
    const int rounds = n > kWalkSmallThreads ? 2 : 1;
    walk_tile<kWalkSmallThreads, 2>(w, w.frontier[buf], n, 0, rounds, w.frontier[1 - buf],
                                    [&](int list, int32_t count) -> int64_t {
                                      const int64_t at = next[list];
                                      next[list] = at + count;
                                      const int64_t cap = list == 0 ? w.frontier_cap : list == 1 ? w.far_cap : w.near_cap;
                                      if (at + count <= cap) return at;
                                      atomicOr(w.st + kOverflow, static_cast<unsigned long long>(
                                                                    list == 0 ? kFullFrontier : list == 1 ? kFullFar : kFullNear));
                                      if (list == 0) atomicMax(w.st + kFrontierNeed, static_cast<unsigned long long>(at + count));
                                      return -1;
                                    });
    n = next[0];
    full = n > w.frontier_cap;
    buf = 1 - buf;
    __syncthreads();  // everyone has read next[0]
  }
  if (threadIdx.x == 0) {
    w.st[kFarCount] = static_cast<unsigned long long>(next[1]);
    w.st[kNearCount] = static_cast<unsigned long long>(next[2]);
    now[2] = static_cast<unsigned long long>(n);
    now[3] = static_cast<unsigned long long>(buf);
  }
}

// ---------------------------------------------------------------------------
// sorted (row << 32 | col) keys -> CSR
// ---------------------------------------------------------------------------

__global__ void __launch_bounds__(256) csr_offsets_kernel(const uint64_t* __restrict__ keys, int64_t K, int32_t rows,
                                                          int32_t* __restrict__ off) {
  const int32_t r = blockIdx.x * 256 + threadIdx.x;
  if (r > rows) return;
  const uint64_t want = uint64_t(r) << 32;
  int64_t lo = 0, hi = K;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (keys[mid] < want) lo = mid + 1;
    else hi = mid;
  }
  off[r] = static_cast<int32_t>(lo);
}

__global__ void __launch_bounds__(256) low_words_kernel(const uint64_t* __restrict__ keys, int64_t K,
                                                        int32_t* __restrict__ col) {
  const int64_t k = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (k < K) col[k] = static_cast<int32_t>(keys[k] & 0xFFFFFFFFull);
}

// the same from keys (row << shift) | col of either width
template <typename K>
__global__ void __launch_bounds__(256) packed_offsets_kernel(const K* __restrict__ keys, int64_t n, int32_t shift,
                                                             int32_t rows, int32_t* __restrict__ off) {
  const int32_t r = blockIdx.x * 256 + threadIdx.x;
  if (r > rows) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (static_cast<int64_t>(keys[mid] >> shift) < r) lo = mid + 1;
    else hi = mid;
  }
  off[r] = static_cast<int32_t>(lo);
}

template <typename K>
__global__ void __launch_bounds__(256) packed_cols_kernel(const K* __restrict__ keys, int64_t n, K mask,
                                                          int32_t* __restrict__ col) {
  const int64_t k = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (k < n) col[k] = static_cast<int32_t>(keys[k] & mask);
}

inline unsigned grid_for(int64_t n, int per_block = 256) {
  return static_cast<unsigned>((n + per_block - 1) / per_block);
}

inline int key_bits(uint64_t max_key) {
  int bits = 0;
  while (bits < 64 && (max_key >> bits) != 0) ++bits;
  return bits;
}

}  // namespace
}  // namespace jfm

using jfm::fail;

extern "C" {

int32_t jfm_tree_bounds_scratch_doubles(void) { return 6 * jfm::kBoundBlocks; }

int32_t jfm_tree_bounds(void* stream, const double* pos, int64_t n, int32_t given, double* scratch, double* bounds6,
                        int32_t* flags) {
  if (!pos || !scratch || !bounds6 || !flags || n < 1) return fail(JFM_ERR_ARG, "jfm_tree_bounds: bad argument");
  const int blocks = static_cast<int>(std::min<int64_t>(jfm::kBoundBlocks, (n + 255) / 256));
  hipLaunchKernelGGL(jfm::bounds_partial_kernel, dim3(blocks), dim3(256), 0, jfm::as_stream(stream), pos, n, scratch,
                     flags);
  if (!given)
    hipLaunchKernelGGL(jfm::bounds_final_kernel, dim3(1), dim3(256), 0, jfm::as_stream(stream), scratch, blocks,
                       bounds6);
  return jfm::check_launch("jfm_tree_bounds");
}

int32_t jfm_tree_morton(void* stream, const double* pos, int64_t n, const double* bounds6, uint64_t* codes,
                        int32_t* index) {
  if (!pos || !bounds6 || !codes || !index || n < 1 || n > (int64_t(1) << 30))
    return fail(JFM_ERR_ARG, "jfm_tree_morton: bad argument");
  hipLaunchKernelGGL(jfm::morton_kernel, dim3(jfm::grid_for(n)), dim3(256), 0, jfm::as_stream(stream), pos, n,
                     bounds6, codes, index);
  return jfm::check_launch("jfm_tree_morton");
}

int32_t jfm_sort_scratch_bytes(int64_t n, int32_t with_values, int64_t* bytes) {
  if (!bytes || n < 0 || n > INT32_MAX) return fail(JFM_ERR_ARG, "jfm_sort_scratch_bytes: bad argument");
  size_t b = 0;
  hipError_t e;
  if (with_values)
    e = hipcub::DeviceRadixSort::SortPairs(nullptr, b, static_cast<const uint64_t*>(nullptr),
                                           static_cast<uint64_t*>(nullptr), static_cast<const int32_t*>(nullptr),
                                           static_cast<int32_t*>(nullptr), static_cast<int>(n), 0, 64);
  else
    e = hipcub::DeviceRadixSort::SortKeys(nullptr, b, static_cast<const uint64_t*>(nullptr),
                                          static_cast<uint64_t*>(nullptr), static_cast<int>(n), 0, 64);
  if (e != hipSuccess) return fail(JFM_ERR_HIP, std::string("jfm_sort_scratch_bytes: ") + hipGetErrorString(e));
  *bytes = static_cast<int64_t>(b);
  return JFM_OK;
}

int32_t jfm_sort_u64(void* stream, int64_t n, int32_t end_bit, const uint64_t* keys_in, uint64_t* keys_out,
                     const int32_t* vals_in, int32_t* vals_out, void* scratch, int64_t scratch_bytes) {
  if (n < 0 || n > INT32_MAX || end_bit < 1 || end_bit > 64 || (n > 0 && (!keys_in || !keys_out)) ||
      ((vals_in == nullptr) != (vals_out == nullptr)))
    return fail(JFM_ERR_ARG, "jfm_sort_u64: bad argument");
  if (n == 0) return JFM_OK;
  int64_t need = 0;
  if (int32_t rc = jfm_sort_scratch_bytes(n, vals_in != nullptr, &need)) return rc;
  if (!scratch || scratch_bytes < need) return fail(JFM_ERR_ARG, "jfm_sort_u64: scratch too small");
  size_t b = static_cast<size_t>(scratch_bytes);
  hipError_t e;
  if (vals_in)
    e = hipcub::DeviceRadixSort::SortPairs(scratch, b, keys_in, keys_out, vals_in, vals_out, static_cast<int>(n), 0,
                                           end_bit, jfm::as_stream(stream));
  else
    e = hipcub::DeviceRadixSort::SortKeys(scratch, b, keys_in, keys_out, static_cast<int>(n), 0, end_bit,
                                          jfm::as_stream(stream));
  if (e != hipSuccess) return fail(JFM_ERR_HIP, std::string("jfm_sort_u64: ") + hipGetErrorString(e));
  return jfm::check_launch("jfm_sort_u64");
}

int32_t jfm_tree_radix(void* stream, int64_t n, int32_t leaf_size, const uint64_t* sorted_codes, int32_t* parent,
                       int32_t* left, int32_t* right, int32_t* node_range) {
  if (n < 1 || n > (int64_t(1) << 30) || leaf_size < 1 || !sorted_codes || !parent || !node_range)
    return fail(JFM_ERR_ARG, "jfm_tree_radix: bad argument");
  const int32_t L = static_cast<int32_t>((n + leaf_size - 1) / leaf_size);
  if (L > 1 && (!left || !right)) return fail(JFM_ERR_ARG, "jfm_tree_radix: left/right NULL");
  jfm::LeafKeys keys{sorted_codes, leaf_size, L};
  hipLaunchKernelGGL(jfm::radix_tree_kernel, dim3(jfm::grid_for(L)), dim3(256), 0, jfm::as_stream(stream), keys, n,
                     parent, left, right, node_range);
  return jfm::check_launch("jfm_tree_radix");
}

int32_t jfm_tree_levels(void* stream, int32_t nodes, int32_t I, const int32_t* parent, int32_t* depth,
                        int32_t* max_depth, int32_t* flags, uint64_t* m2m_keys, uint64_t* l2l_keys) {
  if (nodes < 1 || I < 0 || !parent || !depth || !max_depth || !flags || (I > 0 && (!m2m_keys || !l2l_keys)))
    return fail(JFM_ERR_ARG, "jfm_tree_levels: bad argument");
  hipStream_t s = jfm::as_stream(stream);
  hipLaunchKernelGGL(jfm::depth_kernel, dim3(jfm::grid_for(nodes)), dim3(256), 0, s, nodes, parent, depth, max_depth,
                     flags);
  if (I > 0)
    hipLaunchKernelGGL(jfm::level_keys_kernel, dim3(jfm::grid_for(nodes)), dim3(256), 0, s, nodes, I, depth,
                       max_depth, m2m_keys, l2l_keys);
  return jfm::check_launch("jfm_tree_levels");
}

int32_t jfm_tree_leaf_geometry(void* stream, int32_t L, int32_t I, const double* pos, const double* mass,
                               const int32_t* perm, const int32_t* node_range, double* node_mass, double* center) {
  if (L < 1 || !pos || !mass || !perm || !node_range || !node_mass || !center)
    return fail(JFM_ERR_ARG, "jfm_tree_leaf_geometry: bad argument");
  jfm::Particles P{pos, mass, perm};
  hipLaunchKernelGGL(jfm::leaf_geometry_kernel, dim3(jfm::grid_for(L)), dim3(256), 0, jfm::as_stream(stream), P, L, I,
                     node_range, node_mass, center);
  return jfm::check_launch("jfm_tree_leaf_geometry");
}

int32_t jfm_tree_level_geometry(void* stream, int32_t count, const int32_t* level_nodes, const double* pos,
                                const double* mass, const int32_t* perm, const int32_t* left, const int32_t* right,
                                const int32_t* node_range, double* node_mass, double* center) {
  if (count < 0 || (count > 0 && (!level_nodes || !pos || !mass || !perm || !left || !right || !node_range ||
                                  !node_mass || !center)))
    return fail(JFM_ERR_ARG, "jfm_tree_level_geometry: bad argument");
  if (count == 0) return JFM_OK;
  jfm::Particles P{pos, mass, perm};
  hipLaunchKernelGGL(jfm::internal_geometry_kernel, dim3(jfm::grid_for(count)), dim3(256), 0, jfm::as_stream(stream),
                     P, count, level_nodes, left, right, node_range, node_mass, center);
  return jfm::check_launch("jfm_tree_level_geometry");
}

int32_t jfm_tree_geometry_pass(void* stream, const int32_t* lev_off_host, int32_t nlev, const int32_t* level_nodes,
                               const double* pos, const double* mass, const int32_t* perm, const int32_t* left,
                               const int32_t* right, const int32_t* node_range, double* node_mass, double* center) {
  if (!jfm::valid_levels(lev_off_host, nlev)) return fail(JFM_ERR_ARG, "jfm_tree_geometry_pass: bad level table");
  if (nlev == 0 || lev_off_host[nlev] == lev_off_host[0]) return JFM_OK;
  if (!level_nodes || !pos || !mass || !perm || !left || !right || !node_range || !node_mass || !center)
    return fail(JFM_ERR_ARG, "jfm_tree_geometry_pass: bad argument");
  jfm::Particles P{pos, mass, perm};
  hipStream_t s = jfm::as_stream(stream);
  jfm::for_level_spans(
      lev_off_host, nlev, jfm::kGeometrySpanNodes,
      [&](const jfm::LevelSpan& sp) {
        hipLaunchKernelGGL(jfm::internal_geometry_span_kernel, dim3(1), dim3(jfm::kGeometrySpanThreads), 0, s, P, sp,
                           level_nodes, left, right, node_range, node_mass, center);
      },
      [&](int32_t a, int32_t count) {
        hipLaunchKernelGGL(jfm::internal_geometry_kernel, dim3(jfm::grid_for(count)), dim3(256), 0, s, P, count,
                           level_nodes + a, left, right, node_range, node_mass, center);
      });
  return jfm::check_launch("jfm_tree_geometry_pass");
}

int64_t jfm_tree_radius_work(int32_t nodes, int64_t n, int32_t max_depth) {
  if (nodes < 1 || n < 1 || max_depth < 0) return -1;
  // nodes of one depth are disjoint: at most n / kSmallRadius large ones, whose
  // chunks are at most n / kRadiusChunk full ones and one more each
  return (n / jfm::kRadiusChunk + n / jfm::kSmallRadius + 1) * (int64_t(max_depth) + 1);
}

int32_t jfm_tree_radius(void* stream, int32_t nodes, int64_t n, const double* pos, const int32_t* perm,
                        const int32_t* node_range, const double* center, double* scratch, int32_t* work,
                        int64_t work_cap, double* radius) {
  if (nodes < 1 || n < 1 || !pos || !perm || !node_range || !center || !scratch || !work || work_cap < 1 ||
      work_cap > INT32_MAX / 2 || !radius)
    return fail(JFM_ERR_ARG, "jfm_tree_radius: bad argument");
  hipStream_t s = jfm::as_stream(stream);
  jfm::Particles P{pos, nullptr, perm};
  int2* list = reinterpret_cast<int2*>(work + 2);
  const int32_t cap = static_cast<int32_t>(work_cap);
  hipLaunchKernelGGL(jfm::sorted_positions_kernel, dim3(jfm::grid_for(n)), dim3(256), 0, s, P, n, scratch, work);
  hipLaunchKernelGGL(jfm::radius_small_kernel, dim3(jfm::grid_for(nodes, 4)), dim3(256), 0, s, scratch, nodes,
                     node_range, center, radius, list, cap, work);
  if (n > jfm::kSmallRadius) {
    hipLaunchKernelGGL(jfm::radius_big_kernel, dim3(jfm::kRadiusBlocks), dim3(256), 0, s, scratch, node_range, center,
                       list, cap, work, radius);
    hipLaunchKernelGGL(jfm::radius_root_kernel, dim3(jfm::grid_for(nodes)), dim3(256), 0, s, nodes, node_range,
                       radius);
  }
  return jfm::check_launch("jfm_tree_radius");
}

int32_t jfm_tree_walk_state_words(int32_t steps) { return steps < 0 ? -1 : jfm::kSteps + 2 * (steps + 1); }

int32_t jfm_tree_pack_nodes(void* stream, int32_t nodes, const double* center, const double* radius, void* node4) {
  if (nodes < 1 || !center || !radius || !node4) return fail(JFM_ERR_ARG, "jfm_tree_pack_nodes: bad argument");
  hipLaunchKernelGGL(jfm::pack_nodes_kernel, dim3(jfm::grid_for(nodes)), dim3(256), 0, jfm::as_stream(stream), nodes,
                     center, radius, static_cast<double4*>(node4));
  return jfm::check_launch("jfm_tree_pack_nodes");
}

int32_t jfm_tree_walk(void* stream, int32_t I, const void* node4, const int32_t* left, const int32_t* right,
                      double theta, void* frontier0, void* frontier1, int64_t frontier_cap, void* far,
                      int64_t far_cap, int32_t far_shift, int32_t far_wide, void* near, int64_t near_cap,
                      int32_t near_shift, int32_t near_wide, uint64_t* state, int32_t first_step, int32_t groups,
                      int32_t steps_per_group) {
  if (I < 0 || !node4 || (I > 0 && (!left || !right)) || !(theta > 0.0) || !frontier0 || !frontier1 ||
      frontier_cap < 1 || !far || far_cap < 0 || !near || near_cap < 0 || !state || first_step < 0 || groups < 1 ||
      steps_per_group < 0)
    return fail(JFM_ERR_ARG, "jfm_tree_walk: bad argument");
  if (far_shift < 1 || far_shift > 31 || near_shift < 1 || near_shift > 31 || (!far_wide && far_shift > 16) ||
      (!near_wide && near_shift > 16))
    return fail(JFM_ERR_ARG, "jfm_tree_walk: key shifts out of range");
  hipStream_t s = jfm::as_stream(stream);
  jfm::Walk w;
  w.I = I;
  w.th2 = theta * theta;
  w.node = static_cast<const double4*>(node4);
  w.left = left;
  w.right = right;
  w.frontier[0] = static_cast<int2*>(frontier0);
  w.frontier[1] = static_cast<int2*>(frontier1);
  w.frontier_cap = frontier_cap;
  w.far = far;
  w.far_cap = far_cap;
  w.far_shift = far_shift;
  w.far_wide = far_wide;
  w.near = near;
  w.near_cap = near_cap;
  w.near_shift = near_shift;
  w.near_wide = near_wide;
  w.st = reinterpret_cast<unsigned long long*>(state);
  int32_t step = first_step;
  for (int32_t g = 0; g < groups; ++g) {
    hipLaunchKernelGGL(jfm::walk_small_kernel, dim3(1), dim3(jfm::kWalkSmallThreads), 0, s, w, step++);
    for (int32_t k = 0; k < steps_per_group; ++k)
      hipLaunchKernelGGL(jfm::walk_step_kernel, dim3(jfm::kWalkBlocks), dim3(jfm::kWalkThreads), 0, s, w, step++);
  }
  hipLaunchKernelGGL(jfm::walk_small_kernel, dim3(1), dim3(jfm::kWalkSmallThreads), 0, s, w, step);
  return jfm::check_launch("jfm_tree_walk");
}

int32_t jfm_sort_packed_scratch_bytes(int64_t n, int32_t wide, int64_t* bytes) {
  if (!bytes || n < 0 || n > INT32_MAX) return fail(JFM_ERR_ARG, "jfm_sort_packed_scratch_bytes: bad argument");
  size_t b = 0;
  hipError_t e;
  if (wide)
    e = hipcub::DeviceRadixSort::SortKeys(nullptr, b, static_cast<const uint64_t*>(nullptr),
                                          static_cast<uint64_t*>(nullptr), static_cast<int>(n), 0, 64);
  else
    e = hipcub::DeviceRadixSort::SortKeys(nullptr, b, static_cast<const uint32_t*>(nullptr),
                                          static_cast<uint32_t*>(nullptr), static_cast<int>(n), 0, 32);
  if (e != hipSuccess)
    return fail(JFM_ERR_HIP, std::string("jfm_sort_packed_scratch_bytes: ") + hipGetErrorString(e));
  *bytes = static_cast<int64_t>(b);
  return JFM_OK;
}

int32_t jfm_packed_to_csr(void* stream, int64_t n, int32_t wide, int32_t shift, const void* keys, void* sorted,
                          void* scratch, int64_t scratch_bytes, int32_t rows, int32_t* off, int32_t* col) {
  if (n < 0 || n > INT32_MAX || rows < 0 || shift < 1 || shift > 31 || (!wide && shift > 16) || !off ||
      (n > 0 && (!keys || !sorted || !col)))
    return fail(JFM_ERR_ARG, "jfm_packed_to_csr: bad argument");
  hipStream_t s = jfm::as_stream(stream);
  if (n > 0) {
    int64_t need = 0;
    if (int32_t rc = jfm_sort_packed_scratch_bytes(n, wide, &need)) return rc;
    if (!scratch || scratch_bytes < need) return fail(JFM_ERR_ARG, "jfm_packed_to_csr: scratch too small");
    size_t b = static_cast<size_t>(scratch_bytes);
    hipError_t e;
    if (wide)
      e = hipcub::DeviceRadixSort::SortKeys(scratch, b, static_cast<const uint64_t*>(keys),
                                            static_cast<uint64_t*>(sorted), static_cast<int>(n), 0, 2 * shift, s);
    else
      e = hipcub::DeviceRadixSort::SortKeys(scratch, b, static_cast<const uint32_t*>(keys),
                                            static_cast<uint32_t*>(sorted), static_cast<int>(n), 0, 2 * shift, s);
    if (e != hipSuccess) return fail(JFM_ERR_HIP, std::string("jfm_packed_to_csr: ") + hipGetErrorString(e));
  }
  const dim3 ro(jfm::grid_for(int64_t(rows) + 1)), co(jfm::grid_for(n > 0 ? n : 1));
  if (wide) {
    hipLaunchKernelGGL(jfm::packed_offsets_kernel<uint64_t>, ro, dim3(256), 0, s, static_cast<const uint64_t*>(sorted),
                       n, shift, rows, off);
    if (n > 0)
      hipLaunchKernelGGL(jfm::packed_cols_kernel<uint64_t>, co, dim3(256), 0, s, static_cast<const uint64_t*>(sorted),
                         n, (uint64_t(1) << shift) - 1, col);
  } else {
    hipLaunchKernelGGL(jfm::packed_offsets_kernel<uint32_t>, ro, dim3(256), 0, s, static_cast<const uint32_t*>(sorted),
                       n, shift, rows, off);
    if (n > 0)
      hipLaunchKernelGGL(jfm::packed_cols_kernel<uint32_t>, co, dim3(256), 0, s, static_cast<const uint32_t*>(sorted),
                         n, (uint32_t(1) << shift) - 1, col);
  }
  return jfm::check_launch("jfm_packed_to_csr");
}

int32_t jfm_scan_scratch_bytes(int64_t n, int64_t* bytes) {
  if (!bytes || n < 0 || n > INT32_MAX) return fail(JFM_ERR_ARG, "jfm_scan_scratch_bytes: bad argument");
  size_t b = 0;
  hipError_t e = hipcub::DeviceScan::ExclusiveSum(nullptr, b, static_cast<const int32_t*>(nullptr),
                                                  static_cast<int32_t*>(nullptr), static_cast<int>(n));
  if (e != hipSuccess) return fail(JFM_ERR_HIP, std::string("jfm_scan_scratch_bytes: ") + hipGetErrorString(e));
  *bytes = static_cast<int64_t>(b);
  return JFM_OK;
}

int32_t jfm_scan_i32(void* stream, int64_t n, const int32_t* in, int32_t* out, void* scratch, int64_t scratch_bytes) {
  if (n < 0 || n > INT32_MAX || (n > 0 && (!in || !out))) return fail(JFM_ERR_ARG, "jfm_scan_i32: bad argument");
  if (n == 0) return JFM_OK;
  int64_t need = 0;
  if (int32_t rc = jfm_scan_scratch_bytes(n, &need)) return rc;
  if (!scratch || scratch_bytes < need) return fail(JFM_ERR_ARG, "jfm_scan_i32: scratch too small");
  size_t b = static_cast<size_t>(scratch_bytes);
  hipError_t e = hipcub::DeviceScan::ExclusiveSum(scratch, b, in, out, static_cast<int>(n), jfm::as_stream(stream));
  if (e != hipSuccess) return fail(JFM_ERR_HIP, std::string("jfm_scan_i32: ") + hipGetErrorString(e));
  return jfm::check_launch("jfm_scan_i32");
}

int32_t jfm_keys_to_csr(void* stream, const uint64_t* sorted_keys, int64_t K, int32_t rows, int32_t* off,
                        int32_t* col) {
  if (K < 0 || K > INT32_MAX || rows < 0 || !off || (K > 0 && (!sorted_keys || !col)))
    return fail(JFM_ERR_ARG, "jfm_keys_to_csr: bad argument");
  hipStream_t s = jfm::as_stream(stream);
  hipLaunchKernelGGL(jfm::csr_offsets_kernel, dim3(jfm::grid_for(int64_t(rows) + 1)), dim3(256), 0, s, sorted_keys, K,
                     rows, off);
  if (K > 0)
    hipLaunchKernelGGL(jfm::low_words_kernel, dim3(jfm::grid_for(K)), dim3(256), 0, s, sorted_keys, K, col);
  return jfm::check_launch("jfm_keys_to_csr");
}

int32_t jfm_key_bits(uint64_t max_key) { return jfm::key_bits(max_key); }

}  // extern "C"
