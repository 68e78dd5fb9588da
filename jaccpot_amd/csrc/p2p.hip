// Near-field P2P: softened Newtonian sums over the self leaf and the near-list
// leaves of every target leaf, plus the fused evaluate entry point
// (L2P far field + P2P near field + combine + un-permute).
//
// Mapping: one workgroup per work item (a target leaf, or a range of its source
// slots).  Thread t owns one target of the leaf and one source partition.  The
// leaf's source slots (self leaf first, then the near leaves, each leaf_size
// slots wide) stream through LDS in tiles; inside a tile partition q takes slots
// q, q + NPART, ... so the lanes of a partition read one broadcast address per
// interaction and the tail tile stays balanced.  The next tile's sources are
// fetched into registers while the current one is consumed, with the near-list
// entries loaded one tile further ahead than the positions they address (no load
// is waited for before a tile's interactions).  Per-tile partial sums are folded
// into the running total with Kahan compensation when requested; the partitions
// are reduced through LDS in fixed order (deterministic).
//
// p2p_kernel takes leaves of 8, 16, 32 and 64 (softened, compensated) with the
// leaf width known at compile time; p2p_any_kernel everything else.

#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_math.hpp"
#include "launch.hpp"
#include "rows.hpp"
#include "xcd.hpp"

namespace jfm {
namespace {

constexpr int kThreads = 256;
constexpr int kWave = 64;
// LDS per CU is 160 KiB; a workgroup holding just over 1/(N+1) of it caps the
// CU at N workgroups (LDS is allocated in 512-byte granules).
constexpr int kLdsPerCu = 160 * 1024;
#ifndef JFM_P2P_BLOCKS_PER_CU
#define JFM_P2P_BLOCKS_PER_CU 5
#endif
constexpr int kP2PBlocksPerCu = JFM_P2P_BLOCKS_PER_CU;
constexpr int kP2PLdsBytes = (kLdsPerCu / (kP2PBlocksPerCu + 1) / 512 + 1) * 512;
static_assert(kP2PLdsBytes * (kP2PBlocksPerCu + 1) > kLdsPerCu && kP2PLdsBytes * kP2PBlocksPerCu <= kLdsPerCu,
              "P2P LDS reservation must cap the CU at kP2PBlocksPerCu workgroups");


template <typename T>
__device__ __forceinline__ void kahan_add(T& s, T& c, T v) {
  const T y = v - c;
  const T t = s + y;
  c = (t - s) - y;
  s = t;
}

// Leaf-granular fetch (leaf_size == WT, a power of two): thread t takes the LOADS
// consecutive slots first .. first + LOADS - 1, which lie in one source leaf, so
// one near-list entry and one slot decode serve them all.  fetch_list_leaf loads
// the entry (index clamped into range; an empty list reads `fallback`, a valid
// int32 location, and the value is discarded); the positions are loaded one tile
// later (slots past `total` or past the last particle become zero-mass sources).
template <int WT>
__device__ __forceinline__ int fetch_list_leaf(const int32_t* __restrict__ near_list, int nnear,
                                               const int32_t* __restrict__ fallback, int first) {
  const int32_t* list = nnear > 0 ? near_list : fallback;
  const int qi = static_cast<int>(static_cast<unsigned>(first) / WT);
  return list[min(max(qi - 1, 0), max(nnear - 1, 0))];
}

template <typename T, int WT, int LOADS>
__device__ __forceinline__ void fetch_positions_leaf(const T* __restrict__ pos4, int n, int leaf, int total, int first,
                                                     int v, V4<T> (&out)[LOADS], bool (&valid)[LOADS]) {
  const int qi = static_cast<int>(static_cast<unsigned>(first) / WT);
  const int o = static_cast<int>(static_cast<unsigned>(first) % WT);
  const int g0 = (qi > 0 ? v : leaf) * WT + o;
#pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    const int g = first + l < total ? g0 + l : n;
    valid[l] = g < n;
    out[l] = load4(pos4, min(g, n - 1));
  }
}

// float32 leaf-granular fetch through a raw buffer resource over the n rows
// of pos4 (16 bytes each).  The hardware range check returns zero for a row
// at or past n, i.e. a zero-mass source at the origin, so the missing rows of
// a ragged last leaf and slots past `total` (sent to row n) need no clamp and
// no mask, and the LOADS rows of a thread share one offset register (the row
// steps go into the instructions' immediate offsets).  Requires total and
// first to be multiples of LOADS (slot ranges are whole leaves); row offsets
// reach 16 * (n + WT) with WT <= 128 on this path, kept below 2^31.
constexpr int kBufMaxRows = (1 << 27) - 512;
static_assert((static_cast<int64_t>(kBufMaxRows) + 128) * 16 + 64 < (int64_t(1) << 31), "buffer offsets fit int32");
constexpr int kBufDword3 = 0x00020000;  // untyped 32-bit data format

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pos4_rsrc(const void* pos4, int n) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(pos4), static_cast<short>(0), n * 16, kBufDword3);
}

template <int WT, int LOADS>
__device__ __forceinline__ void fetch_positions_buf(__amdgpu_buffer_rsrc_t rsrc, int n, int leaf, int total,
                                                    int first, int v, V4<float> (&out)[LOADS]) {
  const int qi = static_cast<int>(static_cast<unsigned>(first) / WT);
  const int o = static_cast<int>(static_cast<unsigned>(first) % WT);
  const int g0 = first < total ? (qi > 0 ? v : leaf) * WT + o : n;
#pragma unroll
  for (int l = 0; l < LOADS; ++l)
    out[l] = __builtin_bit_cast(V4<float>, __builtin_amdgcn_raw_buffer_load_b128(rsrc, g0 * 16 + 16 * l, 0, 0));
}

// Work items split the source slots of leaves with long near lists: item k
// covers slots [s0, s1) of leaf `leaf`; part < 0 -> the item is the leaf's
// only one and writes the output rows, else it writes the unscaled partial
// sums of its targets to partials[(part * leaf_size + i) * 4 + c] and
// p2p_reduce_kernel adds a leaf's partials in item order.  leaf == NULL: one
// item per leaf covering all of its slots.
template <typename T>
struct P2PItems {
  const int32_t* leaf;
  const int32_t* s0;
  const int32_t* s1;
  const int32_t* part;
  T* partials;
  int32_t num_part;  // rows of partials (items with part >= num_part write nothing)
};

// Writes one target's sums: partial row of a split leaf, or output row (self
// potential removed, scaled by G).
template <typename T, bool POT>
__device__ __forceinline__ void put_sums(V4<T> r, T mass, int first, int i, int leaf_size, int part_out, T eps2, T G,
                                         const int32_t* __restrict__ out_index, T* __restrict__ acc,
                                         T* __restrict__ pot, int32_t accumulate, const P2PItems<T>& items) {
  if (part_out >= 0) {
    if (part_out >= items.num_part) return;
    T* dst = items.partials + (static_cast<int64_t>(part_out) * leaf_size + i) * 4;
    dst[0] = r.x;
    dst[1] = r.y;
    dst[2] = r.z;
    dst[3] = r.w;
    return;
  }
  T ap = r.w;
  if (POT && eps2 > T(0)) ap -= mass * fast_rsqrt(eps2);  // remove the softened self term
  const int64_t row = out_index ? out_index[first + i] : first + i;
  if (accumulate) {
    acc[3 * row + 0] += G * r.x;
    acc[3 * row + 1] += G * r.y;
    acc[3 * row + 2] += G * r.z;
    if (POT) pot[row] += -G * ap;
  } else {
    acc[3 * row + 0] = G * r.x;
    acc[3 * row + 1] = G * r.y;
    acc[3 * row + 2] = G * r.z;
    if (POT) pot[row] = -G * ap;
  }
}

// Workgroup size of the float32 leaf-granular path for leaves of 8: 128
// threads (16 source partitions), so each thread runs 64 interactions per
// 1024-source tile and the per-item set-up and partition reduction are shared
// by half as many threads as with 256.
#ifndef JFM_P2P_NARROW_THREADS
#define JFM_P2P_NARROW_THREADS 128
#endif
constexpr int kNarrowThreads = JFM_P2P_NARROW_THREADS;
// Narrow workgroups per CU (LDS reservation, as for the 256-thread form): 8 x
// 2 waves, so their registers leave room on every SIMD for a tree-pass wave.
#ifndef JFM_P2P_NARROW_BLOCKS_PER_CU
#define JFM_P2P_NARROW_BLOCKS_PER_CU 8
#endif

// Softened, compensated, leaf_size == WT (the compile-time slot decode and the
// leaf-granular fetch).  THREADS: workgroup size (kThreads, or kNarrowThreads for
// narrow leaves).
template <typename T, int WT, bool POT, int THREADS>
__global__ __launch_bounds__(THREADS) void p2p_kernel(const T* __restrict__ pos4, int32_t n,
                                                      const int32_t* __restrict__ near_off,
                                                      const int32_t* __restrict__ near_src, T eps2, T G,
                                                      const int32_t* __restrict__ out_index, T* __restrict__ acc,
                                                      T* __restrict__ pot, int32_t accumulate, P2PItems<T> items) {
  constexpr int leaf_size = WT;
  constexpr int NPART = THREADS / WT;
  constexpr int TILE = sizeof(T) == 4 ? 1024 : 512;
  constexpr int LOADS = TILE / THREADS;
  static_assert(2 * THREADS <= TILE, "reduction buffer must fit in the tile");
  // Slot s of a tile is stored at (s % LOADS) * ROW + s / LOADS, so the fetching thread writes its LOADS
  // slots to LOADS conflict-free rows and partition p still reads one address
  // per interaction, (p % LOADS) * ROW + p / LOADS + k * NPART / LOADS.  Rows
  // are padded so that the eight partitions a wave reads fall in distinct
  // 4-bank groups: with LOADS = 4 they sit in rows p % 4 at columns p / 4
  // (ROW = THREADS + 2), with LOADS = 8 in rows p at column 0 (ROW = THREADS + 1).
  static_assert(NPART % LOADS == 0, "partitions must cover the tile's rows evenly");
  constexpr bool BUF = sizeof(T) == 4;  // float32: buffer-resource fetch
  constexpr int ROW = THREADS + (LOADS == 8 ? 1 : 2);
  // The tile array is padded so that at most kBlocksPerCu workgroups share a
  // CU: the rest of its registers and LDS stay free for the tree-pass kernels
  // that run beside P2P in an overlapped step (at full occupancy their small
  // dependent launches wait for P2P workgroups to end).
  constexpr int kBlocksPerCu = THREADS == kThreads ? kP2PBlocksPerCu : JFM_P2P_NARROW_BLOCKS_PER_CU;
  constexpr int kPadBytes = (kLdsPerCu / (kBlocksPerCu + 1) / 512 + 1) * 512;
  constexpr int kTileElems = LOADS * ROW;
  constexpr int kPadElems = static_cast<int>(kPadBytes / sizeof(V4<T>));
  __shared__ V4<T> tile[kTileElems > kPadElems ? kTileElems : kPadElems];

  // XCD-aware order: workgroups are dealt round-robin to the XCDs, so hand
  // each XCD a contiguous run of leaves (neighbouring leaves share most of
  // their source leaves, which then stay in that XCD's L2).  Bijective:
  // XCD x < r owns q+1 leaves, the others q, where nblk = 8q + r.
  const int item = xcd_contiguous(blockIdx.x, gridDim.x);
  const int leaf = items.leaf ? items.leaf[item] : item;
  const int i = threadIdx.x % WT;
  const int part = threadIdx.x / WT;
  const int first = leaf * leaf_size;
  const int cnt = min(leaf_size, n - first);
  const V4<T> xi = load4(pos4, first + (i < cnt ? i : 0));
  const int nb = near_off[leaf];
  const int nsl = 1 + (near_off[leaf + 1] - nb);
  // slots [start, total) of the leaf's sequence (self leaf, then near leaves)
  const int start = items.leaf ? items.s0[item] : 0;
  const int total = items.leaf ? items.s1[item] : nsl * leaf_size;
  const int part_out = items.leaf ? items.part[item] : -1;

  // The next tile's sources are fetched into registers while the current
  // tile is being consumed, hiding the global-load latency behind the
  // interaction loop.
  V4<T> next[LOADS];
  bool ok[LOADS];
  int lst;  // near-list entry of the tile after `next`
  const int tid = threadIdx.x;
  const __amdgpu_buffer_rsrc_t rsrc = pos4_rsrc(pos4, BUF ? n : 0);  // used by the float32 fetch only
  lst = fetch_list_leaf<WT>(near_src + nb, nsl - 1, near_off, start + LOADS * tid);
  if constexpr (BUF)
    fetch_positions_buf<WT, LOADS>(rsrc, n, leaf, total, start + LOADS * tid, lst,
                                   reinterpret_cast<V4<float>(&)[LOADS]>(next));
  else
    fetch_positions_leaf<T, WT, LOADS>(pos4, n, leaf, total, start + LOADS * tid, lst, next, ok);
  lst = fetch_list_leaf<WT>(near_src + nb, nsl - 1, near_off, start + TILE + LOADS * tid);
  const int rbase = (part % LOADS) * ROW + part / LOADS;
  constexpr int RSTEP = NPART / LOADS;

  T sx = 0, sy = 0, sz = 0, sp = 0;
  T kx = 0, ky = 0, kz = 0, kp = 0;
  for (int base = start; base < total; base += TILE) {
    __syncthreads();
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      V4<T> q = next[l];
      if (!BUF && !ok[l]) q.w = T(0);
      tile[l * ROW + threadIdx.x] = q;
    }
    __syncthreads();
    // unconditional (past the end they yield invalid slots): a branch here
    // would make the compiler wait for the loads at its join
    if constexpr (BUF)
      fetch_positions_buf<WT, LOADS>(rsrc, n, leaf, total, base + TILE + LOADS * tid, lst,
                                     reinterpret_cast<V4<float>(&)[LOADS]>(next));
    else
      fetch_positions_leaf<T, WT, LOADS>(pos4, n, leaf, total, base + TILE + LOADS * tid, lst, next, ok);
    lst = fetch_list_leaf<WT>(near_src + nb, nsl - 1, near_off, base + 2 * TILE + LOADS * tid);
    // Slots past `total` hold zero-mass sources, so every partition runs the
    // same (wave-uniform, scalar-controlled) trip count.
    const int trips = (min(TILE, total - base) + NPART - 1) / NPART;
    T tx = 0, ty = 0, tz = 0, tp = 0;
#pragma unroll 8
    for (int k = 0; k < trips; ++k) {
      const V4<T> s = tile[rbase + k * RSTEP];
      const T dx = s.x - xi.x;
      const T dy = s.y - xi.y;
      const T dz = s.z - xi.z;
      const T r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
      const T rinv = fast_rsqrt(r2);
      const T mr = s.w * rinv;
      const T mr3 = mr * (rinv * rinv);
      tx = fma(mr3, dx, tx);
      ty = fma(mr3, dy, ty);
      tz = fma(mr3, dz, tz);
      if (POT) tp += mr;
    }
    kahan_add(sx, kx, tx);
    kahan_add(sy, ky, ty);
    kahan_add(sz, kz, tz);
    if (POT) kahan_add(sp, kp, tp);
  }
  // partitions reduced pairwise in LDS (fixed tree order, every thread takes part)
  __syncthreads();
  tile[threadIdx.x] = V4<T>{sx - kx, sy - ky, sz - kz, sp - kp};
  __syncthreads();
#pragma unroll
  for (int w = NPART / 2; w >= 1; w >>= 1) {
    if (part < w) {
      const V4<T> a = tile[threadIdx.x];
      const V4<T> b = tile[threadIdx.x + w * WT];
      tile[threadIdx.x] = V4<T>{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
    }
    __syncthreads();
  }
  if (part == 0 && i < cnt)
    put_sums<T, POT>(tile[i], xi.w, first, i, leaf_size, part_out, eps2, G, out_index, acc, pot, accumulate, items);
}

// Waves a SIMD that p2p_any_kernel is compiled for: the kP2PBlocksPerCu workgroups that
// LDS admits (some instances took 97 to 127 registers, a wave less: float64 leaf 1,
// uncompensated, 470 us against 355).  One float32 instance has 95 registers either way
// and a schedule that suits it better without the request (leaf 128: 2.70 against 3.08 ms).
constexpr int any_waves(int bytes, bool pot, bool comp, bool safe) {
  return bytes == 4 && !pot && !comp && !safe ? 1 : kP2PBlocksPerCu;
}

// Any leaf width (1..256), softening and summation.  Thread t owns target
// t % leaf_size and partition t / leaf_size of floor(256 / leaf_size) (at most 64,
// leaf 1: 32, so that most of the final sums stay in one wave): with the
// width rounded up to a power of two instead, leaves of 24 left a quarter of the
// lanes idle.  A tile's first slot is divided by the width once (the same for the
// workgroup) and the threads' slots by a multiplication with its reciprocal, exact
// for the at most kThreads + TILE slots of a tile (magic = ceil(2^32 / leaf_size)).
// Tiles hold tile_slots <= TILE slots, a multiple of 8 rounds of the partitions
// where they are few, so that full tiles have no remainder of the unrolled loop.
// In LDS a partition's slots follow each other (row_len, odd, apart from the next
// partition's): at a run-time distance every interaction paid an address, 131k Plummer
// bodies, float32, leaf 24 / 96 / 128 / 256 714 / 3021 / 2825 / 4134 us against
// 660 / 2758 / 2542 / 3780.
template <typename T, bool POT, bool COMP, bool SAFE>
__global__ __launch_bounds__(kThreads, any_waves(sizeof(T), POT, COMP, SAFE)) void p2p_any_kernel(
    const T* __restrict__ pos4, int32_t n, int32_t leaf_size, uint32_t magic, int32_t npart, uint32_t part_magic,
    int32_t tile_slots, const int32_t* __restrict__ near_off, const int32_t* __restrict__ near_src, T eps2, T G,
    const int32_t* __restrict__ out_index, T* __restrict__ acc, T* __restrict__ pot, int32_t accumulate,
    P2PItems<T> items) {
  constexpr int TILE = sizeof(T) == 4 ? 1024 : 512;
  constexpr int LOADS = TILE / kThreads;
  constexpr int kElems = TILE + kWave;  // at most kWave rows, padded by a slot each
  constexpr int kPadElems = static_cast<int>(kP2PLdsBytes / sizeof(V4<T>));
  __shared__ V4<T> tile[kElems > kPadElems ? kElems : kPadElems];
  const int tid = threadIdx.x;
  const int item = xcd_contiguous(blockIdx.x, gridDim.x);
  const int leaf = items.leaf ? items.leaf[item] : item;
  auto quotient = [&](uint32_t v) { return leaf_size == 1 ? v : __umulhi(v, magic); };
  int part = static_cast<int>(quotient(tid));
  const int i = tid - part * leaf_size;
  const bool idle = part >= npart;
  if (idle) part = 0;  // stays in step with the others, its sums are dropped
  const int first = leaf * leaf_size;
  const int cnt = min(leaf_size, n - first);
  const V4<T> xi = load4(pos4, first + (i < cnt ? i : 0));
  const int nb = near_off[leaf];
  const int nsl = 1 + (near_off[leaf + 1] - nb);
  const int start = items.leaf ? items.s0[item] : 0;
  const int total = items.leaf ? items.s1[item] : nsl * leaf_size;
  const int part_out = items.leaf ? items.part[item] : -1;
  const int32_t* list = nsl > 1 ? near_src + nb : near_off;  // an empty list reads a valid location, unused
  const int hi = max(nsl - 2, 0);

  V4<T> next[LOADS];
  bool ok[LOADS];
  // of the tile after `next`: near-list entries, slots within the source leaf
  // (complemented for the self leaf)
  int lst[LOADS], off[LOADS];
  auto fetch_list = [&](int base) {
    const int qb = base / leaf_size, ob = base - qb * leaf_size;
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      const uint32_t v = ob + tid + l * kThreads;
      const int dq = static_cast<int>(quotient(v));
      const int q = qb + dq, o = static_cast<int>(v) - dq * leaf_size;
      off[l] = q == 0 ? ~o : o;
      lst[l] = list[min(max(q - 1, 0), hi)];
    }
  };
  auto fetch_positions = [&](int base) {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      const bool self = off[l] < 0;
      const int g = (self ? leaf : lst[l]) * leaf_size + (self ? ~off[l] : off[l]);
      ok[l] = tid + l * kThreads < min(tile_slots, total - base) && g < n;
      next[l] = load4(pos4, ok[l] ? g : 0);
    }
  };
  fetch_list(start);
  fetch_positions(start);
  fetch_list(start + tile_slots);
  const int row_len = static_cast<int>(npart == 1 ? tile_slots : __umulhi(tile_slots, part_magic)) | 1;
  int at[LOADS];  // where this thread's slots of a tile lie (-1: past its slots)
#pragma unroll
  for (int l = 0; l < LOADS; ++l) {
    const int v = tid + l * kThreads;
    const int k = npart == 1 ? v : static_cast<int>(__umulhi(v, part_magic));
    at[l] = v < tile_slots ? (v - k * npart) * row_len + k : -1;
  }

  T sx = 0, sy = 0, sz = 0, sp = 0;
  T kx = 0, ky = 0, kz = 0, kp = 0;
  for (int base = start; base < total; base += tile_slots) {
    __syncthreads();
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      V4<T> q = next[l];
      if (!ok[l]) q.w = T(0);
      if (at[l] >= 0) tile[at[l]] = q;
    }
    __syncthreads();
    // unconditional, as in p2p_kernel: past the end they yield massless slots
    fetch_positions(base + tile_slots);
    fetch_list(base + 2 * tile_slots);
    const int trips = (min(tile_slots, total - base) + npart - 1) / npart;
    T tx = 0, ty = 0, tz = 0, tp = 0;
    const V4<T>* src = tile + part * row_len;
#pragma unroll 8
    for (int k = 0; k < trips; ++k) {
      const V4<T> s = src[k];
      const T dx = s.x - xi.x;
      const T dy = s.y - xi.y;
      const T dz = s.z - xi.z;
      const T r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
      T rinv = fast_rsqrt(r2);
      if (SAFE) rinv = r2 > T(0) ? rinv : T(0);  // the self pair, coincident points
      const T mr = s.w * rinv;
      const T mr3 = mr * (rinv * rinv);
      tx = fma(mr3, dx, tx);
      ty = fma(mr3, dy, ty);
      tz = fma(mr3, dz, tz);
      if (POT) tp += mr;
    }
    if (COMP) {
      kahan_add(sx, kx, tx);
      kahan_add(sy, ky, ty);
      kahan_add(sz, kz, tz);
      if (POT) kahan_add(sp, kp, tp);
    } else {
      sx += tx;
      sy += ty;
      sz += tz;
      if (POT) sp += tp;
    }
  }
  __syncthreads();
  tile[tid] = V4<T>{sx - kx, sy - ky, sz - kz, sp - kp};
  __syncthreads();
  int w = 1;
  while (2 * w < npart) w *= 2;  // pairwise over the partitions, fixed order
  auto fold = [&] {
    if (!idle && part < w && part + w < npart) {
      const V4<T> a = tile[tid];
      const V4<T> b = tile[tid + w * leaf_size];
      tile[tid] = V4<T>{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
    }
  };
  for (; w * leaf_size > kWave; w >>= 1) {
    fold();
    __syncthreads();
  }
  if (tid < kWave)  // the rest within the first wave, whose LDS operations stay in order
    for (; w >= 1; w >>= 1) {
      fold();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  if (!idle && part == 0 && i < cnt)
    put_sums<T, POT>(tile[i], xi.w, first, i, leaf_size, part_out, eps2, G, out_index, acc, pot, accumulate, items);
}

// Leaves split over several items: one workgroup per split leaf.  Target i
// of the leaf has nsub = 256 / leaf_size lanes; lane j adds the partials of
// items p0 + j, p0 + j + nsub, ... (compensated), and lane 0 then adds the
// nsub lane sums in lane order: a fixed summation order for every run.  The
// result gets what the single-item path applies (self potential, G, output row).
template <typename T, bool POT>
__global__ __launch_bounds__(kThreads) void p2p_reduce_kernel(const T* __restrict__ pos4, int32_t n, int32_t leaf_size,
                                                              const int32_t* __restrict__ split_leaf,
                                                              const int32_t* __restrict__ p0,
                                                              const int32_t* __restrict__ p1,
                                                              const T* __restrict__ partials, T eps2, T G,
                                                              const int32_t* __restrict__ out_index,
                                                              T* __restrict__ acc, T* __restrict__ pot,
                                                              int32_t accumulate) {
  __shared__ T red[4][kThreads];
  const int k = blockIdx.x;
  const int nsub = kThreads / leaf_size;
  const int i = threadIdx.x % leaf_size, j = threadIdx.x / leaf_size;
  T s[4] = {0, 0, 0, 0}, c[4] = {0, 0, 0, 0};
  if (j < nsub) {
    const int a = p0[k], b = p1[k];
    for (int p = a + j; p < b; p += nsub) {
      const T* src = partials + (static_cast<int64_t>(p) * leaf_size + i) * 4;
      for (int q = 0; q < 4; ++q) kahan_add(s[q], c[q], src[q]);
    }
  }
  for (int q = 0; q < 4; ++q) red[q][threadIdx.x] = s[q] - c[q];
  __syncthreads();
  const int first = split_leaf[k] * leaf_size;
  if (j != 0 || first + i >= n) return;
  T t[4] = {0, 0, 0, 0}, e[4] = {0, 0, 0, 0};
  for (int jj = 0; jj < nsub; ++jj)
    for (int q = 0; q < 4; ++q) kahan_add(t[q], e[q], red[q][jj * leaf_size + i]);
  for (int q = 0; q < 4; ++q) t[q] -= e[q];
  T ap = t[3];
  if (POT && eps2 > T(0)) ap -= pos4[4 * static_cast<int64_t>(first + i) + 3] * fast_rsqrt(eps2);
  const int64_t row = out_index ? out_index[first + i] : first + i;
  if (accumulate) {
    acc[3 * row + 0] += G * t[0];
    acc[3 * row + 1] += G * t[1];
    acc[3 * row + 2] += G * t[2];
    if (POT) pot[row] += -G * ap;
  } else {
    acc[3 * row + 0] = G * t[0];
    acc[3 * row + 1] = G * t[1];
    acc[3 * row + 2] = G * t[2];
    if (POT) pot[row] = -G * ap;
  }
}

// Leaves of 8 to 64, softened and compensated, run on the kernel
// with the width compiled in: at 1M bodies and leaf 16 its fetch takes 35
// instructions a tile against about 110.  float32 leaves of 8 run in narrow
// workgroups.  Row offsets of its float32 fetch bound n.
template <typename T, int WT>
void launch_p2p_wt(hipStream_t s, const T* pos4, int32_t n, int32_t num_blocks, const int32_t* near_off,
                   const int32_t* near_src, T eps2, T G, const int32_t* out_index, T* acc, T* pot, bool accumulate,
                   P2PItems<T> items) {
  constexpr int kFastThreads = (sizeof(T) == 4 && WT == 8) ? kNarrowThreads : kThreads;
  if (pot)
    p2p_kernel<T, WT, true, kFastThreads><<<num_blocks, kFastThreads, 0, s>>>(
        pos4, n, near_off, near_src, eps2, G, out_index, acc, pot, accumulate ? 1 : 0, items);
  else
    p2p_kernel<T, WT, false, kFastThreads><<<num_blocks, kFastThreads, 0, s>>>(
        pos4, n, near_off, near_src, eps2, G, out_index, acc, pot, accumulate ? 1 : 0, items);
}

template <typename T, bool POT>
void launch_p2p_any(hipStream_t s, const T* pos4, int32_t n, int32_t leaf_size, int32_t num_blocks,
                    const int32_t* near_off, const int32_t* near_src, T eps2, T G, const int32_t* out_index, T* acc,
                    T* pot, bool comp, bool accumulate, P2PItems<T> items) {
  const bool safe = !(eps2 > T(0));
  auto reciprocal = [](int d) { return static_cast<uint32_t>(((uint64_t(1) << 32) + d - 1) / d); };
  const uint32_t magic = reciprocal(leaf_size);
  constexpr int kTile = sizeof(T) == 4 ? 1024 : 512;
  const int npart = leaf_size == 1 ? 32 : std::min(kThreads / leaf_size, kWave);
  const int round = npart <= 32 ? 8 * npart : 4 * npart <= kTile ? 4 * npart : npart;
  const int tile_slots = kTile - kTile % round;
#define JFM_P2P_ANY(COMP, SAFE)                                                                                   \
  p2p_any_kernel<T, POT, COMP, SAFE><<<num_blocks, kThreads, 0, s>>>(                                             \
      pos4, n, leaf_size, magic, npart, reciprocal(npart), tile_slots, near_off, near_src, eps2, G, out_index, acc, \
      pot, accumulate ? 1 : 0, items)
  if (comp && safe)
    JFM_P2P_ANY(true, true);
  else if (comp)
    JFM_P2P_ANY(true, false);
  else if (safe)
    JFM_P2P_ANY(false, true);
  else
    JFM_P2P_ANY(false, false);
#undef JFM_P2P_ANY
}

template <typename T>
int32_t launch_p2p(hipStream_t s, const T* pos4, int32_t n, int32_t leaf_size, int32_t num_leaves,
                   const int32_t* near_off, const int32_t* near_src, T eps2, T G, const int32_t* out_index, T* acc,
                   T* pot, bool comp, bool accumulate, P2PItems<T> items = P2PItems<T>{}) {
  const bool fast = comp && eps2 > T(0) && (sizeof(T) == 8 || n <= kBufMaxRows);
#define JFM_P2P_WT(WT)                                                                                             \
  launch_p2p_wt<T, WT>(s, pos4, n, num_leaves, near_off, near_src, eps2, G, out_index, acc, pot, accumulate, items)
  if (fast && leaf_size == 8)
    JFM_P2P_WT(8);
  else if (fast && leaf_size == 16)
    JFM_P2P_WT(16);
  else if (fast && leaf_size == 32)
    JFM_P2P_WT(32);
  else if (fast && leaf_size == 64)
    JFM_P2P_WT(64);
  else if (pot)
    launch_p2p_any<T, true>(s, pos4, n, leaf_size, num_leaves, near_off, near_src, eps2, G, out_index, acc, pot, comp,
                            accumulate, items);
  else
    launch_p2p_any<T, false>(s, pos4, n, leaf_size, num_leaves, near_off, near_src, eps2, G, out_index, acc, pot,
                             comp, accumulate, items);
#undef JFM_P2P_WT
  return check_launch("jfm_p2p");
}

}  // namespace
}  // namespace jfm

using namespace jfm;

extern "C" {

int32_t jfm_l2p(void* stream, int32_t dtype, int32_t p, const void* pos4, int32_t n, int32_t leaf_size,
                int32_t num_internal, const void* locals, const void* centers4, double G, const int32_t* out_index,
                void* acc, void* pot, int32_t accumulate);

int32_t jfm_p2p(void* stream, int32_t dtype, const void* pos4, int32_t n, int32_t num_leaves, int32_t leaf_size,
                const int32_t* near_off, const int32_t* near_src, double eps2, double G, const int32_t* out_index,
                void* acc, void* pot, int32_t flags, int32_t accumulate) {
  if (n < 1 || leaf_size < 1 || leaf_size > 256 || num_leaves != (n + leaf_size - 1) / leaf_size)
    return fail(JFM_ERR_ARG, "jfm_p2p: inconsistent sizes (leaf_size must be 1..256)");
  if (!pos4 || !near_off || !near_src || !acc) return fail(JFM_ERR_ARG, "jfm_p2p: NULL buffer");
  if (!(eps2 >= 0.0)) return fail(JFM_ERR_ARG, "jfm_p2p: eps2 must be >= 0");
  hipStream_t s = as_stream(stream);
  const bool comp = (flags & JFM_EVAL_COMPENSATED) != 0;
  void* potp = (flags & JFM_EVAL_POTENTIAL) ? pot : nullptr;
  if ((flags & JFM_EVAL_POTENTIAL) && !pot) return fail(JFM_ERR_ARG, "jfm_p2p: potential requested, pot is NULL");
  if (dtype == JFM_F32)
    return launch_p2p<float>(s, (const float*)pos4, n, leaf_size, num_leaves, near_off, near_src,
                             static_cast<float>(eps2), static_cast<float>(G), out_index, (float*)acc, (float*)potp,
                             comp, accumulate != 0);
  if (dtype == JFM_F64)
    return launch_p2p<double>(s, (const double*)pos4, n, leaf_size, num_leaves, near_off, near_src, eps2, G,
                              out_index, (double*)acc, (double*)potp, comp, accumulate != 0);
  return fail(JFM_ERR_ARG, "jfm_p2p: bad dtype");
}

int32_t jfm_p2p_items(void* stream, int32_t dtype, const void* pos4, int32_t n, int32_t num_leaves, int32_t leaf_size,
                      int32_t num_items, const int32_t* item_leaf, const int32_t* item_s0, const int32_t* item_s1,
                      const int32_t* item_part, int32_t num_part, void* partials, const int32_t* near_off,
                      const int32_t* near_src, double eps2, double G, const int32_t* out_index, void* acc, void* pot,
                      int32_t flags, int32_t accumulate) {
  if (n < 1 || leaf_size < 1 || leaf_size > 256 || num_leaves != (n + leaf_size - 1) / leaf_size || num_items < 1 ||
      num_part < 0)
    return fail(JFM_ERR_ARG, "jfm_p2p_items: inconsistent sizes");
  if (!pos4 || !near_off || !near_src || !acc || !item_leaf || !item_s0 || !item_s1 || !item_part ||
      (num_part > 0 && !partials))
    return fail(JFM_ERR_ARG, "jfm_p2p_items: NULL buffer");
  if (!(eps2 >= 0.0)) return fail(JFM_ERR_ARG, "jfm_p2p_items: eps2 must be >= 0");
  if ((flags & JFM_EVAL_POTENTIAL) && !pot) return fail(JFM_ERR_ARG, "jfm_p2p_items: pot is NULL");
  hipStream_t s = as_stream(stream);
  const bool comp = (flags & JFM_EVAL_COMPENSATED) != 0;
  void* potp = (flags & JFM_EVAL_POTENTIAL) ? pot : nullptr;
  if (dtype == JFM_F32)
    return launch_p2p<float>(s, (const float*)pos4, n, leaf_size, num_items, near_off, near_src,
                             static_cast<float>(eps2), static_cast<float>(G), out_index, (float*)acc, (float*)potp,
                             comp, accumulate != 0,
                             P2PItems<float>{item_leaf, item_s0, item_s1, item_part, (float*)partials, num_part});
  if (dtype == JFM_F64)
    return launch_p2p<double>(s, (const double*)pos4, n, leaf_size, num_items, near_off, near_src, eps2, G,
                              out_index, (double*)acc, (double*)potp, comp, accumulate != 0,
                              P2PItems<double>{item_leaf, item_s0, item_s1, item_part, (double*)partials, num_part});
  return fail(JFM_ERR_ARG, "jfm_p2p_items: bad dtype");
}

int32_t jfm_p2p_reduce(void* stream, int32_t dtype, const void* pos4, int32_t n, int32_t leaf_size, int32_t num_split,
                       const int32_t* split_leaf, const int32_t* split_p0, const int32_t* split_p1,
                       const void* partials, double eps2, double G, const int32_t* out_index, void* acc, void* pot,
                       int32_t flags, int32_t accumulate) {
  if (n < 1 || leaf_size < 1 || leaf_size > 256 || num_split < 0) return fail(JFM_ERR_ARG, "jfm_p2p_reduce: sizes");
  if (num_split == 0) return JFM_OK;
  if (!pos4 || !split_leaf || !split_p0 || !split_p1 || !partials || !acc)
    return fail(JFM_ERR_ARG, "jfm_p2p_reduce: NULL buffer");
  const bool want_pot = (flags & JFM_EVAL_POTENTIAL) != 0;
  if (want_pot && !pot) return fail(JFM_ERR_ARG, "jfm_p2p_reduce: pot is NULL");
  hipStream_t s = as_stream(stream);
#define JFM_P2P_REDUCE(T, POT)                                                                                  \
  p2p_reduce_kernel<T, POT><<<num_split, kThreads, 0, s>>>((const T*)pos4, n, leaf_size, split_leaf, split_p0,   \
                                                           split_p1, (const T*)partials, static_cast<T>(eps2), \
                                                           static_cast<T>(G), out_index, (T*)acc, (T*)pot,     \
                                                           accumulate)
  if (dtype == JFM_F32) {
    if (want_pot) JFM_P2P_REDUCE(float, true); else JFM_P2P_REDUCE(float, false);
  } else if (dtype == JFM_F64) {
    if (want_pot) JFM_P2P_REDUCE(double, true); else JFM_P2P_REDUCE(double, false);
  } else {
    return fail(JFM_ERR_ARG, "jfm_p2p_reduce: bad dtype");
  }
#undef JFM_P2P_REDUCE
  return check_launch("jfm_p2p_reduce");
}

int32_t jfm_evaluate(void* stream, int32_t dtype, int32_t p, const void* pos4, int32_t n, int32_t num_leaves,
                     int32_t leaf_size, int32_t num_internal, const int32_t* near_off, const int32_t* near_src,
                     const void* locals, const void* centers4, double eps2, double G, const int32_t* out_index,
                     void* acc, void* pot, int32_t flags) {
  const bool near = (flags & JFM_EVAL_NEAR) != 0;
  const bool far = (flags & JFM_EVAL_FAR) != 0;
  if (!near && !far) return fail(JFM_ERR_ARG, "jfm_evaluate: neither JFM_EVAL_NEAR nor JFM_EVAL_FAR set");
  if (num_internal != num_leaves - 1) return fail(JFM_ERR_ARG, "jfm_evaluate: num_internal must be L-1");
  if ((flags & JFM_EVAL_POTENTIAL) && !pot) return fail(JFM_ERR_ARG, "jfm_evaluate: pot is NULL");
  void* potp = (flags & JFM_EVAL_POTENTIAL) ? pot : nullptr;
  // near field first, far field added onto its rows: the order of a step's launches
  // and of the work items', so that a*G + (-G)*g rounds alike on every path
  if (near) {
    int32_t rc = jfm_p2p(stream, dtype, pos4, n, num_leaves, leaf_size, near_off, near_src, eps2, G, out_index, acc,
                         potp, flags, 0);
    if (rc != JFM_OK) return rc;
  }
  if (far)
    return jfm_l2p(stream, dtype, p, pos4, n, leaf_size, num_internal, locals, centers4, G, out_index, acc, potp,
                   near ? 1 : 0);
  return JFM_OK;
}

}  // extern "C"
