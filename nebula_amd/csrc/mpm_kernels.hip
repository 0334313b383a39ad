// mpm_kernels.hip — the MPM substep as hand-written gfx950 kernels.
//
// One substep (the reference's 11 dispatches, src/engine/MPMEngine.cpp:415-473)
// runs here as:
//   bin   (count in the previous G2P, or k_bin_keys) -> k_bin_tiles (or
//         k_bin_mark -> k_bin_compact) -> k_bin_scatter -> k_bin_sort
//         (replaces zero_cells, mpm_hash_count, hash_scan_local/global,
//          hash_add_base, mpm_hash_sort; output is bit-identical to the stable
//          counting sort with END offsets of tests/helpers/MPMHarness.cpp:132-178,
//          with no group-count limit)
//   P2G   k_p2g: one block per occupied 8^3 tile; its occupied cells are
//         compacted onto threads, each thread walks its cell's particles (one
//         128-byte record each) and sums their 27 node contributions in
//         registers; the sums are merged into the tile's 10^3 LDS node box in 27
//         barrier-separated phases (every thread owns a distinct node in a
//         phase: no atomics, fixed order) and written as a per-tile partial;
//         small scenes: k_p2g_items walks the cells, k_p2g merges
//         (replaces mpm_zero_grid + mpm_p2g.comp's node-centric gather)
//   grid  k_grid_tiles: per occupied tile, its nodes and those around it that no
//         other takes (with noise forces k_grid_noise, in smaller units); sums
//         the <= 8 partials covering each node in a fixed order, then velocity,
//         cap, forces, walls, analytic colliders and the dense-SDF BC in registers
//         (replaces mpm_grid_update.comp + mpm_nanovdb_bc.comp)
//   G2P   k_g2p: one thread per particle in bin order; 27-node gather, F update,
//         register SVD, return map, Hencky stress, guards, advection; also
//         writes the particle's cell key for the next substep's bin
//         (replaces mpm_g2p.comp)
// Particle state lives in an interleaved record per particle (the eight float4
// of the reference's layout side by side: 128 bytes, one cache line), so the
// gathers of P2G and G2P read whole lines; k_soa_to_aos / k_aos_to_soa move it
// to and from the reference's eight arrays at the API boundary.
// Every kernel is deterministic: identical inputs give bit-identical outputs.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "nb_device_math.hpp"
#include "nb_engine.hpp"
#include "nb_kernel_util.hpp"

namespace nb {

const char* const kKernelNames[kNumProfiledKernels] = {
    "bin_keys", "bin_tiles", "bin_compact", "bin_scatter", "bin_sort", "p2g", "grid_update", "g2p", "g2p_grid", "g2p_fb"};

// ---------------------------------------------------------------------------
// P2G's work items: a cell of up to p2g_item particles is one item, a more
// crowded one is split into up to kMaxChunks
// ---------------------------------------------------------------------------
constexpr uint32_t kMaxChunks = 4;

__device__ __forceinline__ uint32_t p2g_chunks(uint32_t count, uint32_t item) {
  return count == 0u ? 0u : min((count + item - 1u) / item, kMaxChunks);
}
// item length groups, longest first: >= 12, 10-11, 8-9, 6-7, <= 5 particles
constexpr uint32_t kGroups = 5;
__device__ __forceinline__ uint32_t p2g_group(uint32_t count, uint32_t chunks) {
  if (chunks == 0u) return 0u;
  const uint32_t per = (count + chunks - 1u) / chunks;
  return per >= 12u ? 0u : (per >= 10u ? 1u : (per >= 8u ? 2u : (per >= 6u ? 3u : 4u)));
}

// ---------------------------------------------------------------------------
// BIN
// ---------------------------------------------------------------------------
// The stable counting sort of the particles by cell, in two levels:
//   count    particles per tile, and each particle's place in its tile, by one
//            atomic per distinct tile of a wave: in G2P for the next substep
//            (its waves hold neighbours, one or two tiles each), or in
//            k_bin_keys when the state came from elsewhere
//   tiles    k_bin_tiles, or k_bin_mark + k_bin_compact for large cubes: the
//            ordered lists of occupied tiles and node tiles, each tile's first
//            slot, P2G's tile order
//   scatter  k_bin_scatter: every particle into its tile's range, any order
//   sort     k_bin_sort: one block per occupied tile counts its cells in LDS
//            and puts the tile's particles in (cell, index) order
// No counter per cell in memory: nothing to clear, and the atomics go to a few
// counters per wave.  Against a count per cell (clear, keys, mark, compact,
// tile scan, tile offsets, scatter, stabilize: eight launches of 2.5-5 us of
// stream time each where the work itself is less) the bin of 4,096 particles
// went from 27 to 12.5 us of a substep; with the FP64 fallback's fix-up, which
// now runs beside it, from 56 to 34 for 262,144 and from 121 to 73 for 4.19 M
// (the count adds 2 and 12 us to G2P there).

// One particle counted into its tile; returns its place there.  One atomic per
// distinct tile among the active lanes.
__device__ __forceinline__ uint32_t count_in_tile(uint32_t key, uint32_t* __restrict__ tile_cnt) {
  const uint32_t tile = key >> kTileBits;
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t below = (1ull << lane) - 1ull;
  uint64_t pending = __ballot(true);
  int leader_of = 0;
  uint32_t place = 0, cnt = 0;
  while (pending) {
    const int leader = __ffsll((unsigned long long)pending) - 1;
    const bool mine = tile == uint32_t(__shfl(int(tile), leader));
    const uint64_t peers = __ballot(mine);
    if (mine) {
      leader_of = leader;
      place = uint32_t(__popcll(peers & below));
    }
    if (int(lane) == leader) cnt = uint32_t(__popcll(peers));
    pending &= ~peers;
  }
  uint32_t base = 0;
  if (place == 0u) base = atomicAdd(&tile_cnt[tile_slot(tile)], cnt);
  return uint32_t(__shfl(int(base), leader_of)) + place;
}

// Key of every particle (computed from its record, or read) and its count.
template <bool FROM_REC, bool BATCH>
__global__ __launch_bounds__(256) void k_bin_keys(SubParams p, const float4* __restrict__ rec,
                                                  uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                                  uint32_t* __restrict__ tile_cnt) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.n) return;
  uint32_t key;
  if (FROM_REC) {
    const float4 x = rec[size_t(i) * kRec + R_P];
    key = cell_key(particle_geo<BATCH>(p, i), x.x, x.y, x.z);
    keys[i] = key;
  } else {
    key = keys[i];
  }
  rank[i] = count_in_tile(key, tile_cnt);
}

__global__ __launch_bounds__(256) void k_zero(uint32_t* __restrict__ a, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0u;
}

// A particle and its cell within its tile: one word while the index fits
// beside the cell (up to 2^23 particles), else a pair.
constexpr uint32_t kPackedParticles = 1u << 23;
template <bool PACKED>
struct BucketEntry;
template <>
struct BucketEntry<true> {
  using T = uint32_t;
  static __device__ __forceinline__ T make(uint32_t i, uint32_t cell) { return (i << kTileBits) | cell; }
  static __device__ __forceinline__ uint32_t index(T e) { return e >> kTileBits; }
  static __device__ __forceinline__ uint32_t cell(T e) { return e & uint32_t(kTileCells - 1); }
};
template <>
struct BucketEntry<false> {
  using T = uint2;
  static __device__ __forceinline__ T make(uint32_t i, uint32_t cell) { return make_uint2(i, cell); }
  static __device__ __forceinline__ uint32_t index(T e) { return e.x; }
  static __device__ __forceinline__ uint32_t cell(T e) { return e.y; }
};
template <bool PACKED>
__device__ __forceinline__ void scatter_one(uint32_t n, uint32_t i, const uint32_t* __restrict__ keys,
                                            const uint32_t* __restrict__ rank, const int32_t* __restrict__ tile_act,
                                            const uint32_t* __restrict__ tile_start, uint2* __restrict__ bucket_) {
  using E = BucketEntry<PACKED>;
  typename E::T* bucket = reinterpret_cast<typename E::T*>(bucket_);
  if (i >= n) return;
  const uint32_t key = keys[i];
  const int32_t a = tile_act[key >> kTileBits];
  const uint32_t slot = tile_start[a] + rank[i];
  if (slot < n) bucket[slot] = E::make(i, key & uint32_t(kTileCells - 1));  // always true: the counts are the keys'
}

// The tile's particles in (cell, index) order, its cells' counts and END
// offsets (the reference's cellOffset).  The counts of different waves arrive
// in any order, so a particle's place in its cell is the number of smaller
// indices there, counted in LDS (a cell holds about 8; lanes of one cell read
// the same words).  A tile beyond the LDS stage places its particles in memory,
// and 4, 16 or 64 lanes sort a cell of up to 32, 128 or 512 in registers; larger cells
// are the block's, in LDS or in memory.  (1,048,576 particles of 16 / 32 / 64 a cell:
// 20 / 44 / 124 us; a wave's cells one after the other 77 / 101 / 614.)
constexpr uint32_t kSortThreads = 512;
constexpr uint32_t kSortStage = 6144;  // particles of a tile sorted in LDS

template <bool PACKED>
__global__ __launch_bounds__(kSortThreads) void k_bin_sort(uint32_t n, const uint2* __restrict__ bucket_,
                                                           uint32_t* __restrict__ cell_count,
                                                           uint32_t* __restrict__ cell_end,
                                                           const uint32_t* __restrict__ act_tiles,
                                                           const uint32_t* __restrict__ tile_start,
                                                           const uint32_t* __restrict__ tile_total,
                                                           uint32_t* __restrict__ sorted,
                                                           const uint32_t* __restrict__ counters,
                                                           uint32_t* __restrict__ fb_ctl, uint32_t p2g_item,
                                                           uint4* __restrict__ items, uint16_t* __restrict__ cell_item,
                                                           uint32_t* __restrict__ tile_items) {
  using E = BucketEntry<PACKED>;
  const typename E::T* bucket = reinterpret_cast<const typename E::T*>(bucket_);
  __shared__ uint32_t s_idx[kSortStage + 3];  // three words past the end, read but not counted
  __shared__ uint16_t s_cell[kSortStage];
  __shared__ uint32_t s_cur[kTileCells], s_start[kTileCells + 1];
  __shared__ uint32_t s_wave[kSortThreads / 64 + 1];
  __shared__ uint64_t s_wave64[kSortThreads / 64 + 1];
  __shared__ uint32_t s_nbig;
  static_assert(kSortThreads == uint32_t(kTileCells), "one thread per cell");
  // the FP64 fallback's queue, worked off beside the scatter, is empty again
  if (fb_ctl != nullptr && blockIdx.x == 0u && threadIdx.x < kFbSlots) fb_ctl[threadIdx.x * kFbCtlStride] = 0u;
  const uint32_t na = counters[CNT_ACTIVE];
  bool dense = false;
  for (uint32_t a = blockIdx.x; a < na; a += gridDim.x) {
    const uint32_t first = tile_start[a], tot = min(tile_total[a], n - min(first, n));
    s_cur[threadIdx.x] = 0u;
    // the first four entries of a thread (2048 of the tile) stay in registers
    typename E::T held[4];
#pragma unroll
    for (uint32_t r = 0; r < 4u; r++) {
      const uint32_t e = r * kSortThreads + threadIdx.x;
      if (e < tot) held[r] = bucket[first + e];
    }
    __syncthreads();
    auto each = [&](auto f) {
#pragma unroll
      for (uint32_t r = 0; r < 4u; r++)
        if (r * kSortThreads + threadIdx.x < tot) f(held[r]);
      for (uint32_t e = 4u * kSortThreads + threadIdx.x; e < tot; e += kSortThreads) f(bucket[first + e]);
    };
    each([&](typename E::T u) { (void)atomicAdd(&s_cur[E::cell(u)], 1u); });
    __syncthreads();
    const uint32_t cnt = s_cur[threadIdx.x];
    uint32_t all;
    const uint32_t ex = block_exclusive_scan<kSortThreads>(cnt, s_wave, all);
    s_cur[threadIdx.x] = ex;
    s_start[threadIdx.x] = ex;
    if (threadIdx.x == 0u) s_start[kTileCells] = all;
    const size_t key = (size_t(act_tiles[a]) << kTileBits) + threadIdx.x;
    cell_count[key] = cnt;
    cell_end[key] = first + ex + cnt;
    if (items != nullptr && na <= kItemTiles) {
      // the tile's P2G work items, in the order k_p2g makes them, at the places
      // of its first particles (an item holds at least one); the other places
      // stay empty
      const uint32_t chunks = p2g_chunks(cnt, p2g_item), group = p2g_group(cnt, chunks);
      uint64_t tot64;
      const uint64_t pre = block_exclusive_scan<kSortThreads>(uint64_t(chunks) << (12 * group), s_wave64, tot64);
      uint32_t at = 0, n_items = 0;
#pragma unroll
      for (int k = 0; k < int(kGroups); k++) {
        if (group == uint32_t(k)) at = n_items + (uint32_t(pre >> (12 * k)) & 4095u);
        n_items += uint32_t(tot64 >> (12 * k)) & 4095u;
      }
      const uint32_t per = chunks ? (cnt + chunks - 1u) / chunks : 0u;
      for (uint32_t q = 0; q < chunks; q++) {
        const uint32_t kbeg = min(q * per, cnt), kend = min(kbeg + per, cnt);
        items[first + at + q] = make_uint4(first + ex + kbeg, kend - kbeg, uint32_t(key), 0u);
      }
      cell_item[key] = uint16_t(at | (chunks << 11));
      const uint32_t layers = __syncthreads_or(chunks == 4u) ? 4u : (__syncthreads_or(chunks == 3u) ? 3u : (__syncthreads_or(chunks == 2u) ? 2u : 1u));
      if (threadIdx.x == 0u) tile_items[a] = n_items | (layers << 16);
      for (uint32_t e = n_items + threadIdx.x; e < tot; e += kSortThreads) items[first + e] = make_uint4(0u, 0u, 0u, 0u);
    }
    __syncthreads();
    if (tot > kSortStage) {
      dense = true;
      continue;
    }
    each([&](typename E::T u) {
      const uint32_t c = E::cell(u), at = atomicAdd(&s_cur[c], 1u);
      s_idx[at] = E::index(u);
      s_cell[at] = uint16_t(c);
    });
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < tot; e += kSortThreads) {
      const uint32_t v = s_idx[e], c = s_cell[e], b = s_start[c], m = s_start[c + 1u];
      uint32_t r = b;
      for (uint32_t j = b; j < m; j += 4u) {  // four reads in flight
        const uint32_t w0 = s_idx[j], w1 = s_idx[j + 1u], w2 = s_idx[j + 2u], w3 = s_idx[j + 3u];
        r += (w0 < v ? 1u : 0u) + (j + 1u < m && w1 < v ? 1u : 0u) + (j + 2u < m && w2 < v ? 1u : 0u) +
             (j + 3u < m && w3 < v ? 1u : 0u);
      }
      sorted[first + r] = v;
    }
    __syncthreads();
  }
  if (!dense) return;
  // (after the others: in one loop with them its registers cost every tile a sixth)
  for (uint32_t a = blockIdx.x; a < na; a += gridDim.x) {
    const uint32_t first = tile_start[a], tot = min(tile_total[a], n - min(first, n));
    if (tot <= kSortStage) continue;
    const size_t key = (size_t(act_tiles[a]) << kTileBits) + threadIdx.x;
    const uint32_t cnt = cell_count[key], ex = cell_end[key] - cnt - first;
    __syncthreads();
    s_cur[threadIdx.x] = ex;
    s_start[threadIdx.x] = ex;
    if (threadIdx.x == 0u) {
      s_start[kTileCells] = tot;
      s_nbig = 0u;
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < tot; e += 4u * kSortThreads) {  // four loads in flight
      typename E::T u[4];
#pragma unroll
      for (uint32_t r = 0; r < 4u; r++)
        if (e + r * kSortThreads < tot) u[r] = bucket[first + e + r * kSortThreads];
#pragma unroll
      for (uint32_t r = 0; r < 4u; r++)
        if (e + r * kSortThreads < tot) sorted[first + atomicAdd(&s_cur[E::cell(u[r])], 1u)] = E::index(u[r]);
    }
    __syncthreads();
    // the wave's cells by the lanes that sort one, smallest first
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t m4 = __ballot(cnt >= 2u && cnt <= 32u), m16 = __ballot(cnt > 32u && cnt <= 128u);
    const uint64_t m64 = __ballot(cnt > 128u && cnt <= 512u);
    const uint32_t e4 = uint32_t(__popcll(m4)), e16 = e4 + uint32_t(__popcll(m16)), e64 = e16 + uint32_t(__popcll(m64));
    uint16_t* order = s_cell + (threadIdx.x & ~63u);
    uint16_t* big = s_cell + kTileCells;
    if (cnt > 512u) {
      big[atomicAdd(&s_nbig, 1u)] = uint16_t(threadIdx.x);
    } else if (cnt >= 2u) {
      order[cnt <= 32u ? uint32_t(__popcll(m4 & below))
                       : (cnt <= 128u ? e4 + uint32_t(__popcll(m16 & below)) : e16 + uint32_t(__popcll(m64 & below)))] =
          uint16_t(threadIdx.x);
    }
    __syncthreads();
    auto sort_cells = [&](auto lanes, uint32_t i, uint32_t stop) {
      constexpr uint32_t G = decltype(lanes)::value;
      for (; i < stop; i += 64u / G) {
        const uint32_t at = i + lane / G;
        const uint32_t c = at < stop ? order[at] : 0u, b = s_start[c];
        group_sort_segment<G, 8>(sorted + first + b, at < stop ? s_start[c + 1u] - b : 0u);
      }
    };
    sort_cells(std::integral_constant<uint32_t, 4u>{}, 0u, e4);
    sort_cells(std::integral_constant<uint32_t, 16u>{}, e4, e16);
    sort_cells(std::integral_constant<uint32_t, 64u>{}, e16, e64);
    const uint32_t nbig = s_nbig;
    for (uint32_t q = 0; q < nbig; q++) {
      const uint32_t c = big[q], m = s_start[c + 1u] - s_start[c];
      uint32_t* seg = sorted + first + s_start[c];
      uint32_t P = 1u;
      while (P < m) P <<= 1;
      if (P > kSortStage) {
        block_bitonic(seg, m, P);
        continue;
      }
      for (uint32_t e = threadIdx.x; e < P; e += kSortThreads) s_idx[e] = e < m ? seg[e] : 0xFFFFFFFFu;
      __syncthreads();
      block_bitonic(s_idx, P, P);
      for (uint32_t e = threadIdx.x; e < m; e += kSortThreads) seg[e] = s_idx[e];
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// P2G
// ---------------------------------------------------------------------------
// P2G: one block per occupied tile.  The tile's occupied cells are compacted
// (in Morton order) onto the block's threads as work items: a cell of up to
// p.p2g_item particles (tuned, 12 by default) is one item, a more crowded cell is split into up to
// kMaxChunks items of consecutive particles (so one crowded cell does not hold
// its wave for the whole walk).  A thread walks its item's particles in bin
// order, reading the first 96 bytes of each record, and sums their
// contributions to the 27 nodes the cell reaches in registers.  The sums are
// merged into the tile's 10^3 LDS node box chunk layer by chunk layer, each in
// 27 barrier-separated phases: within a phase the writing threads hold
// distinct cells, so every one adds to a distinct node, plain read-add-write
// is exact and the order of the sums is fixed.
constexpr int kP2GThreads = 256;
constexpr uint32_t kIdxStage = 4096;  // particle indices staged in LDS per pass

// One particle's node contributions, in the factored chains described at the
// walk below.  MASK: wx and wyz are set to zero at each node whose weight
// (wx wy) wz the reference skips (fma(a, 0, s) leaves s as it was); every
// other node gets the same bits as without the mask.
#define NB_P2G_CHAINS(MASK)                                                                           \
  {                                                                                                   \
    const float mp = q.mp, mvx = q.mvx, mvy = q.mvy, mvz = q.mvz;                                     \
    const float c00 = q.c00, c01 = q.c01, c02 = q.c02, c10 = q.c10, c11 = q.c11, c12 = q.c12;         \
    const float c20 = q.c20, c21 = q.c21, c22 = q.c22;                                                \
    const float t00 = q.t00, t11 = q.t11, t22 = q.t22, t01 = q.t01, t02 = q.t02, t12 = q.t12;         \
    const Axis3 &sx = q.sx, &sy = q.sy, &sz = q.sz;                                                   \
    float mwx[3], Qx[3], Qy[3], Qz[3], Rx[3], Ry[3], Rz[3], Sx[3], Sy[3], Sz[3];                      \
    _Pragma("unroll") for (int i = 0; i < 3; i++) {                                                   \
      mwx[i] = mp * sx.w[i];                                                                          \
      const float wdx = sx.w[i] * sx.dx[i];                                                           \
      Qx[i] = fmaf(-sx.g[i], t00, wdx * c00);                                                         \
      Qy[i] = fmaf(-sx.g[i], t01, wdx * c01);                                                         \
      Qz[i] = fmaf(-sx.g[i], t02, wdx * c02);                                                         \
      Rx[i] = fmaf(sy.w[i], fmaf(c10, sy.dx[i], mvx), -(sy.g[i] * t01));                              \
      Ry[i] = fmaf(sy.w[i], fmaf(c11, sy.dx[i], mvy), -(sy.g[i] * t11));                              \
      Rz[i] = fmaf(sy.w[i], fmaf(c12, sy.dx[i], mvz), -(sy.g[i] * t12));                              \
      const float wdz = sz.w[i] * sz.dx[i];                                                           \
      Sx[i] = fmaf(-sz.g[i], t02, wdz * c20);                                                         \
      Sy[i] = fmaf(-sz.g[i], t12, wdz * c21);                                                         \
      Sz[i] = fmaf(-sz.g[i], t22, wdz * c22);                                                         \
    }                                                                                                 \
    _Pragma("unroll") for (int kz = 0; kz < 3; kz++) {                                                \
      _Pragma("unroll") for (int jy = 0; jy < 3; jy++) {                                              \
        const float wyz = sy.w[jy] * sz.w[kz];                                                        \
        const float Px = fmaf(sz.w[kz], Rx[jy], sy.w[jy] * Sx[kz]);                                   \
        const float Py = fmaf(sz.w[kz], Ry[jy], sy.w[jy] * Sy[kz]);                                   \
        const float Pz = fmaf(sz.w[kz], Rz[jy], sy.w[jy] * Sz[kz]);                                   \
        _Pragma("unroll") for (int ix = 0; ix < 3; ix++) {                                            \
          const int o = (kz * 3 + jy) * 3 + ix;                                                       \
          float wx = sx.w[ix], wn = wyz;                                                              \
          if (MASK) {                                                                                 \
            const bool live = (sx.w[ix] * sy.w[jy]) * sz.w[kz] >= 1e-12f;                             \
            wx = live ? wx : 0.f;                                                                     \
            wn = live ? wn : 0.f;                                                                     \
          }                                                                                           \
          am[o] = fmaf(mwx[ix], wn, am[o]);                                                           \
          ax[o] = fmaf(wn, Qx[ix], fmaf(wx, Px, ax[o]));                                              \
          ay[o] = fmaf(wn, Qy[ix], fmaf(wx, Py, ay[o]));                                              \
          az[o] = fmaf(wn, Qz[ix], fmaf(wx, Pz, az[o]));                                              \
        }                                                                                             \
      }                                                                                               \
    }                                                                                                 \
  }

// A tile's box from its items' sums: four blocks per tile, a node a thread.  Node
// b of the box is reached from the cells b - (0, 1, 2) along each axis; a table
// of the tile's cells with two empty layers on every side tells each one's
// items.  Their sums are loaded together, then added in k_p2g's order: 256 items
// at a time, chunk layer by chunk layer, offset by offset.
constexpr int kTabEdge = 12, kTabCells = kTabEdge * kTabEdge * kTabEdge;
constexpr int kMergeBlocks = 4;
static_assert(kBoxNodes % kMergeBlocks == 0 && kBoxNodes / kMergeBlocks <= kP2GThreads, "a node a thread");

__device__ __forceinline__ void p2g_merge_items(uint16_t* s_tab, uint32_t na, const P2GItems& q,
                                                const uint32_t* __restrict__ act_tiles,
                                                const uint32_t* __restrict__ tile_start, float4* __restrict__ partial) {
  const int at = ((int(morton_compact(threadIdx.x >> 1)) + 2) * kTabEdge + int(morton_compact(threadIdx.x)) + 2) * kTabEdge +
                 int(morton_compact(2u * threadIdx.x)) + 2;
  for (uint32_t w = blockIdx.x; w < kMergeBlocks * na; w += gridDim.x) {
    const uint32_t a = w / kMergeBlocks;
    const uint32_t pair = reinterpret_cast<const uint32_t*>(q.cell_item + (size_t(act_tiles[a]) << kTileBits))[threadIdx.x];
    const uint32_t ti = q.tile_items[a], start = tile_start[a];
    __syncthreads();
    for (int e = threadIdx.x; e < kTabCells / 2; e += kP2GThreads) reinterpret_cast<uint32_t*>(s_tab)[e] = 0u;
    __syncthreads();
    *reinterpret_cast<uint32_t*>(s_tab + at) = pair;  // cells 2t and 2t + 1, neighbours in x
    __syncthreads();
    const uint32_t batches = ((ti & 0xFFFFu) + kP2GThreads - 1u) / kP2GThreads, layers = ti >> 16;
    if (threadIdx.x >= kBoxNodes / kMergeBlocks) continue;
    const int e = int(w % kMergeBlocks) * (kBoxNodes / kMergeBlocks) + int(threadIdx.x);
    const uint16_t* tab = s_tab + ((e / (kBox * kBox) + 2) * kTabEdge + (e / kBox) % kBox + 2) * kTabEdge + e % kBox + 2;
    uint32_t t[27];
#pragma unroll
    for (int o = 0; o < 27; o++) t[o] = tab[-(((o / 9) * kTabEdge + (o / 3) % 3) * kTabEdge + o % 3)];
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[27];
    for (uint32_t b = 0; b < batches; b++)
      for (uint32_t l = 0; l < layers; l++) {
        // with one layer the sums stay loaded from batch to batch
        if (layers > 1u || b == 0u) {
#pragma unroll
          for (int o = 0; o < 27; o++)
            v[o] = l < (t[o] >> 11) ? q.item_sum[size_t(o) * q.item_cap + start + (t[o] & 2047u) + l]
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int o = 0; o < 27; o++) {
          const bool turn = l < (t[o] >> 11) && ((t[o] & 2047u) + l) / kP2GThreads == b;
          s.x += turn ? v[o].x : 0.f; s.y += turn ? v[o].y : 0.f;
          s.z += turn ? v[o].z : 0.f; s.w += turn ? v[o].w : 0.f;
        }
      }
    partial[size_t(a) * kBoxNodes + e] = s;
  }
}

template <bool BATCH, bool ITEMS>
__global__ __launch_bounds__(kP2GThreads, 2) void k_p2g(SubParams p, const float4* __restrict__ rec,
                                                     const nb_material* __restrict__ mats,
                                                     const uint32_t* __restrict__ cell_count,
                                                     const uint32_t* __restrict__ cell_end,
                                                     const uint32_t* __restrict__ sorted,
                                                     const uint32_t* __restrict__ act_tiles,
                                                     const uint32_t* __restrict__ tile_order,
                                                     const uint32_t* __restrict__ tile_start,
                                                     const uint32_t* __restrict__ tile_total,
                                                     const uint32_t* __restrict__ counters,
                                                     P2GItems items, float4* __restrict__ partial) {
  __shared__ float s_m[kBoxNodes], s_x[kBoxNodes], s_y[kBoxNodes], s_z[kBoxNodes];
  __shared__ uint16_t s_item[kTileCells * kMaxChunks];  // cell | chunk << 9
  __shared__ uint32_t s_layers;
  __shared__ uint32_t s_cnt[kTileCells], s_end[kTileCells];
  __shared__ uint32_t s_idx[kIdxStage];
  __shared__ uint64_t s_scan64[kP2GThreads / 64 + 1];
  __shared__ float s_rho0[BATCH ? kBatchMaxMaterials : NB_MAX_MATERIALS];
  const uint32_t na = counters[CNT_ACTIVE];
  if (ITEMS && na <= kItemTiles) {
    static_assert(sizeof(s_idx) >= kTabCells * sizeof(uint16_t), "the table's place");
    p2g_merge_items(reinterpret_cast<uint16_t*>(s_idx), na, items, act_tiles, tile_start, partial);
    return;
  }
  for (uint32_t i = threadIdx.x; i < p.material_count; i += kP2GThreads) s_rho0[i] = mats[i].rho0;
  const bool apic = p.flip_ratio < -0.5f;
  const uint32_t mlast = p.material_count - 1u;

  for (uint32_t a0 = blockIdx.x; a0 < na; a0 += gridDim.x) {
    // the tile of place a0 in the largest-first order (its own index if the
    // order were ever out of range)
    const uint32_t ao = tile_order[a0], a = ao < na ? ao : a0;
    const uint32_t T = act_tiles[a];
    const SceneGeo g = tile_geo<BATCH>(p, T);
    const float D_inv = 4.f / (g.h * g.h);
    const float inv_h = g.inv_h;
    int tx, ty, tz;
    tile_coords(g, T, tx, ty, tz);
    const size_t tbase = size_t(T) << kTileBits;
    for (int e = threadIdx.x; e < kBoxNodes; e += kP2GThreads) {
      s_m[e] = 0.f; s_x[e] = 0.f; s_y[e] = 0.f; s_z[e] = 0.f;
    }
    // Work items of the occupied cells (thread t looks at cells 2t, 2t+1),
    // grouped by particle count (largest first, cell order within a group) so
    // that the lanes of a wave walk similar lengths: a stable counting sort
    // over kGroups groups, whose per-group counts (< 4096) are packed 12 bits
    // each into one 64-bit block scan.
    if (threadIdx.x == 0) s_layers = 0u;
    const uint32_t ca = 2u * threadIdx.x, cb = ca + 1u;
    const uint32_t na_ = cell_count[tbase + ca], nb_ = cell_count[tbase + cb];
    const uint32_t ea = cell_end[tbase + ca], eb = cell_end[tbase + cb];
    // the tile's particles are one contiguous range of the bin order: their
    // indices are staged in LDS with coalesced loads (a tile beyond the stage
    // reads the bin order directly), loaded here so that they are in flight
    // during the scan below and stored to LDS after it
    const uint32_t lo = tile_start[a], tile_n = tile_total[a];
    const bool staged = tile_n <= kIdxStage;
    uint32_t stg[kIdxStage / kP2GThreads];
#pragma unroll
    for (uint32_t r = 0; r < kIdxStage / kP2GThreads; r++) {
      const uint32_t e = threadIdx.x + r * kP2GThreads;
      stg[r] = (staged && e < tile_n) ? sorted[lo + e] : 0u;
    }
    s_cnt[ca] = na_;
    s_cnt[cb] = nb_;
    s_end[ca] = ea;
    s_end[cb] = eb;
    const uint32_t qa = p2g_chunks(na_, p.p2g_item), qb = p2g_chunks(nb_, p.p2g_item);
    const uint32_t ga = p2g_group(na_, qa), gb = p2g_group(nb_, qb);
    const uint64_t mine = (uint64_t(qa) << (12 * ga)) + (uint64_t(qb) << (12 * gb));
    uint64_t tot64;
    const uint64_t pre = block_exclusive_scan<kP2GThreads>(mine, s_scan64, tot64);
    if (max(qa, qb) > 1u) atomicMax(&s_layers, max(qa, qb) - 1u);
    uint32_t gbase[kGroups];
    {
      uint32_t acc = 0;
#pragma unroll
      for (int g = 0; g < int(kGroups); g++) {
        gbase[g] = acc;
        acc += uint32_t(tot64 >> (12 * g)) & 4095u;
      }
    }
    uint32_t pa = 0, pb = 0;
#pragma unroll
    for (int g = 0; g < int(kGroups); g++) {
      if (ga == uint32_t(g)) pa = gbase[g] + (uint32_t(pre >> (12 * g)) & 4095u);
      if (gb == uint32_t(g)) pb = gbase[g] + (uint32_t(pre >> (12 * g)) & 4095u) + (ga == gb ? qa : 0u);
    }
    for (uint32_t q = 0; q < qa; q++) s_item[pa + q] = uint16_t(ca | (q << 9));
    for (uint32_t q = 0; q < qb; q++) s_item[pb + q] = uint16_t(cb | (q << 9));
#pragma unroll
    for (uint32_t r = 0; r < kIdxStage / kP2GThreads; r++) {
      const uint32_t e = threadIdx.x + r * kP2GThreads;
      if (staged && e < tile_n) s_idx[e] = stg[r];
    }
    __syncthreads();
    uint32_t n_items = 0;
#pragma unroll
    for (int g = 0; g < int(kGroups); g++) n_items += uint32_t(tot64 >> (12 * g)) & 4095u;
    const uint32_t n_layers = s_layers + 1u;
    auto idx_of = [&](uint32_t k) -> uint32_t { return staged ? s_idx[k - lo] : sorted[k]; };

    for (uint32_t base = 0; base < n_items; base += kP2GThreads) {
      const uint32_t j = base + threadIdx.x;
      const bool have = j < n_items;
      const uint32_t it = have ? uint32_t(s_item[j]) : 0u;
      const uint32_t c = it & 511u, chunk = it >> 9;
      const int lx = int(morton_compact(c)), ly = int(morton_compact(c >> 1)), lz = int(morton_compact(c >> 2));
      const int cx = tx * 8 + lx, cy = ty * 8 + ly, cz = tz * 8 + lz;
      uint32_t kbeg = 0, kend = 0;
      if (have) {
        const uint32_t cnt = s_cnt[c], end = s_end[c];
        const uint32_t per = (cnt + p2g_chunks(cnt, p.p2g_item) - 1u) / p2g_chunks(cnt, p.p2g_item);
        kbeg = end - cnt + chunk * per;
        kend = min(kbeg + per, end);
      }
      float am[27], ax[27], ay[27], az[27];
#pragma unroll
      for (int o = 0; o < 27; o++) { am[o] = 0.f; ax[o] = 0.f; ay[o] = 0.f; az[o] = 0.f; }

      // Per particle (shaders/mpm_p2g.comp:40-90): mass m = rho0 Vp, affine
      // C = m (4/h^2) B (APIC only), dt Vp tau from the w lanes
      // (shaders/mpm_common.glsl:104-113), and the stencil of its cell.
      struct Src {
        Axis3 sx, sy, sz;
        float mp, mvx, mvy, mvz;
        float c00, c01, c02, c10, c11, c12, c20, c21, c22;
        float t00, t11, t22, t01, t02, t12;
      };
      // (the stencil's quotient (x - wmin)/h is taken as a product with 1/h:
      // the cell is the bin's, only the weights use it)
      // (a particle of the cell takes the fixed-piece form; one the bin
      // placed there from outside the grid, the general one).  Returns
      // whether the particle may have a node the reference skips, w =
      // (wx wy) wz < 1e-12 (shaders/mpm_p2g.comp:60-61): the smallest positive
      // per-axis weights bound every w from below (1.0001e-12 covers the
      // rounding of the product order).  In the fixed-piece form the middle
      // weight is >= 0.5 and the first one > 0, so an axis's smallest
      // positive weight is the smaller outer one (the last counting when > 0).
      auto stencil = [&](const float4& pp, Src& q) -> bool {
        const float fx = (pp.x - g.wmin[0]) * inv_h, fy = (pp.y - g.wmin[1]) * inv_h;
        const float fz = (pp.z - g.wmin[2]) * inv_h;
        bool ok = axis_stencil_cell(fx, pp.x, g.wmin[0], g.h, inv_h, cx, q.sx);
        ok &= axis_stencil_cell(fy, pp.y, g.wmin[1], g.h, inv_h, cy, q.sy);
        ok &= axis_stencil_cell(fz, pp.z, g.wmin[2], g.h, inv_h, cz, q.sz);
        if (ok) {
          auto mpos = [](const Axis3& a) { return a.w[2] > 0.f ? fminf(a.w[0], a.w[2]) : a.w[0]; };
          return (mpos(q.sx) * mpos(q.sy)) * mpos(q.sz) < 1.0001e-12f;
        }
        axis_stencil_f(fx, pp.x, g.wmin[0], g.h, inv_h, cx - 1, q.sx);
        axis_stencil_f(fy, pp.y, g.wmin[1], g.h, inv_h, cy - 1, q.sy);
        axis_stencil_f(fz, pp.z, g.wmin[2], g.h, inv_h, cz - 1, q.sz);
        return (min_positive3(q.sx.w) * min_positive3(q.sy.w)) * min_positive3(q.sz.w) < 1.0001e-12f;
      };
      // keep = 0 scales the particle's contribution to exactly zero
      auto setup = [&](const float4& pp, const float4& vv, const float4& b0, const float4& b1, const float4& b2,
                       const float4& tt, float keep, Src& q) {
        uint32_t mid = __float_as_uint(vv.w);
        mid = mid > mlast ? mlast : mid;
        q.mp = s_rho0[mid] * pp.w * keep;
        const float sc = apic ? q.mp * D_inv : 0.f;
        q.c00 = sc * b0.x; q.c01 = sc * b0.y; q.c02 = sc * b0.z;
        q.c10 = sc * b1.x; q.c11 = sc * b1.y; q.c12 = sc * b1.z;
        q.c20 = sc * b2.x; q.c21 = sc * b2.y; q.c22 = sc * b2.z;
        const float st = p.dt * pp.w * keep;
        q.t00 = st * tt.x; q.t11 = st * tt.y; q.t22 = st * tt.z;
        q.t01 = st * b0.w; q.t02 = st * b1.w; q.t12 = st * b2.w;
        q.mvx = q.mp * vv.x; q.mvy = q.mp * vv.y; q.mvz = q.mp * vv.z;
      };

      // Fast loop.  Node contributions factor as
      //   m w = (m wx) wyz,  mom = wx P(y,z) + wyz Q(x)
      // with P = wyz (m v + C (0, dy, dz)) - tau (0, gy wz, wy gz) and
      // Q = wx dx C e_x - gx tau e_x: 7 FMAs per node (explicit FMA chains;
      // strict evaluation of acc + (a b + c d) costs a multiply, an FMA and an
      // add).  P itself splits into per-axis terms, P = wz R(y) + wy S(z) with
      // R = wy (m v + dy C e_y) - gy tau e_y and S = wz dz C e_z - gz tau e_z,
      // so each of the 9 (y, z) pairs costs a multiply and an FMA per
      // component.  A particle with a sub-cutoff node is scaled to zero here and
      // added by the exact loop below, which visits only those particles:
      // the first two by their offsets from kbeg (16 bits each in tiny_at,
      // 0xFFFF = none), all of the item's particles when there are more (or
      // an offset does not fit).  The next particle's record is loaded while
      // this one is scattered; the walk's last iteration loads the first such
      // particle's record instead (pref), so the exact loop rarely waits.
      uint32_t tiny_at = 0xFFFFFFFFu;
      bool tiny_all = false, pref = false;
      float4 npp, nvv, nb0, nb1, nb2, ntt;
      auto load_rec = [&](uint32_t q) {
        const float4* r = rec + size_t(q) * kRec;
        npp = r[R_P]; nvv = r[R_V];
        nb0 = r[R_B0]; nb1 = r[R_B1]; nb2 = r[R_B2];
        ntt = r[R_T];
      };
      if (kbeg < kend) load_rec(idx_of(kbeg));
      for (uint32_t k = kbeg; k < kend; k++) {
        const float4 pp = npp, vv = nvv, b0 = nb0, b1 = nb1, b2 = nb2, tt = ntt;
        if (k + 1 < kend) {
          load_rec(idx_of(k + 1));
        } else if ((tiny_at & 0xFFFFu) != 0xFFFFu) {
          load_rec(idx_of(kbeg + (tiny_at & 0xFFFFu)));
          pref = true;
        }
        Src q;
        const bool tiny = stencil(pp, q);
        if (tiny) {
          const uint32_t off = k - kbeg;
          if (off >= 0xFFFFu || (tiny_at >> 16) != 0xFFFFu) {
            tiny_all = true;
          } else if ((tiny_at & 0xFFFFu) == 0xFFFFu) {
            tiny_at = 0xFFFF0000u | off;
          } else {
            tiny_at = (tiny_at & 0xFFFFu) | (off << 16);
          }
        }
        setup(pp, vv, b0, b1, b2, tt, tiny ? 0.f : 1.f, q);
        NB_P2G_CHAINS(false)
      }
      // Exact loop: the particles skipped above, the same chains with the
      // cutoff's node mask, in bin order (the order of the adds is the one a
      // walk over the whole item would give).
      const uint32_t n_exact = tiny_all ? kend - kbeg
                                        : ((tiny_at & 0xFFFFu) != 0xFFFFu ? 1u : 0u) + ((tiny_at >> 16) != 0xFFFFu ? 1u : 0u);
      if (__any(n_exact != 0u)) {
        for (uint32_t s = 0; s < n_exact; s++) {
          const uint32_t k = kbeg + (tiny_all ? s : (s == 0u ? (tiny_at & 0xFFFFu) : (tiny_at >> 16)));
          if (!(pref && !tiny_all && s == 0u)) load_rec(idx_of(k));
          Src q;
          const float4 pp = npp;
          if (!stencil(pp, q)) continue;
          setup(pp, nvv, nb0, nb1, nb2, ntt, 1.f, q);
          NB_P2G_CHAINS(true)
        }
      }
      for (uint32_t layer = 0; layer < n_layers; layer++) {
        const bool mine = have && chunk == layer;
#pragma unroll
        for (int kz = 0; kz < 3; kz++)
#pragma unroll
          for (int jy = 0; jy < 3; jy++)
#pragma unroll
            for (int ix = 0; ix < 3; ix++) {
              const int o = (kz * 3 + jy) * 3 + ix;
              const int e = ((lz + kz) * kBox + (ly + jy)) * kBox + (lx + ix);
              __syncthreads();
              if (mine) {
                s_m[e] += am[o];
                s_x[e] += ax[o];
                s_y[e] += ay[o];
                s_z[e] += az[o];
              }
            }
      }
      __syncthreads();
    }
    float4* out = partial + size_t(a) * kBoxNodes;
    for (int e = threadIdx.x; e < kBoxNodes; e += kP2GThreads) out[e] = make_float4(s_x[e], s_y[e], s_z[e], s_m[e]);
    __syncthreads();
  }
}

#undef NB_P2G_CHAINS

// P2G of small scenes: the walk over work items apart from their merge.  A block
// per tile leaves most CUs idle (4,096 particles are 8 tiles, 85,184 are 64) and
// walks a tile's items on one CU.  Here the bin lists the items of all tiles;
// k_p2g_items takes 64 of them a wave, anywhere on the chip, and leaves the sums
// of their 27 nodes in memory, item by item (432 bytes each); k_p2g then collects
// a tile's box from them (p2g_merge_items) in the order in which it merges the
// items of a tile that it walks itself, so a box has the same bits.  SPLIT waves
// share an item's four sums (momentum x, y, z and mass): the walk is bound by its
// chain of up to p2g_item particles, some 490 instructions each for all four
// sums, 320 for two, 230 for one.  Walk and merge against the box form: 11 + 6 us
// for 23 at 4,096 particles (SPLIT 4), 16 + 8 for 41 at 85,184 (SPLIT 2),
// 19 + 9 for 40 at 262,144.  The merge inside the grid update, without a box
// between, spills its 27 places (84 us at 262,144 particles).
template <int CHM, bool BATCH>
__device__ __forceinline__ void p2g_item_sums(const SubParams& p, const float4* __restrict__ rec, const uint4 it,
                                              const uint32_t* __restrict__ sorted, const float* s_rho0,
                                              float* __restrict__ out, size_t stride) {
  constexpr bool CX = CHM & 1, CY = CHM & 2, CZ = CHM & 4, CM = CHM & 8;
  const bool apic = p.flip_ratio < -0.5f;
  const uint32_t mlast = p.material_count - 1u;
  const SceneGeo g = tile_geo<BATCH>(p, it.z >> kTileBits);
  const float D_inv = 4.f / (g.h * g.h);
  const float inv_h = g.inv_h;
  const uint32_t cell = it.z - g.key_base;
  const int cx = int(morton_compact(cell)), cy = int(morton_compact(cell >> 1)), cz = int(morton_compact(cell >> 2));
  float am[27], ax[27], ay[27], az[27];
#pragma unroll
  for (int o = 0; o < 27; o++) { am[o] = 0.f; ax[o] = 0.f; ay[o] = 0.f; az[o] = 0.f; }
  // stencil, set-up and chains: those of k_p2g
  struct Stencil {
    Axis3 x, y, z;
  };
  auto stencil = [&](const float4& pp, Stencil& q) -> bool {
    const float fx = (pp.x - g.wmin[0]) * inv_h, fy = (pp.y - g.wmin[1]) * inv_h;
    const float fz = (pp.z - g.wmin[2]) * inv_h;
    bool ok = axis_stencil_cell(fx, pp.x, g.wmin[0], g.h, inv_h, cx, q.x);
    ok &= axis_stencil_cell(fy, pp.y, g.wmin[1], g.h, inv_h, cy, q.y);
    ok &= axis_stencil_cell(fz, pp.z, g.wmin[2], g.h, inv_h, cz, q.z);
    if (ok) {
      auto mpos = [](const Axis3& a) { return a.w[2] > 0.f ? fminf(a.w[0], a.w[2]) : a.w[0]; };
      return (mpos(q.x) * mpos(q.y)) * mpos(q.z) < 1.0001e-12f;
    }
    axis_stencil_f(fx, pp.x, g.wmin[0], g.h, inv_h, cx - 1, q.x);
    axis_stencil_f(fy, pp.y, g.wmin[1], g.h, inv_h, cy - 1, q.y);
    axis_stencil_f(fz, pp.z, g.wmin[2], g.h, inv_h, cz - 1, q.z);
    return (min_positive3(q.x.w) * min_positive3(q.y.w)) * min_positive3(q.z.w) < 1.0001e-12f;
  };
  struct Rec {
    float4 P, V, B0, B1, B2, T;
  };
  auto load = [&](Rec& r, uint32_t i) {
    const float4* q = rec + size_t(i) * kRec;
    r.P = q[R_P]; r.V = q[R_V];
    r.B0 = q[R_B0]; r.B1 = q[R_B1]; r.B2 = q[R_B2];
    r.T = q[R_T];
  };
  auto add = [&](const Rec& r, const Stencil& q, float keep, auto masked) {
    constexpr bool MASK = decltype(masked)::value;
    const uint32_t mid = __float_as_uint(r.V.w);
    const float m = s_rho0[mid > mlast ? mlast : mid] * r.P.w * keep;
    const float sc = apic ? m * D_inv : 0.f, st = p.dt * r.P.w * keep;
    float mwx[3], Q[3][3], R[3][3], S[3][3];  // [sum][offset]
    auto one = [&](int c, float b0, float b1, float b2, float t0_, float t1_, float t2_, float v) {
      const float c0 = sc * b0, c1 = sc * b1, c2 = sc * b2, t0 = st * t0_, t1 = st * t1_, t2 = st * t2_, mv = m * v;
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const float wdx = q.x.w[i] * q.x.dx[i], wdz = q.z.w[i] * q.z.dx[i];
        Q[c][i] = fmaf(-q.x.g[i], t0, wdx * c0);
        R[c][i] = fmaf(q.y.w[i], fmaf(c1, q.y.dx[i], mv), -(q.y.g[i] * t1));
        S[c][i] = fmaf(-q.z.g[i], t2, wdz * c2);
      }
    };
    if (CX) one(0, r.B0.x, r.B1.x, r.B2.x, r.T.x, r.B0.w, r.B1.w, r.V.x);
    if (CY) one(1, r.B0.y, r.B1.y, r.B2.y, r.B0.w, r.T.y, r.B2.w, r.V.y);
    if (CZ) one(2, r.B0.z, r.B1.z, r.B2.z, r.B1.w, r.B2.w, r.T.z, r.V.z);
#pragma unroll
    for (int i = 0; i < 3; i++) mwx[i] = m * q.x.w[i];
#pragma unroll
    for (int kz = 0; kz < 3; kz++)
#pragma unroll
      for (int jy = 0; jy < 3; jy++) {
        const float wyz = q.y.w[jy] * q.z.w[kz];
        float P[3];
#pragma unroll
        for (int c = 0; c < 3; c++)
          if ((CHM >> c) & 1) P[c] = fmaf(q.z.w[kz], R[c][jy], q.y.w[jy] * S[c][kz]);
#pragma unroll
        for (int ix = 0; ix < 3; ix++) {
          const int o = (kz * 3 + jy) * 3 + ix;
          float wx = q.x.w[ix], wn = wyz;
          if (MASK) {
            const bool live = (q.x.w[ix] * q.y.w[jy]) * q.z.w[kz] >= 1e-12f;
            wx = live ? wx : 0.f;
            wn = live ? wn : 0.f;
          }
          if (CM) am[o] = fmaf(mwx[ix], wn, am[o]);
          if (CX) ax[o] = fmaf(wn, Q[0][ix], fmaf(wx, P[0], ax[o]));
          if (CY) ay[o] = fmaf(wn, Q[1][ix], fmaf(wx, P[1], ay[o]));
          if (CZ) az[o] = fmaf(wn, Q[2][ix], fmaf(wx, P[2], az[o]));
        }
      }
  };
  // the walk of k_p2g: sub-cutoff particles scaled to zero here and added
  // after it by the masked chains; the next record is loaded while this one is
  // scattered, its index one step before
  const uint32_t kbeg = it.x, kend = it.x + it.y;
  uint32_t tiny_at = 0xFFFFFFFFu;
  bool tiny_all = false;
  Rec next;
  uint32_t i1 = 0;
  if (kbeg < kend) load(next, sorted[kbeg]);
  if (kbeg + 1u < kend) i1 = sorted[kbeg + 1u];
  for (uint32_t k = kbeg; k < kend; k++) {
    const Rec r = next;
    if (k + 1u < kend) load(next, i1);
    if (k + 2u < kend) i1 = sorted[k + 2u];
    Stencil q;
    const bool tiny = stencil(r.P, q);
    if (tiny) {
      const uint32_t off = k - kbeg;
      if (off >= 0xFFFFu || (tiny_at >> 16) != 0xFFFFu) tiny_all = true;
      else if ((tiny_at & 0xFFFFu) == 0xFFFFu) tiny_at = 0xFFFF0000u | off;
      else tiny_at = (tiny_at & 0xFFFFu) | (off << 16);
    }
    add(r, q, tiny ? 0.f : 1.f, std::false_type{});
  }
  const uint32_t n_exact = tiny_all ? kend - kbeg
                                    : ((tiny_at & 0xFFFFu) != 0xFFFFu ? 1u : 0u) + ((tiny_at >> 16) != 0xFFFFu ? 1u : 0u);
  for (uint32_t x = 0; x < n_exact; x++) {
    load(next, sorted[kbeg + (tiny_all ? x : (x == 0u ? (tiny_at & 0xFFFFu) : (tiny_at >> 16)))]);
    Stencil q;
    if (stencil(next.P, q)) add(next, q, 1.f, std::true_type{});
  }
#pragma unroll
  for (int o = 0; o < 27; o++) {
    float* w = out + size_t(o) * stride;
    if (CHM == 15) {
      *reinterpret_cast<float4*>(w) = make_float4(ax[o], ay[o], az[o], am[o]);
    } else {
      if (CX) w[0] = ax[o];
      if (CY) w[1] = ay[o];
      if (CZ) w[2] = az[o];
      if (CM) w[3] = am[o];
    }
  }
}

// grid: SPLIT times the chunks of 64 places, the chunks padded to a multiple of
// the XCDs so that an item's waves share an L2
template <int SPLIT, bool BATCH>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_p2g_items(
    SubParams p, const float4* __restrict__ rec, const nb_material* __restrict__ mats,
    const uint32_t* __restrict__ sorted, const uint4* __restrict__ items, float4* __restrict__ item_sum,
    uint32_t item_cap, const uint32_t* __restrict__ counters) {
  if (counters[CNT_ACTIVE] > kItemTiles) return;
  __shared__ float s_rho0[BATCH ? kBatchMaxMaterials : NB_MAX_MATERIALS];
  const uint32_t chunks = gridDim.x / uint32_t(SPLIT);
  const uint32_t slot = xcd_chunk(blockIdx.x % chunks, chunks) * 64u + threadIdx.x;
  const uint4 it = slot < p.n ? items[slot] : make_uint4(0u, 0u, 0u, 0u);
  for (uint32_t i = threadIdx.x; i < p.material_count; i += 64u) s_rho0[i] = mats[i].rho0;
  __syncthreads();
  if (it.y == 0u) return;
  float* out = reinterpret_cast<float*>(item_sum + slot);
  const size_t stride = size_t(item_cap) * 4u;
  const uint32_t part = blockIdx.x / chunks;
  if (SPLIT == 1) {
    p2g_item_sums<15, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
  } else if (SPLIT == 2) {
    if (part == 0u) p2g_item_sums<9, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
    else p2g_item_sums<6, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
  } else {
    if (part == 0u) p2g_item_sums<1, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
    else if (part == 1u) p2g_item_sums<2, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
    else if (part == 2u) p2g_item_sums<4, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
    else p2g_item_sums<8, BATCH>(p, rec, it, sorted, s_rho0, out, stride);
  }
}


// ---------------------------------------------------------------------------
// GRID UPDATE
// ---------------------------------------------------------------------------
// Mass and momentum of node (local (lx, ly, lz) in tile (tx, ty, tz) of scene
// g): the partial boxes of the occupied tiles whose 10^3 box contains it,
// summed in a fixed order.  False when no occupied tile's box contains it
// (then it lies in no particle's stencil).
__device__ __forceinline__ bool sum_partials(const SceneGeo& g, int tx, int ty, int tz, int lx, int ly, int lz,
                                             const int32_t* __restrict__ tile_act,
                                             const float4* __restrict__ partial, float& mx, float& my, float& mz,
                                             float& mass) {
  const int td = int(g.tile_dim);
  mx = my = mz = mass = 0.f;
  bool covered = false;
  for (int dz = -1; dz <= 1; dz++) {
    if ((dz < 0 && lz != 0) || (dz > 0 && lz != 7)) continue;
    const int sz = tz + dz;
    if (sz < 0 || sz >= td) continue;
    for (int dy = -1; dy <= 1; dy++) {
      if ((dy < 0 && ly != 0) || (dy > 0 && ly != 7)) continue;
      const int sy = ty + dy;
      if (sy < 0 || sy >= td) continue;
      for (int dx = -1; dx <= 1; dx++) {
        if ((dx < 0 && lx != 0) || (dx > 0 && lx != 7)) continue;
        const int sx = tx + dx;
        if (sx < 0 || sx >= td) continue;
        const int32_t a = tile_act[tile_id(g, sx, sy, sz)];
        if (a < 0) continue;
        const int bx = lx - 8 * dx + 1, by = ly - 8 * dy + 1, bz = lz - 8 * dz + 1;
        const float4 q = partial[size_t(a) * kBoxNodes + (bz * kBox + by) * kBox + bx];
        mx += q.x; my += q.y; mz += q.z; mass += q.w;
        covered = true;
      }
    }
  }
  return covered;
}

// The update of a node with mass >= 1e-10 at grid coordinates (nx, ny, nz),
// in registers and in this order: the 15 m/s cap, the saved (pre-force)
// velocity, forces, walls, analytic colliders, the dense-SDF BC
// (shaders/mpm_grid_update.comp:30-110, shaders/mpm_nanovdb_bc.comp:23-54).
// v enters as momentum / mass; o receives the saved velocity.  node_update is
// the whole of it for force lists without turbulence and noise.
__device__ __forceinline__ void node_cap(float& vx, float& vy, float& vz) {
  const float sp = len3(vx, vy, vz);
  const float vmax = 15.f;
  if (sp > vmax) {
    const float k = vmax / sp;
    vx *= k; vy *= k; vz *= k;
  }
}
// walls, analytic colliders and the dense SDF; (px, py, pz) is the node's position
__device__ __forceinline__ void node_bc(const SubParams& p, const SceneGeo& g, int nx, int ny, int nz, float px,
                                        float py, float pz, float& vx, float& vy, float& vz,
                                        const float* __restrict__ sdf, const nb_collider* __restrict__ cols) {
  // separating walls on the two outer node layers (shaders/mpm_grid_update.comp:54-60)
  const int Nx = g.grid_res[0] - 1, Ny = g.grid_res[1] - 1, Nz = g.grid_res[2] - 1;
  if (nx <= 1 && vx < 0.f) vx = 0.f;
  if (nx >= Nx - 1 && vx > 0.f) vx = 0.f;
  if (ny <= 1 && vy < 0.f) vy = 0.f;
  if (ny >= Ny - 1 && vy > 0.f) vy = 0.f;
  if (nz <= 1 && vz < 0.f) vz = 0.f;
  if (nz >= Nz - 1 && vz > 0.f) vz = 0.f;
  for (uint32_t ci = 0; ci < p.collider_count; ci++) {
    const nb_collider c = cols[ci];
    float cnx, cny, cnz;
    const float sd = collider_sdf(c, px, py, pz, cnx, cny, cnz);
    if (sd <= 0.f) collider_bc(vx, vy, vz, cnx, cny, cnz, c);
  }
  // dense-SDF BC (shaders/mpm_nanovdb_bc.comp:23-54)
  if (sdf) {
    const float sd = sample_sdf(sdf, g, nx, ny, nz);
    if (sd < 0.f) {
      vx = vy = vz = 0.f;
    } else if (sd < g.h * 1.5f) {
      const float gx = sample_sdf(sdf, g, nx + 1, ny, nz) - sample_sdf(sdf, g, nx - 1, ny, nz);
      const float gy = sample_sdf(sdf, g, nx, ny + 1, nz) - sample_sdf(sdf, g, nx, ny - 1, nz);
      const float gz = sample_sdf(sdf, g, nx, ny, nz + 1) - sample_sdf(sdf, g, nx, ny, nz - 1);
      const float gl = len3(gx, gy, gz);
      if (gl > 1e-6f) {
        const float ux = gx / gl, uy = gy / gl, uz = gz / gl;
        const float vn = vx * ux + vy * uy + vz * uz;
        if (vn < 0.f) {
          vx -= vn * ux; vy -= vn * uy; vz -= vn * uz;
        }
      }
    }
  }
}
__device__ __forceinline__ void node_update(const SubParams& p, const SceneGeo& g, int nx, int ny, int nz, float& vx,
                                            float& vy, float& vz, float& ox, float& oy, float& oz,
                                            const float* __restrict__ sdf, const nb_collider* __restrict__ cols,
                                            const nb_force* __restrict__ forces) {
  node_cap(vx, vy, vz);
  ox = vx; oy = vy; oz = vz;
  const float3 x = node_pos(g, nx, ny, nz);
  apply_forces(vx, vy, vz, forces, p.force_count, p.dt);
  node_bc(p, g, nx, ny, nz, x.x, x.y, x.z, vx, vy, vz, sdf, cols);
}

// node_update with turbulence or noise in the force list, and its stores, for a block
// as tile_forces takes it
template <uint32_t ROLES>
__device__ __forceinline__ void grid_node_noise(const SubParams& p, const SceneGeo& g, int nx, int ny, int nz, size_t nid,
                                                bool live, const float4 m, float3 first, float3 last,
                                                float4* __restrict__ grid_node, float4* __restrict__ grid_old,
                                                const float* __restrict__ sdf, const nb_collider* __restrict__ cols,
                                                const nb_force* __restrict__ forces, NoiseLds& lds) {
  const bool own = live && threadIdx.x < kNoiseThreads / ROLES;
  float vx = 0.f, vy = 0.f, vz = 0.f;
  if (own) {
    vx = m.x / m.w; vy = m.y / m.w; vz = m.z / m.w;
    node_cap(vx, vy, vz);
    if (p.write_old) grid_old[nid] = make_float4(vx, vy, vz, 0.f);
  }
  const float3 x = node_pos(g, nx, ny, nz);
  tile_forces<ROLES>(vx, vy, vz, x.x, x.y, x.z, live, first, last, forces, p.force_count, p.dt, lds);
  if (own) {
    node_bc(p, g, nx, ny, nz, x.x, x.y, x.z, vx, vy, vz, sdf, cols);
    grid_node[nid] = make_float4(vx, vy, vz, m.w);
  }
}

// The grid update of the grid's own contents, node tile by node tile.
template <bool BATCH, bool NOISE>
__global__ __launch_bounds__(512) void k_grid(SubParams p, const uint32_t* __restrict__ tiles,
                                              const uint32_t* __restrict__ count, float4* __restrict__ grid_node,
                                              float4* __restrict__ grid_old, float4* __restrict__ grid_pre,
                                              const float* __restrict__ sdf, const nb_collider* __restrict__ cols,
                                              const nb_force* __restrict__ forces) {
  const uint32_t nb_tiles = *count;
  // thread j holds the tile's j-th node in Morton order (contiguous in HBM)
  const uint32_t j = threadIdx.x;
  for (uint32_t b = blockIdx.x; b < nb_tiles; b += gridDim.x) {
    const uint32_t N = tiles[b];
    const SceneGeo g = tile_geo<BATCH>(p, N);
    int tx, ty, tz;
    tile_coords(g, N, tx, ty, tz);
    const int nx = tx * 8 + int(morton_compact(j)), ny = ty * 8 + int(morton_compact(j >> 1)),
              nz = tz * 8 + int(morton_compact(j >> 2));
    const size_t nid = (size_t(N) << kTileBits) | j;
    const float4 m = grid_node[nid];
    const float mass = m.w;
    if (grid_pre)
      grid_pre[nid] = mass < 1e-10f ? make_float4(0.f, 0.f, 0.f, mass) : make_float4(m.x / mass, m.y / mass, m.z / mass, mass);
    // massless nodes keep their momentum (shaders/mpm_grid_update.comp:109-110)
    const bool live = !(mass < 1e-10f);
    if constexpr (NOISE) {
      __shared__ NoiseLds s_noise;
      if (!__syncthreads_or(live)) continue;
      grid_node_noise<1>(p, g, nx, ny, nz, nid, live, m, node_pos(g, tx * 8, ty * 8, tz * 8),
                      node_pos(g, tx * 8 + 7, ty * 8 + 7, tz * 8 + 7), grid_node, grid_old, sdf, cols, forces, s_noise);
    } else if (live) {
      float vx = m.x / mass, vy = m.y / mass, vz = m.z / mass, ox, oy, oz;
      node_update(p, g, nx, ny, nz, vx, vy, vz, ox, oy, oz, sdf, cols, forces);
      if (p.write_old) grid_old[nid] = make_float4(ox, oy, oz, 0.f);
      grid_node[nid] = make_float4(vx, vy, vz, mass);
    }
  }
}

// The grid update from the boxes, per occupied tile (see NeighbourTiles).
template <bool UPDATE, bool BATCH>
__global__ __launch_bounds__(512) void k_grid_tiles(SubParams p, const float4* __restrict__ partial,
                                                    const int32_t* __restrict__ tile_act,
                                                    const uint32_t* __restrict__ act_tiles,
                                                    const uint32_t* __restrict__ counters, float4* __restrict__ grid_node,
                                                    float4* __restrict__ grid_old, float4* __restrict__ grid_pre,
                                                    const float* __restrict__ sdf, const nb_collider* __restrict__ cols,
                                                    const nb_force* __restrict__ forces) {
  __shared__ NeighbourTiles s_near;
  const uint32_t na = counters[CNT_ACTIVE];
  const bool split = na <= kGridSplitTiles;
  for (uint32_t w = blockIdx.x; w < (split ? 2u * na : na); w += gridDim.x) {
    const uint32_t T = act_tiles[w < na ? w : w - na];
    const SceneGeo g = tile_geo<BATCH>(p, T);
    int tx, ty, tz;
    tile_coords(g, T, tx, ty, tz);
    load_neighbours(g, tx, ty, tz, tile_act, s_near);
    const int last = s_near.open && (!split || w >= na) ? 1 : 0;
#pragma unroll 1
    for (int shell = w < na ? 0 : 1; shell <= last; shell++) {
      int bx, by, bz;
      float4 m;
      if (!box_node(shell != 0, bx, by, bz) || !sum_boxes(s_near, shell != 0, bx, by, bz, partial, m)) continue;
      const int nx = tx * 8 + bx - 1, ny = ty * 8 + by - 1, nz = tz * 8 + bz - 1;
      const size_t nid = node_id(g, uint32_t(nx), uint32_t(ny), uint32_t(nz));
      const float mass = m.w;
      if (grid_pre)
        grid_pre[nid] = mass < 1e-10f ? make_float4(0.f, 0.f, 0.f, mass) : make_float4(m.x / mass, m.y / mass, m.z / mass, mass);
      // massless nodes keep their momentum (shaders/mpm_grid_update.comp:109-110)
      if (!UPDATE || mass < 1e-10f) {
        grid_node[nid] = m;
        continue;
      }
      float vx = m.x / mass, vy = m.y / mass, vz = m.z / mass, ox, oy, oz;
      node_update(p, g, nx, ny, nz, vx, vy, vz, ox, oy, oz, sdf, cols, forces);
      if (p.write_old) grid_old[nid] = make_float4(ox, oy, oz, 0.f);
      grid_node[nid] = make_float4(vx, vy, vz, mass);
    }
  }
}

// The same with turbulence or noise.
template <uint32_t ROLES, bool BATCH>
__device__ __forceinline__ void grid_noise(const SubParams& p, const float4* __restrict__ partial,
                                           const int32_t* __restrict__ tile_act, const uint32_t* __restrict__ act_tiles,
                                           uint32_t na, float4* __restrict__ grid_node, float4* __restrict__ grid_old,
                                           float4* __restrict__ grid_pre, const float* __restrict__ sdf,
                                           const nb_collider* __restrict__ cols, const nb_force* __restrict__ forces,
                                           NeighbourTiles& near, NoiseLds& lds, uint64_t* s_live) {
  constexpr uint32_t kNodes = kNoiseThreads / ROLES;
  for (uint32_t w = blockIdx.x; w < noise_units<ROLES>() * na; w += gridDim.x) {
    const uint32_t unit = w / na, T = act_tiles[w % na];
    const SceneGeo g = tile_geo<BATCH>(p, T);
    int tx, ty, tz, b[3], lo[3], hi[3];
    tile_coords(g, T, tx, ty, tz);
    load_neighbours(g, tx, ty, tz, tile_act, near);
    const bool shell = noise_shell<ROLES>(unit);
    if (shell && !near.open) continue;
    float4 m = make_float4(0.f, 0.f, 0.f, 0.f);
    const bool node = noise_unit_node<ROLES>(unit, int(threadIdx.x % kNodes), b, lo, hi);
    const bool covered = node && threadIdx.x < kNodes && sum_boxes(near, shell, b[0], b[1], b[2], partial, m);
    const int nx = tx * 8 + b[0] - 1, ny = ty * 8 + b[1] - 1, nz = tz * 8 + b[2] - 1;
    const size_t nid = covered ? node_id(g, uint32_t(nx), uint32_t(ny), uint32_t(nz)) : 0;
    bool live = covered && !(m.w < 1e-10f), any;
    if (covered && grid_pre)
      grid_pre[nid] = live ? make_float4(m.x / m.w, m.y / m.w, m.z / m.w, m.w) : make_float4(0.f, 0.f, 0.f, m.w);
    // massless nodes keep their momentum (shaders/mpm_grid_update.comp:109-110)
    if (covered && !live) grid_node[nid] = m;
    live = noise_live<ROLES>(live, s_live, any);
    if (!any) continue;
    grid_node_noise<ROLES>(p, g, nx, ny, nz, nid, live, m,
                           node_pos(g, tx * 8 + lo[0] - 1, ty * 8 + lo[1] - 1, tz * 8 + lo[2] - 1),
                           node_pos(g, tx * 8 + hi[0] - 1, ty * 8 + hi[1] - 1, tz * 8 + hi[2] - 1), grid_node, grid_old,
                           sdf, cols, forces, lds);
  }
}
template <bool BATCH>
__global__ __launch_bounds__(kNoiseThreads) void k_grid_noise(SubParams p, const float4* __restrict__ partial,
                                                              const int32_t* __restrict__ tile_act,
                                                              const uint32_t* __restrict__ act_tiles,
                                                              const uint32_t* __restrict__ counters,
                                                              float4* __restrict__ grid_node,
                                                              float4* __restrict__ grid_old,
                                                              float4* __restrict__ grid_pre,
                                                              const float* __restrict__ sdf,
                                                              const nb_collider* __restrict__ cols,
                                                              const nb_force* __restrict__ forces) {
  __shared__ NeighbourTiles s_near;
  __shared__ NoiseLds s_noise;
  __shared__ uint64_t s_live[2];
  const uint32_t na = counters[CNT_ACTIVE];
  if (na <= kNoiseSplitTiles)
    grid_noise<4, BATCH>(p, partial, tile_act, act_tiles, na, grid_node, grid_old, grid_pre, sdf, cols, forces, s_near,
                         s_noise, s_live);
  else
    grid_noise<1, BATCH>(p, partial, tile_act, act_tiles, na, grid_node, grid_old, grid_pre, sdf, cols, forces, s_near,
                         s_noise, s_live);
}

// ---------------------------------------------------------------------------
// G2P
// ---------------------------------------------------------------------------
// What the 27-node gather gives a particle (shaders/mpm_g2p.comp:80-113): the
// PIC velocity, FLIP's saved-velocity interpolant, the velocity gradient
// vg.m[col = gradient axis][row = component] and APIC's B.
struct G2PGather {
  float vpx, vpy, vpz, vox, voy, voz;
  m3 vg, Bn;
};

// The gather.  node(ix, iy, iz, v, vo) returns whether the stencil node
// (base + (ix, iy, iz)) takes part (in the grid, mass >= 1e-10) and its
// velocity in v (and FLIP's saved velocity in vo), both zero when it does not.
// The 27 nodes are contracted axis by axis (x, then y, then z) in three rolled
// z slabs, so only one slab's node loads are live.  When some node of the
// particle has 0 < w < 1e-12 (tiny), the reference's weight cut
// (shaders/mpm_g2p.comp:93-101) changes the sums, and they are taken node by
// node with the cut instead; each lane decides alone, so each particle's
// result depends on its own data only.
template <bool FLIP, class NodeFn>
__device__ __forceinline__ void g2p_gather(const Axis3 (&ax3)[3], bool tiny, NodeFn node, G2PGather& o) {
  float vpx = 0.f, vpy = 0.f, vpz = 0.f, vox = 0.f, voy = 0.f, voz = 0.f;
  m3 vg = m3_zero(), Bn = m3_zero();
  const Axis3 &X = ax3[0], &Y = ax3[1];
  // the slab's z stencil values sit in position 0 and rotate at the end of
  // each iteration
  float zw[3] = {ax3[2].w[0], ax3[2].w[1], ax3[2].w[2]};
  float zg[3] = {ax3[2].g[0], ax3[2].g[1], ax3[2].g[2]};
  float zd[3] = {ax3[2].dx[0], ax3[2].dx[1], ax3[2].dx[2]};
  if (!tiny) {
    float wdx[3], wdy[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      wdx[i] = X.w[i] * X.dx[i];
      wdy[i] = Y.w[i] * Y.dx[i];
    }
#pragma unroll 1
    for (int iz = 0; iz < 3; iz++) {
      // sums start from their first term (no zero-initialised accumulators)
      float Y00[3], Y01[3], Y02[3], Y1[3], Y2[3], YO[3];
#pragma unroll
      for (int iy = 0; iy < 3; iy++) {
        float gv[3][3], go[3][3];
#pragma unroll
        for (int ix = 0; ix < 3; ix++) (void)node(ix, iy, iz, gv[ix], go[ix]);
        float X0[3], X1[3], X2[3], XO[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
          X0[c] = X.w[0] * gv[0][c] + X.w[1] * gv[1][c] + X.w[2] * gv[2][c];
          X1[c] = X.g[0] * gv[0][c] + X.g[1] * gv[1][c] + X.g[2] * gv[2][c];
          X2[c] = wdx[0] * gv[0][c] + wdx[1] * gv[1][c] + wdx[2] * gv[2][c];
          if (FLIP) XO[c] = X.w[0] * go[0][c] + X.w[1] * go[1][c] + X.w[2] * go[2][c];
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
          if (iy == 0) {
            Y00[c] = Y.w[0] * X0[c];
            Y01[c] = Y.g[0] * X0[c];
            Y02[c] = wdy[0] * X0[c];
            Y1[c] = Y.w[0] * X1[c];
            Y2[c] = Y.w[0] * X2[c];
            if (FLIP) YO[c] = Y.w[0] * XO[c];
          } else {
            Y00[c] += Y.w[iy] * X0[c];
            Y01[c] += Y.g[iy] * X0[c];
            Y02[c] += wdy[iy] * X0[c];
            Y1[c] += Y.w[iy] * X1[c];
            Y2[c] += Y.w[iy] * X2[c];
            if (FLIP) YO[c] += Y.w[iy] * XO[c];
          }
        }
      }
      const float wz = zw[0], gz = zg[0], wdz = zw[0] * zd[0];
      float* vp3[3] = {&vpx, &vpy, &vpz};
      float* vo3[3] = {&vox, &voy, &voz};
#pragma unroll
      for (int c = 0; c < 3; c++) {
        *vp3[c] += wz * Y00[c];
        if (FLIP) *vo3[c] += wz * YO[c];
        // vg = sum outer(v_i, grad w_i): vg.m[col = grad axis][row = velocity component]
        vg.m[0][c] += wz * Y1[c];
        vg.m[1][c] += wz * Y01[c];
        vg.m[2][c] += gz * Y00[c];
        // Bn = sum outer(w_i v_i, x_i - x_p)
        Bn.m[0][c] += wz * Y2[c];
        Bn.m[1][c] += wz * Y02[c];
        Bn.m[2][c] += wdz * Y00[c];
      }
      zw[0] = zw[1]; zw[1] = zw[2];
      zg[0] = zg[1]; zg[1] = zg[2];
      zd[0] = zd[1]; zd[1] = zd[2];
    }
  } else {
#pragma unroll 1
    for (int iz = 0; iz < 3; iz++) {
      const float wz = zw[0], gz = zg[0], dxz = zd[0];
#pragma unroll
      for (int iy = 0; iy < 3; iy++) {
#pragma unroll
        for (int ix = 0; ix < 3; ix++) {
          float gvv[3], gov[3];
          const bool in = node(ix, iy, iz, gvv, gov);
          const float wx = X.w[ix], wy = Y.w[iy];
          const float w0 = wx * wy * wz;
          const bool live = in && w0 >= 1e-12f;
          const float gx = live ? gvv[0] : 0.f, gy = live ? gvv[1] : 0.f, gzv = live ? gvv[2] : 0.f;
          const float w = live ? w0 : 0.f;
          const float dwx = live ? X.g[ix] * wy * wz : 0.f;
          const float dwy = live ? wx * Y.g[iy] * wz : 0.f;
          const float dwz = live ? wx * wy * gz : 0.f;
          const float dxx = X.dx[ix], dxy = Y.dx[iy];
          vpx += w * gx; vpy += w * gy; vpz += w * gzv;
          // outerProduct(vi, dw)[j][i] = vi[i]*dw[j]
          vg.m[0][0] += gx * dwx; vg.m[0][1] += gy * dwx; vg.m[0][2] += gzv * dwx;
          vg.m[1][0] += gx * dwy; vg.m[1][1] += gy * dwy; vg.m[1][2] += gzv * dwy;
          vg.m[2][0] += gx * dwz; vg.m[2][1] += gy * dwz; vg.m[2][2] += gzv * dwz;
          const float wgx = w * gx, wgy = w * gy, wgz = w * gzv;
          Bn.m[0][0] += wgx * dxx; Bn.m[0][1] += wgy * dxx; Bn.m[0][2] += wgz * dxx;
          Bn.m[1][0] += wgx * dxy; Bn.m[1][1] += wgy * dxy; Bn.m[1][2] += wgz * dxy;
          Bn.m[2][0] += wgx * dxz; Bn.m[2][1] += wgy * dxz; Bn.m[2][2] += wgz * dxz;
          if (FLIP) {
            vox += w * (live ? gov[0] : 0.f);
            voy += w * (live ? gov[1] : 0.f);
            voz += w * (live ? gov[2] : 0.f);
          }
        }
      }
      zw[0] = zw[1]; zw[1] = zw[2];
      zg[0] = zg[1]; zg[1] = zg[2];
      zd[0] = zd[1]; zd[1] = zd[2];
    }
  }
  o.vpx = vpx; o.vpy = vpy; o.vpz = vpz;
  o.vox = vox; o.voy = voy; o.voz = voz;
  o.vg = vg;
  o.Bn = Bn;
}

// Stencil of particle position x: per axis the first stencil node base =
// floor((x - wmin)/h) - 1 (the quotient clamped to a range that keeps every
// integer below in bounds without changing which nodes are valid) and the
// weights; tiny: some node has 0 < w < 1e-12 (the smallest positive
// per-axis weights bound every w from below).
__device__ __forceinline__ bool g2p_stencil(const SceneGeo& g, float xp, float yp, float zp, int (&base)[3],
                                            Axis3 (&ax3)[3]) {
  const float xs[3] = {xp, yp, zp};
  float fq[3];
  bool ok = true;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    fq[a] = cell_coord(g, xs[a], a);
    const float f = fminf(fmaxf(fq[a], -4.f), float(g.grid_res[a]) + 4.f);
    base[a] = int(floorf(f)) - 1;
    ok &= axis_stencil_cell(fq[a], xs[a], g.wmin[a], g.h, g.inv_h, base[a] + 1, ax3[a]);
  }
  if (!ok) {  // the first cell layer, or outside the grid
#pragma unroll
    for (int a = 0; a < 3; a++) axis_stencil_f(fq[a], xs[a], g.wmin[a], g.h, g.inv_h, base[a], ax3[a]);
  }
  return (min_positive3(ax3[0].w) * min_positive3(ax3[1].w)) * min_positive3(ax3[2].w) < 1e-12f;
}

// The fallback's counters (NB_SVD_FB_*): one set of atomics per wave, from
// ballots over the lanes that reach the call together.
__device__ __forceinline__ void fb_count_stats(unsigned long long* st, bool dp_lane, bool fb_proj, bool fb_stress) {
  const uint64_t b_dp = __ballot(dp_lane), b_pr = __ballot(fb_proj), b_st = __ballot(fb_stress);
  if ((threadIdx.x & 63u) == uint32_t(__ffsll((unsigned long long)__ballot(true)) - 1)) {
    if (b_dp) {
      atomicAdd(&st[NB_SVD_FB_DP_LANES], (unsigned long long)__popcll(b_dp));
      atomicAdd(&st[NB_SVD_FB_DP_WAVES], 1ull);
    }
    if (b_pr) atomicAdd(&st[NB_SVD_FB_PROJ_LANES], (unsigned long long)__popcll(b_pr));
    if (b_st) atomicAdd(&st[NB_SVD_FB_STRESS_LANES], (unsigned long long)__popcll(b_st));
    if (b_pr | b_st) atomicAdd(&st[NB_SVD_FB_FB_WAVES], 1ull);
  }
}

// The FP64 fallback's computation, from an FP32 trial F: the return map
// (SVD, projection, recomposition) and the Hencky stress of its result, in
// FP64 and rounded once.  All of it stays FP64: the stress SVD of a
// recomposed F' with a close pair is as sensitive to F' as the first SVD is
// to F, so an F' rounded to FP32 (or built with FP32 exp) would decide its
// singular vectors again.
struct FTau {
  m3 F, tau;
};
__device__ __forceinline__ FTau plastic_fp64(const m3& F, bool dp, float mu_f, float lam_f, float q_max, float M,
                                             float q_c, bool cs) {
  const double mu = mu_f, lam = lam_f;
  const PlasticOutT<double> pd =
      project_plastic(m3_convert<double>(F), dp, mu, lam, double(q_max), double(M), double(q_c), cs);
  FTau r;
  r.F = m3_round(pd.F);
  r.tau = m3_round((cs || !pd.recomposed) ? hencky_from_log(pd.U, pd.eps[0], pd.eps[1], pd.eps[2], mu, lam)
                                          : hencky_stress(pd.F, mu, lam, cs));
  return r;
}

// The FP64 fallback's queue: kFbSlots slots of p.fb_region = ceil(n /
// kFbSlots) entries; a particle at place k of the G2P order goes to slot
// k / fb_region, so a slot never overflows and its atomics come from a
// fraction of the waves.  An entry is kFbEntry float4: q, mode, then F_old
// and the velocity gradient, 9 floats each in m[0][0], m[0][1], ..., m[2][2]
// order (m[col][row] storage).  mode 1: return map and stress from the trial
// F = (I + dt grad v) F_old; 2: stress of the record's F; 0: dropped.  Slot
// counters sit kFbCtlStride words apart, the k_g2p_fb block count after them.
constexpr uint32_t kFbNone = 0xFFFFFFFFu;

// queue the particle if it takes the fallback (all lanes of the wave call
// this together); returns its entry or kFbNone
__device__ __forceinline__ uint32_t queue_fb(const SubParams& p, uint32_t k, uint32_t q, const float4* r,
                                             const m3& vg, bool fb_proj, bool fb_stress) {
  const bool fb = fb_proj || fb_stress;
  uint64_t pending = __ballot(fb);
  if (!pending) return kFbNone;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t slot = k / p.fb_region;
  uint32_t at = kFbNone;
  // the wave's queued lanes grouped by slot (one group unless the wave
  // straddles a slot boundary); one atomic per group
  while (pending) {
    const uint32_t leader = uint32_t(__ffsll((unsigned long long)pending) - 1);
    const uint32_t ls = uint32_t(__shfl(int(slot), int(leader)));
    const uint64_t peers = __ballot(fb && slot == ls);
    uint32_t base = 0u;
    if (lane == leader) base = atomicAdd(&p.fb_ctl[ls * kFbCtlStride], uint32_t(__popcll(peers)));
    base = uint32_t(__shfl(int(base), int(leader)));
    if (fb && slot == ls) at = ls * p.fb_region + base + uint32_t(__popcll(peers & ((1ull << lane) - 1ull)));
    pending &= ~peers;
  }
  if (fb) {
    float4* e = p.fb_queue + size_t(at) * kFbEntry;
    if (fb_proj) {
      // F_old is still the record's (the record is written after this)
      const float4 rt = r[R_T], fa = r[R_FA], fb4 = r[R_FB];
      e[0] = make_float4(__uint_as_float(q), __uint_as_float(1u), rt.w, fa.x);
      e[1] = make_float4(fa.y, fa.z, fa.w, fb4.x);
      e[2] = make_float4(fb4.y, fb4.z, fb4.w, vg.m[0][0]);
      e[3] = make_float4(vg.m[0][1], vg.m[0][2], vg.m[1][0], vg.m[1][1]);
      e[4] = make_float4(vg.m[1][2], vg.m[2][0], vg.m[2][1], vg.m[2][2]);
    } else {
      e[0] = make_float4(__uint_as_float(q), __uint_as_float(2u), 0.f, 0.f);
    }
  }
  return at;
}

// Everything of G2P after the gather (shaders/mpm_g2p.comp:115-272): F
// update, constitutive update (fluid; elastic; Von Mises / Drucker-Prager
// family return map with the FP64 fallback for near-degenerate F), mud
// viscosity, Jacobian reset, PIC/APIC/FLIP velocity, advection, SDF push-out,
// world clamp; writes the record and the next substep's cell key.
// A particle whose update the FP64 fallback takes over finishes here in FP32
// with its stress set to the mud viscosity term alone (zero for the other
// models) and is queued for k_g2p_fb (queue_fb), which replaces F and tau
// with the FP64 results; if the Jacobian reset or the SDF push-out then sets
// F = I, tau = 0 (both decided on the FP32 F), its entry is cancelled.  The
// FP64 code thus stays out of the kernels that run every particle (a call
// site alone costs such a kernel registers and time even when no lane takes
// it).  k: the particle's place in the G2P order, which picks its queue slot.
template <bool FLIP, bool BATCH>
__device__ __forceinline__ void g2p_particle(const SubParams& p, uint32_t k, uint32_t q, const float4* r, float4* ro,
                                             uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                             uint32_t* __restrict__ tile_cnt, const nb_material& mat,
                                             const G2PGather& gth, const float4 pp, const float4 vel,
                                             const float* __restrict__ sdf) {
  const float xp = pp.x, yp = pp.y, zp = pp.z, Vp = pp.w;
  constexpr bool flip = FLIP;  // flip_ratio > 0.01
  float vpx = gth.vpx, vpy = gth.vpy, vpz = gth.vpz;
  m3 Bn = gth.Bn;
  const float4 rt = r[R_T], fa = r[R_FA], fb = r[R_FB];
  m3 F;
  F.m[0][0] = rt.w; F.m[0][1] = fa.x; F.m[0][2] = fa.y;
  F.m[1][0] = fa.z; F.m[1][1] = fa.w; F.m[1][2] = fb.x;
  F.m[2][0] = fb.y; F.m[2][1] = fb.z; F.m[2][2] = fb.w;
  m3 L;
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int rr = 0; rr < 3; rr++) L.m[c][rr] = (c == rr ? 1.f : 0.f) + p.dt * gth.vg.m[c][rr];
  m3 Fn = m3_mul(L, F);

  m3 tau;
  const bool cs = p.corrected_svd != 0u;
  bool dp_lane = false, fb_proj = false, fb_stress = false;  // for the fallback's counters
  if (mat.model == NB_MAT_FLUID) {
    float J = fmaxf(m3_det(Fn), 1e-4f);
    const float cr = powf(J, 1.f / 3.f);
    Fn = m3_diag(cr, cr, cr);
    const float pr = mat.bulkK * (J - 1.f);
    tau = m3_diag(pr, pr, pr);
  } else {
    // elastic: Hencky stress of F; Von Mises / Drucker-Prager (also granular
    // powder and viscoplastic mud): return map, then Hencky stress of the
    // projected F.  In corrected mode the return map's SVD is the true SVD of
    // the projected F, so its factors give the stress without a second SVD.
    // In either mode a Von Mises particle inside the yield surface keeps F
    // unchanged, so the second SVD would repeat the first on the same input.
    const bool dp = mat.model == NB_MAT_DRUCKER_PRAGER || mat.model == NB_MAT_GRANULAR_POWDER ||
                    mat.model == NB_MAT_VISCOPLASTIC_MUD;
    const bool plastic = dp || mat.model == NB_MAT_VON_MISES;
    const bool fb_on = dp && p.svd_fp64 != 0u;
    dp_lane = dp;
    bool have_tau = false;
    if (plastic) {
      const PlasticOut po = project_plastic(Fn, dp, mat.mu, mat.lambda, mat.q_max, mat.M_friction, mat.q_cohesion, cs);
      Fn = po.F;
      if (cs || !po.recomposed) {
        tau = hencky_from_log(po.U, po.eps[0], po.eps[1], po.eps[2], mat.mu, mat.lambda);
        have_tau = true;
      }
      if (fb_on && fb_rounding_decides(po.sig, p.svd_gap_rel, p.svd_zero_rel, cs, po.recomposed, Fn, po.eps,
                                       have_tau, tau, po.eps, mat.mu, mat.lambda)) {
        // rounding decides the trial F's singular vectors and the result
        // depends on them: k_g2p_fb redoes the return map and the stress in
        // FP64 from the same FP32 trial F
        have_tau = true;
        fb_proj = true;
      }
    }
    if (!have_tau) {
      // Hencky stress of F (hencky_stress written out, so that a particle that
      // does not take the fallback runs the same instructions whether it is on
      // or off); the stress SVD of a recomposed Drucker-Prager F is tested on
      // its own singular values
      m3 U, V;
      float sig[3];
      svd3(Fn, U, sig, V, cs);
      const float e[3] = {log_strain(sig[0]), log_strain(sig[1]), log_strain(sig[2])};
      tau = hencky_from_log(U, e[0], e[1], e[2], mat.mu, mat.lambda);
      if (fb_on && fb_rounding_decides(sig, p.svd_gap_rel, p.svd_zero_rel, cs, false, Fn, e, true, tau, e, mat.mu,
                                       mat.lambda))
        fb_stress = true;
    }
    if (fb_proj || fb_stress) tau = m3_zero();  // k_g2p_fb adds the FP64 stress
    if (mat.model == NB_MAT_VISCOPLASTIC_MUD) {
      m3 D;
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int rr = 0; rr < 3; rr++) D.m[c][rr] = 0.5f * (gth.vg.m[c][rr] + gth.vg.m[rr][c]);
      const float trD = D.m[0][0] + D.m[1][1] + D.m[2][2];
      const float k2 = 2.f * mat.viscosity;
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int rr = 0; rr < 3; rr++) tau.m[c][rr] += k2 * (D.m[c][rr] - (c == rr ? trD / 3.f : 0.f));
    }
  }
  // every lane of the wave is here
  if (p.svd_stats) fb_count_stats(p.svd_stats, dp_lane, fb_proj, fb_stress);
  const uint32_t fb_at = p.svd_fp64 ? queue_fb(p, k, q, r, gth.vg, fb_proj, fb_stress) : kFbNone;

  bool jreset = false;
  {
    const float Jd = fabsf(m3_det(Fn));
    if (Jd < 0.15f || Jd > 10.f) {
      Fn = m3_ident();
      tau = m3_zero();
      jreset = true;
    }
  }
  if (p.flip_ratio > -0.5f) Bn = m3_zero();

  float vnx, vny, vnz;
  if (flip) {
    const float rf = p.flip_ratio;
    const float fx = vel.x + (vpx - gth.vox), fy = vel.y + (vpy - gth.voy), fz = vel.z + (vpz - gth.voz);
    vnx = vpx * (1.f - rf) + fx * rf;
    vny = vpy * (1.f - rf) + fy * rf;
    vnz = vpz * (1.f - rf) + fz * rf;
  } else {
    vnx = vpx; vny = vpy; vnz = vpz;
  }
  if (jreset) { vnx *= 0.1f; vny *= 0.1f; vnz *= 0.1f; }
  float xn = xp + p.dt * vnx, yn = yp + p.dt * vny, zn = zp + p.dt * vnz;

  // The geometry is read again for the tail rather than kept live through
  // the SVD (a plain engine re-reads its kernel arguments).
  const SceneGeo ge = particle_geo<BATCH>(p, q);
  // particle-level SDF push-out (shaders/mpm_g2p.comp:220-252)
  bool pushed = false;
  if (sdf) {
    const int gx = ge.grid_res[0] - 1, gy = ge.grid_res[1] - 1, gz = ge.grid_res[2] - 1;
    float fx = fminf(fmaxf(cell_coord(ge, xn, 0), -4.f), float(ge.grid_res[0]) + 4.f);
    float fy = fminf(fmaxf(cell_coord(ge, yn, 1), -4.f), float(ge.grid_res[1]) + 4.f);
    float fz = fminf(fmaxf(cell_coord(ge, zn, 2), -4.f), float(ge.grid_res[2]) + 4.f);
    const int ix = min(max(int(floorf(fx)), 0), gx);
    const int iy = min(max(int(floorf(fy)), 0), gy);
    const int iz = min(max(int(floorf(fz)), 0), gz);
    const float psdf = sdf[morton3(ix, iy, iz)];
    if (psdf < 0.f) {
      const float gnx = sdf[morton3(min(ix + 1, gx), iy, iz)] - sdf[morton3(max(ix - 1, 0), iy, iz)];
      const float gny = sdf[morton3(ix, min(iy + 1, gy), iz)] - sdf[morton3(ix, max(iy - 1, 0), iz)];
      const float gnz = sdf[morton3(ix, iy, min(iz + 1, gz))] - sdf[morton3(ix, iy, max(iz - 1, 0))];
      const float gl = len3(gnx, gny, gnz);
      if (gl > 1e-6f) {
        const float ux = gnx / gl, uy = gny / gl, uz = gnz / gl;
        xn -= psdf * ux; yn -= psdf * uy; zn -= psdf * uz;
        const float vn = vnx * ux + vny * uy + vnz * uz;
        if (vn < 0.f) { vnx -= vn * ux; vny -= vn * uy; vnz -= vn * uz; }
      } else {
        xn = xp; yn = yp; zn = zp;
        vnx = vny = vnz = 0.f;
      }
      Fn = m3_ident();
      tau = m3_zero();
      pushed = true;
    }
  }
  // world clamp at a 1.5h margin (shaders/mpm_g2p.comp:255-263)
  {
    const float mg = ge.h * 1.5f;
    const float lox = ge.wmin[0] + mg, loy = ge.wmin[1] + mg, loz = ge.wmin[2] + mg;
    const float hix = ge.wmax[0] - mg, hiy = ge.wmax[1] - mg, hiz = ge.wmax[2] - mg;
    if (xn < lox) { xn = lox; vnx = fmaxf(vnx, 0.f); }
    if (xn > hix) { xn = hix; vnx = fminf(vnx, 0.f); }
    if (yn < loy) { yn = loy; vny = fmaxf(vny, 0.f); }
    if (yn > hiy) { yn = hiy; vny = fminf(vny, 0.f); }
    if (zn < loz) { zn = loz; vnz = fmaxf(vnz, 0.f); }
    if (zn > hiz) { zn = hiz; vnz = fminf(vnz, 0.f); }
  }
  ro[R_P] = make_float4(xn, yn, zn, Vp);
  ro[R_V] = make_float4(vnx, vny, vnz, vel.w);
  ro[R_B0] = make_float4(Bn.m[0][0], Bn.m[0][1], Bn.m[0][2], tau.m[0][1]);
  ro[R_B1] = make_float4(Bn.m[1][0], Bn.m[1][1], Bn.m[1][2], tau.m[0][2]);
  ro[R_B2] = make_float4(Bn.m[2][0], Bn.m[2][1], Bn.m[2][2], tau.m[1][2]);
  ro[R_T] = make_float4(tau.m[0][0], tau.m[1][1], tau.m[2][2], Fn.m[0][0]);
  ro[R_FA] = make_float4(Fn.m[0][1], Fn.m[0][2], Fn.m[1][0], Fn.m[1][1]);
  ro[R_FB] = make_float4(Fn.m[1][2], Fn.m[2][0], Fn.m[2][1], Fn.m[2][2]);
  const uint32_t key = cell_key(ge, xn, yn, zn);  // the next substep's bin key, and its count
  keys[q] = key;
  if (tile_cnt != nullptr) rank[q] = count_in_tile(key, tile_cnt);
  // F and tau were set to I and 0: the fallback's entry is dropped
  if (fb_at != kFbNone && (jreset || pushed)) reinterpret_cast<uint32_t*>(p.fb_queue + size_t(fb_at) * kFbEntry)[1] = 0u;
}

// the material of a particle: clamp to materialCount-1 (shaders/mpm_g2p.comp:128-130)
__device__ __forceinline__ uint32_t particle_material(const SubParams& p, const float4 vel) {
  const uint32_t mid = __float_as_uint(vel.w);
  return mid > p.material_count - 1u ? p.material_count - 1u : mid;
}

// G2P of particle q (place k of the G2P order) reading the updated grid from HBM.
template <bool FLIP, bool BATCH>
__device__ __forceinline__ void g2p_one(const SubParams& p, uint32_t k, uint32_t q, const float4* rec_in, float4* rec_out,
                                        uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                        uint32_t* __restrict__ tile_cnt, const nb_material* __restrict__ mats,
                                        const nb_material* s_mats, const float4* __restrict__ grid_node,
                                        const float4* __restrict__ grid_old, const float* __restrict__ sdf) {
  const SceneGeo g = particle_geo<BATCH>(p, q);
  const float4* r = rec_in + size_t(q) * kRec;
  float4* ro = rec_out + size_t(q) * kRec;
  const float4 pp = r[R_P];
  int base[3];
  Axis3 ax3[3];
  const bool tiny = g2p_stencil(g, pp.x, pp.y, pp.z, base, ax3);
  // out-of-grid nodes read a clamped (valid) address and are dropped together
  // with the massless ones
  auto node = [&](int ix, int iy, int iz, float (&v)[3], float (&vo)[3]) -> bool {
    const int nx = base[0] + ix, ny = base[1] + iy, nz = base[2] + iz;
    const uint32_t cx = uint32_t(min(max(nx, 0), g.grid_res[0] - 1));
    const uint32_t cy = uint32_t(min(max(ny, 0), g.grid_res[1] - 1));
    const uint32_t cz = uint32_t(min(max(nz, 0), g.grid_res[2] - 1));
    const uint32_t id = node_id(g, cx, cy, cz);
    const float4 gn = grid_node[id];
    // bitwise, not short-circuit: the load then has a use on every path and
    // stays one unconditional 16-byte load, issued with the slab's others
    const bool live = (uint32_t(nx) < uint32_t(g.grid_res[0])) & (uint32_t(ny) < uint32_t(g.grid_res[1])) &
                      (uint32_t(nz) < uint32_t(g.grid_res[2])) & (gn.w >= 1e-10f);
    v[0] = live ? gn.x : 0.f;
    v[1] = live ? gn.y : 0.f;
    v[2] = live ? gn.z : 0.f;
    if (FLIP) {
      const float4 o = grid_old[id];
      vo[0] = live ? o.x : 0.f;
      vo[1] = live ? o.y : 0.f;
      vo[2] = live ? o.z : 0.f;
    }
    return live;
  };
  G2PGather gth;
  g2p_gather<FLIP>(ax3, tiny, node, gth);
  const float4 vel = r[R_V];
  const uint32_t mid = particle_material(p, vel);
  const nb_material mat = BATCH ? mats[mid] : s_mats[mid];
  g2p_particle<FLIP, BATCH>(p, k, q, r, ro, keys, rank, tile_cnt, mat, gth, pp, vel, sdf);
}

// a plain engine's material table is staged in LDS; a batch's (up to
// kBatchMaxMaterials) is read through the caches
template <bool BATCH>
__device__ __forceinline__ void stage_materials(const SubParams& p, const nb_material* __restrict__ mats,
                                                nb_material* s_mats) {
  if constexpr (!BATCH) {
    float* dst = reinterpret_cast<float*>(s_mats);
    const float* src = reinterpret_cast<const float*>(mats);
    const uint32_t nf = p.material_count * uint32_t(sizeof(nb_material) / 4);
    for (uint32_t e = threadIdx.x; e < nf; e += blockDim.x) dst[e] = src[e];
    __syncthreads();
  }
}

// G2P reading the updated grid from HBM, one thread per particle in bin order.
// rec_out may equal rec_in: every record slot written is data-dependent on the
// load of the same slot (or not read at all), so updating in place is safe.
// 4 waves per SIMD (<= 128 VGPRs): the gather's latency needs the occupancy.
// FLIP gathers a second grid and keeps 168: at 4 waves it spilled 37 registers,
// at 3 none (85,184 particles 29.8 -> 23.5 us; a whole FLIP substep of 4.19 M
// 1029 -> 953 us, of 262,144 132 -> 127).
template <bool FLIP, bool BATCH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(FLIP ? 3 : 4))) void k_g2p(SubParams p,
                                                                                   const float4* rec_in,
                                                                                   float4* rec_out,
                                             uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                             uint32_t* __restrict__ tile_cnt,
                                             const nb_material* __restrict__ mats,
                                             const uint32_t* __restrict__ sorted,
                                             const float4* __restrict__ grid_node,
                                             const float4* __restrict__ grid_old, const float* __restrict__ sdf) {
  __shared__ nb_material s_mats[BATCH ? 1 : NB_MAX_MATERIALS];
  stage_materials<BATCH>(p, mats, s_mats);
  const uint32_t k = xcd_chunk(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (k >= p.n) return;
  const uint32_t q = sorted ? sorted[k] : k;
  g2p_one<FLIP, BATCH>(p, k, q, rec_in, rec_out, keys, rank, tile_cnt, mats, s_mats, grid_node, grid_old, sdf);
}

// The FP64 fallback's second half: for every entry G2P queued (queue_fb),
// the return map and Hencky stress in FP64 from the trial F (mode 1), or the
// Hencky stress of the record's F (mode 2), rounded once; F is replaced and
// the stress added to the record's (the mud viscosity term, or zero).
// Every block reads the slots' lengths and the `blocks` blocks stride over
// their concatenation.  Within a call it runs beside the next substep's
// scatter, which does not touch the records (a launch of its own was 12-19 us
// of latency chain per substep), and the sort after that zeroes the lengths; a
// call's last substep runs it alone
// (k_g2p_fb), then k_g2p_fb_reset.  (A count of finished blocks, the last one
// zeroing, cost tens of ns per block: device-scope atomics on one address
// serialise across the XCDs.)
template <bool BATCH>
__device__ __forceinline__ void fb_entries(const SubParams& p, float4* rec, const nb_material* __restrict__ mats,
                                           uint32_t block, uint32_t blocks) {
  __shared__ nb_material s_mats[BATCH ? 1 : NB_MAX_MATERIALS];
  stage_materials<BATCH>(p, mats, s_mats);
  // the slots' lengths and their exclusive prefix (wave 0), so that the
  // grid's threads share the queue's entries evenly whatever the slots hold
  __shared__ uint32_t s_pre[kFbSlots + 1];
  if (threadIdx.x < 64u) {
    const uint32_t len = threadIdx.x < kFbSlots ? p.fb_ctl[threadIdx.x * kFbCtlStride] : 0u;
    uint32_t inc = len;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = uint32_t(__shfl_up(int(inc), d));
      if (threadIdx.x >= uint32_t(d)) inc += o;
    }
    if (threadIdx.x < kFbSlots) s_pre[threadIdx.x] = inc - len;
    if (threadIdx.x == kFbSlots - 1u) s_pre[kFbSlots] = inc;
  }
  __syncthreads();
  const uint32_t total = s_pre[kFbSlots];
  const bool cs = p.corrected_svd != 0u;
  // consecutive waves of entries go to different blocks, so that a short queue
  // is spread over the CUs (its FP64 chains are latency: 1,400 entries in two
  // blocks of 1024 took 28 us, spread 14)
  const uint32_t wave_of = (threadIdx.x >> 6) * blocks + block;
  for (uint32_t i = wave_of * 64u + (threadIdx.x & 63u); i < total; i += blocks * blockDim.x) {
    // the slot holding entry i of the concatenated queue: the last s with s_pre[s] <= i
    uint32_t slot = 0u;
#pragma unroll
    for (uint32_t step = kFbSlots / 2u; step > 0u; step >>= 1)
      if (s_pre[slot + step] <= i) slot += step;
    const float4* e = p.fb_queue + (size_t(slot) * p.fb_region + (i - s_pre[slot])) * kFbEntry;
    const float4 e0 = e[0];
    const uint32_t q = __float_as_uint(e0.x), mode = __float_as_uint(e0.y);
    if (mode == 0u) continue;
    float4* ro = rec + size_t(q) * kRec;
    const uint32_t mid = particle_material(p, ro[R_V]);
    const nb_material mat = BATCH ? mats[mid] : s_mats[mid];
    const bool dp = true;  // only the Drucker-Prager family is queued
    const float4 rt = ro[R_T];
    float* b0 = reinterpret_cast<float*>(ro + R_B0);
    float* b1 = reinterpret_cast<float*>(ro + R_B1);
    float* b2 = reinterpret_cast<float*>(ro + R_B2);
    m3 F, tau;
    if (mode == 1u) {
      const float4 e1 = e[1], e2 = e[2], e3 = e[3], e4 = e[4];
      m3 Fo, L;
      Fo.m[0][0] = e0.z; Fo.m[0][1] = e0.w; Fo.m[0][2] = e1.x;
      Fo.m[1][0] = e1.y; Fo.m[1][1] = e1.z; Fo.m[1][2] = e1.w;
      Fo.m[2][0] = e2.x; Fo.m[2][1] = e2.y; Fo.m[2][2] = e2.z;
      const float vg[9] = {e2.w, e3.x, e3.y, e3.z, e3.w, e4.x, e4.y, e4.z, e4.w};
#pragma unroll
      for (int c = 0; c < 3; c++)
#pragma unroll
        for (int rr = 0; rr < 3; rr++) L.m[c][rr] = (c == rr ? 1.f : 0.f) + p.dt * vg[c * 3 + rr];
      const FTau ft = plastic_fp64(m3_mul(L, Fo), dp, mat.mu, mat.lambda, mat.q_max, mat.M_friction,
                                   mat.q_cohesion, cs);
      F = ft.F;
      tau = ft.tau;
    } else {
      const float4 fa = ro[R_FA], fb = ro[R_FB];
      F.m[0][0] = rt.w; F.m[0][1] = fa.x; F.m[0][2] = fa.y;
      F.m[1][0] = fa.z; F.m[1][1] = fa.w; F.m[1][2] = fb.x;
      F.m[2][0] = fb.y; F.m[2][1] = fb.z; F.m[2][2] = fb.w;
      tau = m3_round(hencky_stress(m3_convert<double>(F), double(mat.mu), double(mat.lambda), cs));
    }
    // the record's stress: the viscosity term G2P left there
    ro[R_T] = make_float4(tau.m[0][0] + rt.x, tau.m[1][1] + rt.y, tau.m[2][2] + rt.z, F.m[0][0]);
    b0[3] = tau.m[0][1] + b0[3];
    b1[3] = tau.m[0][2] + b1[3];
    b2[3] = tau.m[1][2] + b2[3];
    if (mode == 1u) {
      ro[R_FA] = make_float4(F.m[0][1], F.m[0][2], F.m[1][0], F.m[1][1]);
      ro[R_FB] = make_float4(F.m[1][2], F.m[2][0], F.m[2][1], F.m[2][2]);
    }
  }
}

template <bool BATCH>
__global__ __launch_bounds__(256) void k_g2p_fb(SubParams p, float4* rec, const nb_material* __restrict__ mats) {
  fb_entries<BATCH>(p, rec, mats, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(64) void k_g2p_fb_reset(uint32_t* __restrict__ fb_ctl) {
  if (threadIdx.x < kFbSlots) fb_ctl[threadIdx.x * kFbCtlStride] = 0u;
}

// ---------------------------------------------------------------------------
// the bin's tile pass and scatter (after the fallback, which runs beside them)
// ---------------------------------------------------------------------------
// Every particle and its cell into its tile's range, at its place of the count.
// The launch's first fb_blocks blocks work off the FP64 fallback's queue of the
// G2P before (they are the longer ones); the sort empties it.
template <bool PACKED, bool BATCH>
__global__ __launch_bounds__(256) void k_bin_scatter_fb(SubParams p, float4* rec, const nb_material* __restrict__ mats,
                                                        const uint32_t* __restrict__ keys,
                                                        const uint32_t* __restrict__ rank,
                                                        const int32_t* __restrict__ tile_act,
                                                        const uint32_t* __restrict__ tile_start,
                                                        uint2* __restrict__ bucket, uint32_t fb_blocks) {
  if (blockIdx.x < fb_blocks) fb_entries<BATCH>(p, rec, mats, blockIdx.x, fb_blocks);
  else scatter_one<PACKED>(p.n, (blockIdx.x - fb_blocks) * blockDim.x + threadIdx.x, keys, rank, tile_act, tile_start, bucket);
}
template <bool PACKED>
__global__ __launch_bounds__(256) void k_bin_scatter(uint32_t n, const uint32_t* __restrict__ keys,
                                                     const uint32_t* __restrict__ rank,
                                                     const int32_t* __restrict__ tile_act,
                                                     const uint32_t* __restrict__ tile_start,
                                                     uint2* __restrict__ bucket) {
  scatter_one<PACKED>(n, blockIdx.x * blockDim.x + threadIdx.x, keys, rank, tile_act, tile_start, bucket);
}

// P2G's order of the tiles: four classes by particle count, largest first,
// tile order within a class.  A block's work grows with its tile's particles,
// so the long tiles start first and the short ones fill the end of the launch.
// Which block takes which tile does not change any result.
__device__ __forceinline__ uint32_t tile_class(uint32_t t) {
  return t >= 2048u ? 0u : (t >= 1024u ? 1u : (t >= 512u ? 2u : 3u));
}
__device__ __forceinline__ uint32_t tile_units(uint32_t t) { return (t + kG2PUnit - 1u) / kG2PUnit; }

// Cubes of up to kSmallTiles tiles (128^3 cells): one block does the whole
// pass in one launch.  Thread t holds the tiles [t C, (t + 1) C).  Per tile:
// occupied; node tile (a tile of its 3x3x3 neighbourhood is occupied: its nodes
// can receive mass), found axis by axis in LDS (27 reads a tile at once took
// 25 us for 4,096 tiles, all on one CU).  4.6 us for 64 tiles, 5.7 for 512, 10.4
// for 4,096, where the two launches below take 5.8 + 6.0; they spread larger
// cubes over the chip.
constexpr uint32_t kSmallTiles = 4096;
template <bool BATCH>
__global__ __launch_bounds__(1024) void k_bin_tiles(SubParams p, uint32_t* __restrict__ tile_cnt,
                                                    int32_t* __restrict__ tile_act,
                                                    uint32_t* __restrict__ act_tiles,
                                                    uint32_t* __restrict__ node_tiles,
                                                    uint32_t* __restrict__ tile_total,
                                                    uint32_t* __restrict__ tile_start,
                                                    uint32_t* __restrict__ tile_order,
                                                    uint32_t* __restrict__ counters, uint2* __restrict__ units,
                                                    uint32_t nt) {
  constexpr uint32_t C = kSmallTiles / 1024u;
  __shared__ uint8_t s_occ[2][kSmallTiles];
  __shared__ uint64_t s_scan[3 * (1024 / 64 + 1)];
  const uint32_t c = (nt + 1023u) / 1024u, t0 = threadIdx.x * c;
  uint32_t cnt[C];
  int at3[C][3], td[C];
  SceneGeo g;
#pragma unroll
  for (uint32_t k = 0; k < C; k++) {
    const uint32_t T = t0 + k;
    cnt[k] = 0u;
    if (k < c && T < nt) {
      cnt[k] = tile_cnt[tile_slot(T)];
      g = tile_geo<BATCH>(p, T);  // neighbours stay inside the tile's scene
      tile_coords(g, T, at3[k][0], at3[k][1], at3[k][2]);
      td[k] = int(g.tile_dim);
      s_occ[0][T] = cnt[k] ? 1 : 0;
      if (cnt[k]) tile_cnt[tile_slot(T)] = 0u;  // ready for the next count
    }
  }
  // occupied in the 3x3x3 neighbourhood, axis by axis
  uint32_t node = 0;  // bit k: tile t0 + k is a node tile
#pragma unroll
  for (int axis = 0; axis < 3; axis++) {
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < C; k++) {
      const uint32_t T = t0 + k;
      if (k < c && T < nt) {
        const SceneGeo gk = BATCH ? tile_geo<BATCH>(p, T) : g;
        uint32_t any = s_occ[axis & 1][T];
#pragma unroll
        for (int d = -1; d <= 1; d += 2) {
          const int v = at3[k][axis] + d;
          const bool in = uint32_t(v) < uint32_t(td[k]);
          const int w = in ? v : at3[k][axis];
          any |= s_occ[axis & 1][tile_id(gk, axis == 0 ? w : at3[k][0], axis == 1 ? w : at3[k][1], axis == 2 ? w : at3[k][2])];
        }
        s_occ[1 - (axis & 1)][T] = uint8_t(any);
        if (axis == 2 && any) node |= 1u << k;
      }
    }
  }
  uint64_t lists = 0, places = 0, classes = 0;
#pragma unroll
  for (uint32_t k = 0; k < C; k++) {
    lists += uint64_t(cnt[k] ? 1u : 0u) | (uint64_t((node >> k) & 1u) << 32);
    places += uint64_t(cnt[k]) | (uint64_t(tile_units(cnt[k])) << 32);
    if (cnt[k]) classes += uint64_t(1) << (16u * tile_class(cnt[k]));
  }
  const uint64_t own[3] = {lists, places, classes};
  uint64_t pre3[3], tot3[3];
  block_exclusive_scan3<1024>(own, s_scan, pre3, tot3);
  const uint64_t l0 = pre3[0], p0 = pre3[1], c0 = pre3[2];
  const uint64_t n_lists = tot3[0], n_places = tot3[1], n_classes = tot3[2];
  uint32_t oa = uint32_t(l0), on = uint32_t(l0 >> 32), os = uint32_t(p0), ou = uint32_t(p0 >> 32);
  uint32_t at[4], before = 0;
#pragma unroll
  for (uint32_t q = 0; q < 4u; q++) {
    at[q] = before + (uint32_t(c0 >> (16u * q)) & 0xFFFFu);
    before += uint32_t(n_classes >> (16u * q)) & 0xFFFFu;
  }
#pragma unroll
  for (uint32_t k = 0; k < C; k++) {
    const uint32_t T = t0 + k;
    if (!(k < c && T < nt)) continue;
    tile_act[T] = cnt[k] ? int32_t(oa) : -1;
    if (cnt[k]) {
      act_tiles[oa] = T;
      tile_total[oa] = cnt[k];
      tile_start[oa] = os;
      for (uint32_t u = 0, nu = tile_units(cnt[k]); u < nu; u++) units[ou++] = make_uint2(oa, u);
      const uint32_t q = tile_class(cnt[k]);
      tile_order[q == 0u ? at[0]++ : (q == 1u ? at[1]++ : (q == 2u ? at[2]++ : at[3]++))] = oa;
      os += cnt[k];
      oa++;
    }
    if ((node >> k) & 1u) node_tiles[on++] = T;
  }
  if (threadIdx.x == 0u) {
    counters[CNT_ACTIVE] = uint32_t(n_lists);
    counters[CNT_NODE_TILES] = uint32_t(n_lists >> 32);
    counters[CNT_UNITS] = uint32_t(n_places >> 32);
  }
}

// Larger cubes: 256 tiles a block in two launches.  k_bin_mark: each tile's
// marks (bit 0 occupied, bit 1 node tile) and its block's sums; the blocks after
// the first `tile_blocks` work off the fallback's queue.
template <bool BATCH>
__global__ __launch_bounds__(256) void k_bin_mark(SubParams p, float4* rec, const nb_material* __restrict__ mats,
                                                  const uint32_t* __restrict__ tile_cnt,
                                                  uint8_t* __restrict__ tile_mark, TileSums* __restrict__ sums,
                                                  uint32_t nt, uint32_t tile_blocks) {
  if (blockIdx.x >= tile_blocks) {
    fb_entries<BATCH>(p, rec, mats, blockIdx.x - tile_blocks, gridDim.x - tile_blocks);
    return;
  }
  __shared__ uint64_t s_scan[3 * (256 / 64 + 1)];
  const uint32_t T = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t m = 0, cnt = 0;
  if (T < nt) {
    const SceneGeo g = tile_geo<BATCH>(p, T);
    int tx, ty, tz;
    tile_coords(g, T, tx, ty, tz);
    const int td = int(g.tile_dim);
    cnt = tile_cnt[tile_slot(T)];
    uint32_t any = 0;
#pragma unroll
    for (int o = 0; o < 27; o++) {  // all loads in flight together
      const int x = tx + o % 3 - 1, y = ty + (o / 3) % 3 - 1, z = tz + o / 9 - 1;
      const bool in = uint32_t(x) < uint32_t(td) && uint32_t(y) < uint32_t(td) && uint32_t(z) < uint32_t(td);
      any |= in ? tile_cnt[tile_slot(tile_id(g, in ? x : tx, in ? y : ty, in ? z : tz))] : 0u;
    }
    m = (cnt ? 1u : 0u) | (any ? 2u : 0u);
    tile_mark[T] = uint8_t(m);
  }
  const uint64_t own[3] = {uint64_t(m & 1u) | (uint64_t(m >> 1) << 32), uint64_t(cnt) | (uint64_t(tile_units(cnt)) << 32),
                           cnt ? uint64_t(1) << (16u * tile_class(cnt)) : uint64_t(0)};
  uint64_t pre3[3], tot3[3];
  block_exclusive_scan3<256>(own, s_scan, pre3, tot3);
  if (threadIdx.x == 0u) {
    TileSums t;
    t.lists = tot3[0];
    t.places = tot3[1];
#pragma unroll
    for (uint32_t q = 0; q < 4u; q++) t.cls[q] = uint32_t(tot3[2] >> (16u * q)) & 0xFFFFu;
    sums[blockIdx.x] = t;
  }
}

// Beyond kSumBlocks blocks: their sums scanned in place by one block, the
// total behind the last (a block of k_bin_compact otherwise adds up those
// before it, and all of them, by itself).
constexpr uint32_t kSumBlocks = 1024;
__global__ __launch_bounds__(1024) void k_bin_sums(TileSums* __restrict__ sums, uint32_t nb) {
  __shared__ uint64_t s_scan[1024 / 64 + 1];
  const uint32_t per = (nb + 1023u) / 1024u, lo = min(nb, threadIdx.x * per), hi = min(nb, lo + per);
  TileSums t{};
  for (uint32_t i = lo; i < hi; i++) {
    t.lists += sums[i].lists;
    t.places += sums[i].places;
    for (int q = 0; q < 4; q++) t.cls[q] += sums[i].cls[q];
  }
  TileSums run, tot;
  run.lists = block_exclusive_scan<1024>(t.lists, s_scan, tot.lists);
  run.places = block_exclusive_scan<1024>(t.places, s_scan, tot.places);
  uint64_t c01, c23;
  const uint64_t a = block_exclusive_scan<1024>(uint64_t(t.cls[0]) | (uint64_t(t.cls[1]) << 32), s_scan, c01);
  const uint64_t b = block_exclusive_scan<1024>(uint64_t(t.cls[2]) | (uint64_t(t.cls[3]) << 32), s_scan, c23);
  run.cls[0] = uint32_t(a); run.cls[1] = uint32_t(a >> 32); run.cls[2] = uint32_t(b); run.cls[3] = uint32_t(b >> 32);
  tot.cls[0] = uint32_t(c01); tot.cls[1] = uint32_t(c01 >> 32); tot.cls[2] = uint32_t(c23); tot.cls[3] = uint32_t(c23 >> 32);
  for (uint32_t i = lo; i < hi; i++) {
    const TileSums x = sums[i];
    sums[i] = run;
    run.lists += x.lists;
    run.places += x.places;
    for (int q = 0; q < 4; q++) run.cls[q] += x.cls[q];
  }
  if (threadIdx.x == 0u) sums[nb] = tot;
}

template <bool SCANNED>
__global__ __launch_bounds__(256) void k_bin_compact(const uint8_t* __restrict__ tile_mark,
                                                     const TileSums* __restrict__ sums,
                                                     uint32_t* __restrict__ tile_cnt, int32_t* __restrict__ tile_act,
                                                     uint32_t* __restrict__ act_tiles,
                                                     uint32_t* __restrict__ node_tiles,
                                                     uint32_t* __restrict__ tile_total,
                                                     uint32_t* __restrict__ tile_start,
                                                     uint32_t* __restrict__ tile_order,
                                                     uint32_t* __restrict__ counters, uint2* __restrict__ units,
                                                     uint32_t nt) {
  __shared__ uint64_t s_scan[3 * (256 / 64 + 1)];
  __shared__ uint64_t s_sum[256 / 64][8];
  TileSums pre, tot;
  if (SCANNED) {
    pre = sums[blockIdx.x];
    tot = sums[gridDim.x];
  } else {
    uint64_t v[8] = {};  // lists, places, two pairs of classes: of the blocks before this one, and of all
    for (uint32_t i = threadIdx.x; i < gridDim.x; i += blockDim.x) {
      const TileSums x = sums[i];
      const uint64_t w[4] = {x.lists, x.places, uint64_t(x.cls[0]) | (uint64_t(x.cls[1]) << 32),
                             uint64_t(x.cls[2]) | (uint64_t(x.cls[3]) << 32)};
      const bool before = i < blockIdx.x;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        v[q] += before ? w[q] : 0u;
        v[4 + q] += w[q];
      }
    }
#pragma unroll
    for (int q = 0; q < 8; q++) {
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) v[q] += __shfl_xor(v[q], d);
      if ((threadIdx.x & 63u) == 0u) s_sum[threadIdx.x >> 6][q] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 8; q++) v[q] = (s_sum[0][q] + s_sum[1][q]) + (s_sum[2][q] + s_sum[3][q]);
    pre.lists = v[0];
    pre.places = v[1];
    pre.cls[0] = uint32_t(v[2]); pre.cls[1] = uint32_t(v[2] >> 32); pre.cls[2] = uint32_t(v[3]); pre.cls[3] = uint32_t(v[3] >> 32);
    tot.lists = v[4];
    tot.places = v[5];
    tot.cls[0] = uint32_t(v[6]); tot.cls[1] = uint32_t(v[6] >> 32); tot.cls[2] = uint32_t(v[7]); tot.cls[3] = uint32_t(v[7] >> 32);
  }
  const uint32_t T = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t m = T < nt ? tile_mark[T] : 0u, cnt = (m & 1u) ? tile_cnt[tile_slot(T)] : 0u;
  const uint32_t q = tile_class(cnt);
  const uint64_t own[3] = {uint64_t(m & 1u) | (uint64_t(m >> 1) << 32), uint64_t(cnt) | (uint64_t(tile_units(cnt)) << 32),
                           cnt ? uint64_t(1) << (16u * q) : uint64_t(0)};
  uint64_t pre3[3], tot3[3];
  block_exclusive_scan3<256>(own, s_scan, pre3, tot3);
  const uint64_t l0 = pre.lists + pre3[0], p0 = pre.places + pre3[1], c0 = pre3[2];
  if (T < nt) {
    const uint32_t oa = uint32_t(l0);
    tile_act[T] = cnt ? int32_t(oa) : -1;
    if (cnt) {
      act_tiles[oa] = T;
      tile_total[oa] = cnt;
      tile_start[oa] = uint32_t(p0);
      for (uint32_t u = 0, nu = tile_units(cnt); u < nu; u++) units[uint32_t(p0 >> 32) + u] = make_uint2(oa, u);
      uint32_t at = uint32_t(c0 >> (16u * q)) & 0xFFFFu;
#pragma unroll
      for (uint32_t k = 0; k < 4u; k++) at += k < q ? tot.cls[k] : (k == q ? pre.cls[k] : 0u);
      tile_order[at] = oa;
      tile_cnt[tile_slot(T)] = 0u;  // ready for the next count
    }
    if (m & 2u) node_tiles[uint32_t(l0 >> 32)] = T;
  }
  if (blockIdx.x == 0u && threadIdx.x == 0u) {
    counters[CNT_ACTIVE] = uint32_t(tot.lists);
    counters[CNT_NODE_TILES] = uint32_t(tot.lists >> 32);
    counters[CNT_UNITS] = uint32_t(tot.places >> 32);
  }
}

// Grid update and G2P fused, one block per work unit: a unit is up to
// kG2PUnit particles of one occupied tile (a tile's particles are one
// contiguous range of the bin order; the bin's tile pass lists the units).
// The block builds the tile's 10^3 node box in LDS from the partials (the
// same sums and node update as k_grid_tiles, bit for bit), stores each node's
// G2P view (velocity, or zero for a node that does not take part, and FLIP's
// saved velocity), then runs G2P for the unit's particles gathering from
// LDS.  A particle whose stencil leaves the box (its position lies outside
// the grid) reads the box with a range check: the nodes outside it are
// outside the grid too.  Results equal k_grid_tiles + k_g2p bit for bit; the
// grid itself is not written (the last substep of a call runs unfused, so the
// exported grid stays that of the last substep).
template <bool FLIP, bool BATCH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_g2p_tile(
    SubParams p, const float4* rec_in, float4* rec_out, uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
    uint32_t* __restrict__ tile_cnt,
    const nb_material* __restrict__ mats, const uint32_t* __restrict__ sorted, const uint2* __restrict__ units,
    const uint32_t* __restrict__ act_tiles, const uint32_t* __restrict__ tile_start,
    const uint32_t* __restrict__ tile_total, const uint32_t* __restrict__ counters,
    const int32_t* __restrict__ tile_act, const float4* __restrict__ partial, const float* __restrict__ sdf,
    const nb_collider* __restrict__ cols, const nb_force* __restrict__ forces) {
  __shared__ float4 s_v[kBoxNodes];                 // xyz: velocity (0 when not taking part), w: 1 / 0
  __shared__ float4 s_o[FLIP ? kBoxNodes : 1];      // FLIP's saved velocity
  __shared__ nb_material s_mats[BATCH ? 1 : NB_MAX_MATERIALS];
  if constexpr (!BATCH) {
    float* dst = reinterpret_cast<float*>(s_mats);
    const float* src = reinterpret_cast<const float*>(mats);
    const uint32_t nf = p.material_count * uint32_t(sizeof(nb_material) / 4);
    for (uint32_t e = threadIdx.x; e < nf; e += blockDim.x) dst[e] = src[e];
  }
  const uint32_t n_units = counters[CNT_UNITS];
  for (uint32_t u = blockIdx.x; u < n_units; u += gridDim.x) {
    const uint2 unit = units[u];
    const uint32_t a = unit.x, chunk = unit.y;
    const uint32_t T = act_tiles[a];
    const SceneGeo g = tile_geo<BATCH>(p, T);
    int tx, ty, tz;
    tile_coords(g, T, tx, ty, tz);
    __syncthreads();  // the previous unit's particles are done with the box
    for (uint32_t e = threadIdx.x; e < kBoxNodes; e += blockDim.x) {
      const int bx = int(e % kBox), by = int((e / kBox) % kBox), bz = int(e / (kBox * kBox));
      const int nx = tx * 8 - 1 + bx, ny = ty * 8 - 1 + by, nz = tz * 8 - 1 + bz;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f), o = make_float4(0.f, 0.f, 0.f, 0.f);
      if (nx >= 0 && nx < g.grid_res[0] && ny >= 0 && ny < g.grid_res[1] && nz >= 0 && nz < g.grid_res[2]) {
        // the node's own tile and its place in it, as the grid update sees the node
        const int ntx = nx >> 3, nty = ny >> 3, ntz = nz >> 3;
        float mx, my, mz, mass;
        (void)sum_partials(g, ntx, nty, ntz, nx & 7, ny & 7, nz & 7, tile_act, partial, mx, my, mz, mass);
        if (mass >= 1e-10f) {
          float vx = mx / mass, vy = my / mass, vz = mz / mass, ox, oy, oz;
          node_update(p, g, nx, ny, nz, vx, vy, vz, ox, oy, oz, sdf, cols, forces);
          v = make_float4(vx, vy, vz, 1.f);
          o = make_float4(ox, oy, oz, 0.f);
        }
      }
      s_v[e] = v;
      if (FLIP) s_o[e] = o;
    }
    __syncthreads();
    const uint32_t first = tile_start[a] + chunk * kG2PUnit;
    const uint32_t last = min(tile_start[a] + tile_total[a], first + kG2PUnit);
    // box node of grid node n along each axis: n - (8 t - 1)
    const int ox0 = tx * 8 - 1, oy0 = ty * 8 - 1, oz0 = tz * 8 - 1;
    for (uint32_t k = first + threadIdx.x; k < last; k += blockDim.x) {
      const uint32_t q = sorted[k];
      const float4* r = rec_in + size_t(q) * kRec;
      float4* ro = rec_out + size_t(q) * kRec;
      const float4 pp = r[R_P];
      int base[3];
      Axis3 ax3[3];
      const bool tiny = g2p_stencil(g, pp.x, pp.y, pp.z, base, ax3);
      const int bx0 = base[0] - ox0, by0 = base[1] - oy0, bz0 = base[2] - oz0;
      const bool inbox = bx0 >= 0 && bx0 <= kBox - 3 && by0 >= 0 && by0 <= kBox - 3 && bz0 >= 0 && bz0 <= kBox - 3;
      const int e0 = (bz0 * kBox + by0) * kBox + bx0;
      G2PGather gth;
      if (inbox) {
        auto node = [&](int ix, int iy, int iz, float (&v)[3], float (&vo)[3]) -> bool {
          const int e = e0 + (iz * kBox + iy) * kBox + ix;
          const float4 n4 = s_v[e];
          v[0] = n4.x; v[1] = n4.y; v[2] = n4.z;
          if (FLIP) {
            const float4 o4 = s_o[e];
            vo[0] = o4.x; vo[1] = o4.y; vo[2] = o4.z;
          }
          return n4.w != 0.f;
        };
        g2p_gather<FLIP>(ax3, tiny, node, gth);
      } else {
        auto node = [&](int ix, int iy, int iz, float (&v)[3], float (&vo)[3]) -> bool {
          const int bx = bx0 + ix, by = by0 + iy, bz = bz0 + iz;
          const bool in = bx >= 0 && bx < kBox && by >= 0 && by < kBox && bz >= 0 && bz < kBox;
          const int e = in ? (bz * kBox + by) * kBox + bx : 0;
          const float4 n4 = s_v[e];
          const bool live = in && n4.w != 0.f;
          v[0] = live ? n4.x : 0.f; v[1] = live ? n4.y : 0.f; v[2] = live ? n4.z : 0.f;
          if (FLIP) {
            const float4 o4 = s_o[e];
            vo[0] = live ? o4.x : 0.f; vo[1] = live ? o4.y : 0.f; vo[2] = live ? o4.z : 0.f;
          }
          return live;
        };
        g2p_gather<FLIP>(ax3, tiny, node, gth);
      }
      const float4 vel = r[R_V];
      const uint32_t mid = particle_material(p, vel);
      const nb_material mat = BATCH ? mats[mid] : s_mats[mid];
      g2p_particle<FLIP, BATCH>(p, k, q, r, ro, keys, rank, tile_cnt, mat, gth, pp, vel, sdf);
    }
  }
}

// ---------------------------------------------------------------------------
// utilities
// ---------------------------------------------------------------------------
__global__ void k_sdf_sphere(float* __restrict__ sdf, SubParams p, float r, float cx, float cy, float cz) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t nc = p.cube_res * p.cube_res * p.cube_res;
  if (c >= nc) return;
  const int x = int(morton_compact(c)), y = int(morton_compact(c >> 1)), z = int(morton_compact(c >> 2));
  if (x >= p.grid_res[0] || y >= p.grid_res[1] || z >= p.grid_res[2]) {
    sdf[c] = 0.f;  // cells outside gridRes stay unwritten (zero) as in the reference's host loop
    return;
  }
  // src/engine/MPMEngine.cpp:186-193 (cell centres from the origin)
  const float wx = (float(x) + 0.5f) * p.h, wy = (float(y) + 0.5f) * p.h, wz = (float(z) + 0.5f) * p.h;
  const float d = sqrtf((wx - cx) * (wx - cx) + (wy - cy) * (wy - cy) + (wz - cz) * (wz - cz));
  sdf[c] = d - r;
}

// rows of 0, 1, ..., n - 1
__global__ void k_fill_identity(uint32_t* __restrict__ a, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[size_t(blockIdx.y) * n + i] = i;
}

// F = I, B = 0, tau = 0 for rows [first, first+count) (appendParticles)
__global__ void k_init_FB(float4* F0, float4* F1, float4* F2, float4* B0, float4* B1, float4* B2, uint32_t first,
                          uint32_t count) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const uint32_t q = first + i;
  F0[q] = make_float4(1.f, 0.f, 0.f, 0.f);
  F1[q] = make_float4(0.f, 1.f, 0.f, 0.f);
  F2[q] = make_float4(0.f, 0.f, 1.f, 0.f);
  B0[q] = make_float4(0.f, 0.f, 0.f, 0.f);
  B1[q] = make_float4(0.f, 0.f, 0.f, 0.f);
  B2[q] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// reference layout (eight float4 arrays) <-> one 128-byte record per particle
// Bound by memory.  A lane storing its particle's record would write 64 lines of 16
// bytes an instruction (349 us for 4.19 M particles, 3.1 TB/s); the wave's 64
// records go through LDS instead (slots rotated by the particle, so that neither
// side meets in a bank) and leave as whole kilobytes.  COUNT: the keys and tile
// counts of the bin, for which k_bin_keys would read the records again (126 us):
// both together take 207 us.
template <bool COUNT, bool BATCH>
__global__ __launch_bounds__(256) void k_soa_to_aos(SubParams p, FieldPtrs f, float4* __restrict__ rec, uint32_t n,
                                                    uint32_t* __restrict__ keys, uint32_t* __restrict__ rank,
                                                    uint32_t* __restrict__ tile_cnt) {
  __shared__ float4 s_rec[256 * kRec];
  const uint32_t lane = threadIdx.x & 63u, first = blockIdx.x * blockDim.x + (threadIdx.x & ~63u), i = first + lane;
  float4* s = s_rec + (threadIdx.x & ~63u) * kRec;
  if (i < n) {
    const float4 x = f.f[NB_FIELD_P][i];
    const float4 F0 = f.f[NB_FIELD_F0][i], F1 = f.f[NB_FIELD_F1][i], F2 = f.f[NB_FIELD_F2][i];
    auto put = [&](uint32_t slot, const float4 v) { s[lane * kRec + ((slot + lane) & (kRec - 1u))] = v; };
    put(R_P, x);
    put(R_V, f.f[NB_FIELD_V][i]);
    put(R_B0, f.f[NB_FIELD_B0][i]);
    put(R_B1, f.f[NB_FIELD_B1][i]);
    put(R_B2, f.f[NB_FIELD_B2][i]);
    put(R_T, make_float4(F0.w, F1.w, F2.w, F0.x));
    put(R_FA, make_float4(F0.y, F0.z, F1.x, F1.y));
    put(R_FB, make_float4(F1.z, F2.x, F2.y, F2.z));
    if (COUNT) {
      const uint32_t key = cell_key(particle_geo<BATCH>(p, i), x.x, x.y, x.z);
      keys[i] = key;
      rank[i] = count_in_tile(key, tile_cnt);
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < uint32_t(kRec); k++) {
    const uint32_t e = k * 64u + lane, r = e / kRec;
    if (first + r < n) rec[size_t(first) * kRec + e] = s[r * kRec + ((e + r) & (kRec - 1u))];
  }
}
static_assert(kRec == 8, "a record's slots rotate within eight");
__global__ __launch_bounds__(256) void k_aos_to_soa(const float4* __restrict__ rec, FieldPtrs f, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4* r = rec + size_t(i) * kRec;
  const float4 t = r[R_T], a = r[R_FA], b = r[R_FB];
  f.f[NB_FIELD_P][i] = r[R_P];
  f.f[NB_FIELD_V][i] = r[R_V];
  f.f[NB_FIELD_B0][i] = r[R_B0];
  f.f[NB_FIELD_B1][i] = r[R_B1];
  f.f[NB_FIELD_B2][i] = r[R_B2];
  f.f[NB_FIELD_F0][i] = make_float4(t.w, a.x, a.y, t.x);
  f.f[NB_FIELD_F1][i] = make_float4(a.z, a.w, b.x, t.y);
  f.f[NB_FIELD_F2][i] = make_float4(b.y, b.z, b.w, t.z);
}

// plain streaming copy (HBM byte-counter calibration)
__global__ __launch_bounds__(256) void k_copy(float4* __restrict__ dst, const float4* __restrict__ src, uint64_t n4) {
  for (uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += uint64_t(gridDim.x) * blockDim.x)
    dst[i] = src[i];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline uint32_t cdiv(uint32_t a, uint32_t b) { return (a + b - 1) / b; }
// blocks for a tile-stride kernel: never more than tiles, at most the tuned cap
static inline uint32_t tile_grid(uint32_t n_tiles, uint32_t cap) {
  const uint32_t c = cap ? cap : 2048u;
  return n_tiles < c ? (n_tiles ? n_tiles : 1u) : c;
}

struct ProfScope {
  Prof* pf;
  int id;
  hipStream_t s;
  ProfScope(Prof* pf_, int id_, hipStream_t s_) : pf(pf_), id(id_), s(s_) {
    if (pf) (void)hipEventRecord(pf->ev[2 * id], s);
  }
  ~ProfScope() {
    if (pf) {
      (void)hipEventRecord(pf->ev[2 * id + 1], s);
      pf->record(id);
    }
  }
};

// blocks of `threads` for the fallback's queue: at most one thread per
// particle, and enough for a queue of a million entries to have a thread each
// (a block past the queue's end only reads the 64 lengths)
static inline uint32_t fb_blocks(const SubParams& p, uint32_t threads) {
  return p.svd_fp64 ? std::min(cdiv(p.n, threads), (1u << 20) / threads) : 0u;
}

// the fallback's queue in a launch of its own
static void launch_fb_entries(const DevState& d, const SubParams& p, float4* rec, hipStream_t s) {
  const uint32_t g = fb_blocks(p, 256);
  if (!g) return;
  if (p.n_scenes > 0)
    k_g2p_fb<true><<<g, 256, 0, s>>>(p, rec, d.materials);
  else
    k_g2p_fb<false><<<g, 256, 0, s>>>(p, rec, d.materials);
}

void launch_clear_counts(const DevState& d, uint32_t n_tiles, hipStream_t s) {
  k_zero<<<cdiv(tile_slots(n_tiles), 256), 256, 0, s>>>(d.tile_cnt, tile_slots(n_tiles));
}

void launch_bin(const DevState& d, const SubParams& p, uint32_t n_tiles, BinFrom from, hipStream_t s, Prof* pf) {
  const uint32_t tg = tile_grid(n_tiles, p.tile_blocks);
  const bool batch = p.n_scenes > 0;
  // The fallback's queue of the G2P before.  Large cubes: beside k_bin_mark.  Small
  // ones: beside the scatter, while that is short (262,144 particles: 14.7 us together,
  // 5 + 14 apart); beyond 2^20 particles its registers would slow the scatter (4.19 M:
  // 39 against 20 + 16).  By itself when timed, to be booked under its own name.
  const bool small = n_tiles <= kSmallTiles, apart = pf != nullptr || (small && p.n > (1u << 20));
  if (apart && p.svd_fp64) {
    ProfScope ps(pf, 9, s);
    launch_fb_entries(d, p, d.rec, s);
  }
  if (from != BinFrom::COUNTED) {
    ProfScope ps(pf, 0, s);
    const uint32_t nb = cdiv(p.n, 256);
    if (from == BinFrom::KEYS)
      k_bin_keys<false, false><<<nb, 256, 0, s>>>(p, d.rec, d.keys, d.rank, d.tile_cnt);
    else if (batch)
      k_bin_keys<true, true><<<nb, 256, 0, s>>>(p, d.rec, d.keys, d.rank, d.tile_cnt);
    else
      k_bin_keys<true, false><<<nb, 256, 0, s>>>(p, d.rec, d.keys, d.rank, d.tile_cnt);
  }
  {
    ProfScope ps(pf, 1, s);
    if (small) {
#define NB_TILES(BT)                                                                                             \
  k_bin_tiles<BT><<<1, 1024, 0, s>>>(p, d.tile_cnt, d.tile_act, d.act_tiles, d.node_tiles, d.tile_total,         \
                                     d.tile_start, d.tile_order, d.counters, d.units, n_tiles)
      if (batch) NB_TILES(true); else NB_TILES(false);
#undef NB_TILES
    } else {
      const uint32_t tb = cdiv(n_tiles, 256), g = tb + (apart ? 0u : fb_blocks(p, 256));
      if (batch)
        k_bin_mark<true><<<g, 256, 0, s>>>(p, d.rec, d.materials, d.tile_cnt, d.tile_mark, d.tile_sums, n_tiles, tb);
      else
        k_bin_mark<false><<<g, 256, 0, s>>>(p, d.rec, d.materials, d.tile_cnt, d.tile_mark, d.tile_sums, n_tiles, tb);
    }
  }
  if (!small) {
    ProfScope ps(pf, 2, s);
    const uint32_t tb = cdiv(n_tiles, 256);
#define NB_COMPACT(SC)                                                                                            \
  k_bin_compact<SC><<<tb, 256, 0, s>>>(d.tile_mark, d.tile_sums, d.tile_cnt, d.tile_act, d.act_tiles, d.node_tiles, \
                                       d.tile_total, d.tile_start, d.tile_order, d.counters, d.units, n_tiles)
    if (tb > kSumBlocks) {
      k_bin_sums<<<1, 1024, 0, s>>>(d.tile_sums, tb);
      NB_COMPACT(true);
    } else {
      NB_COMPACT(false);
    }
#undef NB_COMPACT
  }
  {
    ProfScope ps(pf, 3, s);
    const uint32_t nb = cdiv(p.n, 256), fb = small && !apart ? fb_blocks(p, 256) : 0u;
#define NB_SCATTER_FB(PK, BT)                                                                                   \
  k_bin_scatter_fb<PK, BT><<<nb + fb, 256, 0, s>>>(p, d.rec, d.materials, d.keys, d.rank, d.tile_act, d.tile_start, \
                                                   d.bucket, fb)
    const bool packed = p.n <= kPackedParticles;
    if (!fb) {
      if (packed) k_bin_scatter<true><<<nb, 256, 0, s>>>(p.n, d.keys, d.rank, d.tile_act, d.tile_start, d.bucket);
      else k_bin_scatter<false><<<nb, 256, 0, s>>>(p.n, d.keys, d.rank, d.tile_act, d.tile_start, d.bucket);
    } else if (packed) {
      if (batch) NB_SCATTER_FB(true, true); else NB_SCATTER_FB(true, false);
    } else {
      if (batch) NB_SCATTER_FB(false, true); else NB_SCATTER_FB(false, false);
    }
#undef NB_SCATTER_FB
  }
  {
    ProfScope ps(pf, 4, s);
    uint32_t* fb_ctl = p.svd_fp64 ? p.fb_ctl : nullptr;
    uint4* items = p.by_item ? d.items : nullptr;
    if (p.n <= kPackedParticles)
      k_bin_sort<true><<<tg, kSortThreads, 0, s>>>(p.n, d.bucket, d.cell_count, d.cell_end, d.act_tiles, d.tile_start,
                                                   d.tile_total, d.sorted, d.counters, fb_ctl, p.p2g_item, items, d.cell_item, d.tile_items);
    else
      k_bin_sort<false><<<tg, kSortThreads, 0, s>>>(p.n, d.bucket, d.cell_count, d.cell_end, d.act_tiles, d.tile_start,
                                                    d.tile_total, d.sorted, d.counters, fb_ctl, p.p2g_item, items, d.cell_item, d.tile_items);
  }
}

void launch_p2g(const DevState& d, const SubParams& p, uint32_t n_tiles, hipStream_t s, Prof* pf) {
  ProfScope ps(pf, 5, s);
  const P2GItems q{d.cell_item, d.tile_items, d.item_sum, d.item_cap};
  if (p.by_item) {
    const uint32_t chunks = cdiv(cdiv(p.n, 64), kXCDs) * kXCDs;
#define NB_ITEMS(SP, BT) \
  k_p2g_items<SP, BT><<<SP * chunks, 64, 0, s>>>(p, d.rec, d.materials, d.sorted, d.items, d.item_sum, d.item_cap, d.counters)
    if (p.by_item == 4u) {
      if (p.n_scenes > 0) NB_ITEMS(4, true); else NB_ITEMS(4, false);
    } else if (p.by_item == 2u) {
      if (p.n_scenes > 0) NB_ITEMS(2, true); else NB_ITEMS(2, false);
    } else {
      if (p.n_scenes > 0) NB_ITEMS(1, true); else NB_ITEMS(1, false);
    }
#undef NB_ITEMS
  }
#define NB_P2G(BT, IT)                                                                                                   \
  k_p2g<BT, IT><<<IT ? tile_grid(kMergeBlocks * n_tiles, p.tile_blocks) : tile_grid(n_tiles, p.tile_blocks), kP2GThreads, 0, \
                  s>>>(p, d.rec, d.materials, d.cell_count, d.cell_end, d.sorted, d.act_tiles, d.tile_order,             \
                       d.tile_start, d.tile_total, d.counters, q, d.partial)
  if (p.n_scenes > 0) {
    if (p.by_item) NB_P2G(true, true); else NB_P2G(true, false);
  } else {
    if (p.by_item) NB_P2G(false, true); else NB_P2G(false, false);
  }
#undef NB_P2G
}

void launch_grid(const DevState& d, const SubParams& p, uint32_t n_tiles, bool from_partials, bool update,
                 const uint32_t* tiles, const uint32_t* count, hipStream_t s, Prof* pf) {
  ProfScope ps(pf, 6, s);
  const uint32_t g = tile_grid(n_tiles, p.tile_blocks);
#define NB_GRID_LAUNCH(BT, NZ)                                                                                            \
  k_grid<BT, NZ><<<g, 512, 0, s>>>(p, tiles, count, d.grid_node, d.grid_old, d.grid_pre, d.sdf, d.colliders, d.forces)
#define NB_GRID_TILES(K, BLOCKS, THREADS)                                                                                 \
  K<<<BLOCKS, THREADS, 0, s>>>(p, d.partial, d.tile_act, d.act_tiles, d.counters, d.grid_node, d.grid_old, d.grid_pre, \
                               d.sdf, d.colliders, d.forces)
  const bool nz = p.noise_forces != 0 && update, bt = p.n_scenes > 0;
  if (from_partials && nz) {
    const uint32_t gn = tile_grid(noise_units<4>() * n_tiles, p.tile_blocks);
    if (bt) NB_GRID_TILES(k_grid_noise<true>, gn, kNoiseThreads);
    else NB_GRID_TILES(k_grid_noise<false>, gn, kNoiseThreads);
  } else if (from_partials) {
    const uint32_t gt = tile_grid(2u * n_tiles, p.tile_blocks);
    if (bt) {
      if (update) NB_GRID_TILES((k_grid_tiles<true, true>), gt, 512);
      else NB_GRID_TILES((k_grid_tiles<false, true>), gt, 512);
    } else {
      if (update) NB_GRID_TILES((k_grid_tiles<true, false>), gt, 512);
      else NB_GRID_TILES((k_grid_tiles<false, false>), gt, 512);
    }
  } else if (bt) {
    if (nz) NB_GRID_LAUNCH(true, true); else NB_GRID_LAUNCH(true, false);
  } else {
    if (nz) NB_GRID_LAUNCH(false, true); else NB_GRID_LAUNCH(false, false);
  }
#undef NB_GRID_TILES
#undef NB_GRID_LAUNCH
}

// The fused grid update + G2P (k_g2p_tile) over the work units the bin listed
// (not with turbulence or noise forces: their noise code would halve the
// kernel's occupancy; those substeps run k_grid_noise + k_g2p).
void launch_g2p_fused(const DevState& d, const SubParams& p, uint32_t n_tiles, hipStream_t s, Prof* pf) {
  // units <= occupied tiles + n / kG2PUnit; blocks stride over them
  const uint32_t max_units = n_tiles + p.n / kG2PUnit + 1u;
  const uint32_t g = tile_grid(max_units, p.tile_blocks);
  const bool flip = p.flip_ratio > 0.01f, bt = p.n_scenes > 0;
#define NB_G2PT(FL, BT)                                                                                    \
  k_g2p_tile<FL, BT><<<g, 256, 0, s>>>(p, d.rec, d.rec, d.keys, d.rank, d.tile_cnt, d.materials, d.sorted, d.units, d.act_tiles, \
                                       d.tile_start, d.tile_total, d.counters, d.tile_act, d.partial, d.sdf, \
                                       d.colliders, d.forces)
  {
    ProfScope ps(pf, 8, s);
    if (bt) {
      if (flip) NB_G2PT(true, true); else NB_G2PT(false, true);
    } else {
      if (flip) NB_G2PT(true, false); else NB_G2PT(false, false);
    }
  }
#undef NB_G2PT
}

// The FP64 fallback's fix-up after a call's last G2P, which leaves its queue
// empty (nothing to do when it is off); without records it only empties it.
void launch_g2p_fb(const DevState& d, const SubParams& p, float4* rec, hipStream_t s, Prof* pf) {
  if (!p.svd_fp64) return;
  ProfScope ps(pf, 9, s);
  if (rec) launch_fb_entries(d, p, rec, s);
  k_g2p_fb_reset<<<1, 64, 0, s>>>(p.fb_ctl);
}

void launch_g2p(const DevState& d, const SubParams& p, bool use_sorted, bool count, hipStream_t s, Prof* pf,
                float4* rec_out) {
  uint32_t* tile_cnt = count ? d.tile_cnt : nullptr;
  const uint32_t* srt = use_sorted ? d.sorted : nullptr;
  float4* out = rec_out ? rec_out : d.rec;
  const bool flip = p.flip_ratio > 0.01f, bt = p.n_scenes > 0;
  {
    ProfScope ps(pf, 7, s);
#define NB_G2P_LAUNCH(FL, BT) \
  k_g2p<FL, BT><<<cdiv(p.n, bs), bs, 0, s>>>(p, d.rec, out, d.keys, d.rank, tile_cnt, d.materials, srt, d.grid_node, d.grid_old, d.sdf)
    const uint32_t bs = (p.g2p_block == 64u || p.g2p_block == 128u) ? p.g2p_block : 256u;  // launch bound 256
    if (bt) {
      if (flip) NB_G2P_LAUNCH(true, true);
      else NB_G2P_LAUNCH(false, true);
    } else {
      if (flip) NB_G2P_LAUNCH(true, false);
      else NB_G2P_LAUNCH(false, false);
    }
#undef NB_G2P_LAUNCH
  }
}

// ---------------------------------------------------------------------------
// mesh SDF (src/core/MeshSDF.h:85-126): per cell of the grid, the distance to
// the closest point of any triangle (Ericson's closest-point regions,
// MeshSDF.h:42-75), signed by that triangle's normal (the first triangle at
// the minimum distance); cube cells outside the grid hold 1e9.  Every product
// and sum of a distance is rounded as written (no FMA contraction), as on the
// host.
//
// A cell's result is the minimum over all triangles, but few of them can hold
// it: a block takes one 8^3 brick of cells, measures the triangle of the nearest
// centroid from each (U: the largest of these distances) and keeps, in index
// order, the triangles whose own lower bound does not exceed U; each wave then
// does the same for its 4^3 sub-brick over that list, holds for each triangle a
// linear lower bound (a distance to a triangle is convex), measures the nearest
// one and then only those whose bound is not above some lane's best.  What is
// compared with a bound is always a distance measured, and a bound is lowered by
// what rounding can take from the distance that would be measured (mesh_error),
// so a triangle dropped is neither a minimum nor a tie: values and signs have the
// bits of the pass over all triangles.  On 128^3 cells and 3,360 triangles a cell
// measures about 26 distances instead of 3,360 and the search takes 0.64 ms
// where the pass over all takes 10.1 (VALU-bound; 0.98 with the wave's bound alone).
// ---------------------------------------------------------------------------
// The closest point of triangle t (normal, v0, v1, v2) to p.  EXACT adds the
// region of the edge v1-v2 that closestPtOnTriangle leaves out.
template <bool EXACT>
__device__ __forceinline__ float3 tri_closest(const float* t, float px, float py, float pz) {
#pragma clang fp contract(off)
  auto dot3 = [](float ax, float ay, float az, float bx, float by, float bz) {
#pragma clang fp contract(off)
    return (ax * bx + ay * by) + az * bz;
  };
  const float ax = t[3], ay = t[4], az = t[5];
  const float abx = t[6] - ax, aby = t[7] - ay, abz = t[8] - az;
  const float acx = t[9] - ax, acy = t[10] - ay, acz = t[11] - az;
  const float apx = px - ax, apy = py - ay, apz = pz - az;
  const float d1 = dot3(abx, aby, abz, apx, apy, apz), d2 = dot3(acx, acy, acz, apx, apy, apz);
  if (d1 <= 0.f && d2 <= 0.f) return make_float3(ax, ay, az);
  const float bpx = px - t[6], bpy = py - t[7], bpz = pz - t[8];
  const float d3 = dot3(abx, aby, abz, bpx, bpy, bpz), d4 = dot3(acx, acy, acz, bpx, bpy, bpz);
  const float vc = d1 * d4 - d3 * d2;
  if (d3 >= 0.f && d4 <= d3) return make_float3(t[6], t[7], t[8]);
  if (vc <= 0.f && d1 >= 0.f && d3 <= 0.f) {
    const float v = d1 / (d1 - d3);
    return make_float3(ax + v * abx, ay + v * aby, az + v * abz);
  }
  const float cpx = px - t[9], cpy = py - t[10], cpz = pz - t[11];
  const float d5 = dot3(abx, aby, abz, cpx, cpy, cpz), d6 = dot3(acx, acy, acz, cpx, cpy, cpz);
  const float vb = d5 * d2 - d1 * d6;
  if (d6 >= 0.f && d5 <= d6) return make_float3(t[9], t[10], t[11]);
  if (vb <= 0.f && d2 >= 0.f && d6 <= 0.f) {
    const float w = d2 / (d2 - d6);
    return make_float3(ax + w * acx, ay + w * acy, az + w * acz);
  }
  const float va = d3 * d6 - d5 * d4;
  if (EXACT && va <= 0.f && d4 - d3 >= 0.f && d5 - d6 >= 0.f) {  // edge v1-v2
    const float w = (d4 - d3) / ((d4 - d3) + (d5 - d6));
    return make_float3(t[6] + w * (t[9] - t[6]), t[7] + w * (t[10] - t[7]), t[8] + w * (t[11] - t[8]));
  }
  const float sum = va + vb + vc;
  const float v = vb / sum, w = vc / sum;
  return make_float3(ax + v * abx + w * acx, ay + v * aby + w * acy, az + v * abz + w * acz);
}

constexpr uint32_t kMeshThreads = 512;       // cells of a brick
constexpr uint32_t kMeshList = 2048;         // triangles a block holds at a time
constexpr int kMeshHeld = 8;                 // of them, those a lane holds bounds of at a time
constexpr float kMeshSlack = 1e-3f;          // of the lengths in a bound: far above their rounding
// What rounding can do to a distance.  With l the triangle's longest edge, N its
// cross product, k = l^2 / |N| (longest edge over height), R the distance to its
// farthest vertex and u = 2^-24: the dot products of tri_closest are off by up to 6 u
// l R and the barycentric numerators of a point within about l of the triangle
// sideways by some 24 u l^3 R.  A point up to 48 u k^2 R beside the triangle may so be
// taken to lie over it, which takes that much at most from its distance: from there on
// the closest point lies in the plane, wherever.  The closest point of a point over
// the triangle moves within the plane, by 3.4 u k^2 R at most in 8e7 tries over k of 1.2
// to 90 and R / l of 0.3 to 10^4.  All this while the error is below the triangle's
// size; beyond, a distance may be anything down to that to the plane, and the triangle
// is measured everywhere.
constexpr float kMeshError = 2.9e-6f;  // 48 u

// Centroid and radius of each triangle, and its kMeshError k^2.  A triangle of no
// height (below a hundredth of its longest edge), not finite or beyond the range
// where its products are gets a negative radius: it bounds nothing and is never
// dropped.  bounded: how many have bounds.
__global__ __launch_bounds__(256) void k_mesh_spheres(const float* __restrict__ tris, uint32_t n_tris,
                                                      float4* __restrict__ sph, float* __restrict__ err,
                                                      uint32_t* __restrict__ bounded) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_tris) return;
  const float* t = tris + size_t(i) * 12;
  const float gx = (t[3] + t[6] + t[9]) / 3.f, gy = (t[4] + t[7] + t[10]) / 3.f, gz = (t[5] + t[8] + t[11]) / 3.f;
  float r = 0.f;
#pragma unroll
  for (int k = 0; k < 3; k++) r = fmaxf(r, len3(t[3 + 3 * k] - gx, t[4 + 3 * k] - gy, t[5 + 3 * k] - gz));
  const float ax = t[6] - t[3], ay = t[7] - t[4], az = t[8] - t[5], bx = t[9] - t[3], by = t[10] - t[4], bz = t[11] - t[5];
  const float nx = ay * bz - az * by, ny = az * bx - ax * bz, nz = ax * by - ay * bx;
  const float cx = bx - ax, cy = by - ay, cz = bz - az;
  const float l2 = fmaxf(fmaxf(ax * ax + ay * ay + az * az, bx * bx + by * by + bz * bz), cx * cx + cy * cy + cz * cz);
  const float n2 = nx * nx + ny * ny + nz * nz;
  const bool good = n2 > 1e-4f * l2 * l2 && n2 > 1e-30f && l2 < 1e14f && fabsf(gx) + fabsf(gy) + fabsf(gz) < 1e15f;
  sph[i] = make_float4(gx, gy, gz, good ? r * (1.f + kMeshSlack) : -1.f);
  err[i] = good ? kMeshError * (l2 * l2 / n2) : 0.f;
  const uint64_t bound = __ballot(good), here = __ballot(true);
  if ((threadIdx.x & 63u) == uint32_t(__ffsll((unsigned long long)here)) - 1u) atomicAdd(bounded, uint32_t(__popcll(bound)));
}

// Whether a mesh of n triangles is for k_mesh_all.
__device__ __forceinline__ bool mesh_mostly_unbounded(uint32_t bounded, uint32_t n) { return bounded <= n / 2u; }

// What rounding can take from a distance to a triangle of radius rad none of whose
// vertices is farther than R; INFINITY where that is not bounded.
__device__ __forceinline__ float mesh_error(float err, float rad, float R) {
  const float e = err * R;
  return e <= rad ? e : INFINITY;
}

// Whether some point of the ball (centre (cx, cy, cz), radius r) can lie in the
// region of the edge v1-v2 that the closest point without EXACT leaves out,
// where it takes its distance to the triangle's plane, and within `most` of
// that plane: the slab between the planes through v1 and v2 across the edge,
// on the far side of it.
__device__ __forceinline__ bool mesh_edge_slab(const float* __restrict__ t, float cx, float cy, float cz, float r,
                                               float slack, float most) {
  const float ax = t[3], ay = t[4], az = t[5];
  const float abx = t[6] - ax, aby = t[7] - ay, abz = t[8] - az, acx = t[9] - ax, acy = t[10] - ay, acz = t[11] - az;
  const float nx = aby * acz - abz * acy, ny = abz * acx - abx * acz, nz = abx * acy - aby * acx;
  const float in = 1.f / len3(nx, ny, nz);
  const float ex = acx - abx, ey = acy - aby, ez = acz - abz, le = len3(ex, ey, ez), ie = 1.f / le;
  const float px = cx - t[6], py = cy - t[7], pz = cz - t[8];
  const float along = (px * ex + py * ey + pz * ez) * ie;
  // the in-plane direction out of the triangle across the edge: e x n
  const float mx = ey * nz - ez * ny, my = ez * nx - ex * nz, mz = ex * ny - ey * nx;
  const float beyond = (px * mx + py * my + pz * mz) * ie * in;
  const float off = fabsf(px * nx + py * ny + pz * nz) * in;
  const float rs = r + slack;
  return along >= -rs && along <= le + rs && beyond >= -rs && !(off - r > most + slack);
}

// Whether triangle t, its centroid's distance dg and its radius rad from the
// centre (cx, cy, cz) of a ball of radius r known, may hold the minimum of a
// point of the ball when a distance of at most U is known for each.
template <bool EXACT>
__device__ __forceinline__ bool mesh_may_hold(const float* __restrict__ t, float dg, float rad, float err, float cx,
                                              float cy, float cz, float r, float U) {
  if (!(rad >= 0.f)) return true;
  const float R = dg + rad + r, slack = kMeshSlack * R + mesh_error(err, rad, R);
  if (!(dg - rad - r > U + slack)) return true;
  return !EXACT && mesh_edge_slab(t, cx, cy, cz, r, slack, U);
}

// One block per 8^3 brick of the cube (first_brick + blockIdx.x), one cell a
// thread in Morton order, so that each wave holds a 4^3 sub-brick.
template <bool EXACT>
__global__ __launch_bounds__(kMeshThreads) void k_mesh_sdf(const float* __restrict__ tris,
                                                           const float4* __restrict__ sph,
                                                           const float* __restrict__ err,
                                                           const uint32_t* __restrict__ bounded, uint32_t n_tris, int rx,
                                                           int ry, int rz, uint32_t nc, uint32_t first_brick, float cs,
                                                           float* __restrict__ sdf) {
#pragma clang fp contract(off)
  if (mesh_mostly_unbounded(*bounded, n_tris)) return;
  constexpr uint32_t kWaves = kMeshThreads / 64;
  __shared__ uint32_t s_list[kMeshList];
  __shared__ float4 s_tri[kWaves][64][4];  // a triangle and its index
  __shared__ float s_min[kWaves], s_max[kWaves];
  __shared__ uint32_t s_arg[kWaves], s_cnt[kWaves];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t m = (first_brick + blockIdx.x) * kMeshThreads + threadIdx.x;
  const int ix = int(morton_compact(m)), iy = int(morton_compact(m >> 1)), iz = int(morton_compact(m >> 2));
  const bool valid = m < nc && ix < rx && iy < ry && iz < rz;
  const int bx = ix & ~7, by = iy & ~7, bz = iz & ~7;
  if (bx >= rx || by >= ry || bz >= rz) {  // the whole brick lies outside the grid
    if (m < nc) sdf[m] = 1e9f;
    return;
  }
  const float px = (float(ix) + 0.5f) * cs, py = (float(iy) + 0.5f) * cs, pz = (float(iz) + 0.5f) * cs;
  // the least distance measured so far and its triangle (a cell outside the grid
  // wants none)
  float best = valid ? 1e9f : -INFINITY;
  uint32_t best_j = 0u;
  bool outer = true;
  auto measure = [&](const float* t, uint32_t j) {
    const float3 q = tri_closest<EXACT>(t, px, py, pz);
    const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
    const float d = sqrtf((dx * dx + dy * dy) + dz * dz);
    if (d < best || (d == best && j < best_j)) {
      best = d;
      best_j = j;
      outer = (dx * t[0] + dy * t[1]) + dz * t[2] >= 0.f;
    }
  };
  auto wave_max = [](float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d));
    return v;
  };
  // the brick's ball; the triangle of the nearest centroid, and the largest of its
  // distances from the brick's cells
  const float bcx = float(bx + 4) * cs, bcy = float(by + 4) * cs, bcz = float(bz + 4) * cs;
  const float br = 6.0622f * cs * (1.f + kMeshSlack);  // 3.5 sqrt(3) cells
  float u = INFINITY;
  uint32_t u_j = 0u;
  for (uint32_t i = threadIdx.x; i < n_tris; i += kMeshThreads) {
    const float4 g = sph[i];
    const float d = len3(g.x - bcx, g.y - bcy, g.z - bcz);
    if (g.w >= 0.f && d < u) { u = d; u_j = i; }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    const float v = __shfl_xor(u, d);
    const uint32_t j = uint32_t(__shfl_xor(int(u_j), d));
    if (v < u || (v == u && j < u_j)) { u = v; u_j = j; }
  }
  if (lane == 0u) { s_min[wave] = u; s_arg[wave] = u_j; }
  __syncthreads();
  u = s_min[0];
  u_j = s_arg[0];
#pragma unroll
  for (uint32_t w = 1; w < kWaves; w++)
    if (s_min[w] < u) { u = s_min[w]; u_j = s_arg[w]; }
  u_j = uint32_t(__builtin_amdgcn_readfirstlane(int(u_j)));  // one triangle for all
  measure(tris + size_t(u_j) * 12, u_j);
  const float most = wave_max(best);
  if (lane == 0u) s_max[wave] = most;
  __syncthreads();
  float U = -INFINITY;
#pragma unroll
  for (uint32_t w = 0; w < kWaves; w++) U = fmaxf(U, s_max[w]);

  const int wx = ix & ~3, wy = iy & ~3, wz = iz & ~3;
  const float wcx = float(wx + 2) * cs, wcy = float(wy + 2) * cs, wcz = float(wz + 2) * cs;
  const float wr = 2.5981f * cs * (1.f + kMeshSlack);  // 1.5 sqrt(3) cells
  uint32_t count = 0;
  for (uint32_t base = 0; base < n_tris; base += kMeshThreads) {
    const uint32_t i = base + threadIdx.x;
    bool keep = false;
    if (i < n_tris) {
      const float4 g = sph[i];
      keep = mesh_may_hold<EXACT>(tris + size_t(i) * 12, len3(g.x - bcx, g.y - bcy, g.z - bcz), g.w, err[i], bcx, bcy, bcz,
                                  br, U);
    }
    const uint64_t kept = __ballot(keep);
    __syncthreads();  // the last round's counts are read, its list entries used
    if (lane == 0u) s_cnt[wave] = uint32_t(__popcll(kept));
    __syncthreads();
    uint32_t at = count;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; w++) {
      if (w < wave) at += s_cnt[w];
      count += s_cnt[w];
    }
    if (keep) s_list[at + uint32_t(__popcll(kept & ((1ull << lane) - 1ull)))] = i;
    if (count + kMeshThreads <= kMeshList && base + kMeshThreads < n_tris) continue;
    __syncthreads();
    for (uint32_t c0 = 0; c0 < count; c0 += 64u * kMeshHeld) {
      // a lane's triangles of this part of the list: distance from the
      // sub-brick's centre and its gradient there.  The distance to a triangle
      // is convex, so d + g . (p - centre) bounds it from below at any p, less
      // what rounding does to d, to g and to the distance measured; a
      // triangle that bounds nothing there holds g = 0 and d = 0 (the missing
      // edge region makes the distance jump; too thin; the centre lies on it).
      float hd[kMeshHeld], hx[kMeshHeld], hy[kMeshHeld], hz[kMeshHeld], hs[kMeshHeld];
      float near = INFINITY;
      int near_k = 0;
#pragma unroll
      for (int k = 0; k < kMeshHeld; k++) {
        hd[k] = hx[k] = hy[k] = hz[k] = hs[k] = 0.f;
        const uint32_t e = c0 + uint32_t(k) * 64u + lane;
        if (e < count) {
          const uint32_t j = s_list[e];
          const float rad = sph[j].w;
          const float* t = tris + size_t(j) * 12;
          if (rad >= 0.f) {
            const float3 q = tri_closest<true>(t, wcx, wcy, wcz);
            const float gx = wcx - q.x, gy = wcy - q.y, gz = wcz - q.z, d = len3(gx, gy, gz);
            if (d < near) { near = d; near_k = k; }
            const float R = d + 2.f * rad + wr, e_d = mesh_error(err[j], rad, R);
            if (d > 0.25f * wr && e_d < 0.25f * d &&
                (EXACT || !mesh_edge_slab(t, wcx, wcy, wcz, wr, kMeshSlack * R + e_d, INFINITY))) {
              hd[k] = d;
              hx[k] = gx / d; hy[k] = gy / d; hz[k] = gz / d;
              hs[k] = 4.f * kMeshSlack * (d + wr) + e_d * (2.f + 3.f * wr / d);
            }
          }
        }
      }
      // the wave's nearest triangle first (any order gives the same result:
      // equal distances go to the lower index), then the others in turn
      float nearest = near;
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) nearest = fminf(nearest, __shfl_xor(nearest, d));
      const uint64_t at_min = __ballot(near == nearest && near < INFINITY);
      if (at_min) {
        const int l = __ffsll((unsigned long long)at_min) - 1;
        const uint32_t j = uint32_t(__builtin_amdgcn_readfirstlane(
            int(s_list[c0 + uint32_t(__builtin_amdgcn_readlane(near_k, l)) * 64u + uint32_t(l)])));
        measure(tris + size_t(j) * 12, j);
      }
      const float W = wave_max(best);
#pragma unroll
      for (int k = 0; k < kMeshHeld; k++) {
        const uint32_t e0 = c0 + uint32_t(k) * 64u;
        if (e0 >= count) break;
        const bool listed = e0 + lane < count, wanted = listed && !(hd[k] - wr > W + hs[k]);
        uint64_t todo = __ballot(wanted);
        if (!todo) continue;
        const uint32_t j = listed ? s_list[e0 + lane] : 0u;
        // through LDS, 64 triangles at a time (read one by one from memory each would
        // wait for its own loads), first those that have no bound
        const uint64_t all = __ballot(wanted && hd[k] == 0.f), below = (1ull << lane) - 1ull;
        const uint32_t n_all = uint32_t(__popcll(all));
        todo &= ~all;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (wanted) {
          const float4* t = reinterpret_cast<const float4*>(tris + size_t(j) * 12);
          float4* at = s_tri[wave][(all >> lane) & 1ull ? uint32_t(__popcll(all & below)) : n_all + uint32_t(__popcll(todo & below))];
#pragma unroll
          for (int q = 0; q < 3; q++) at[q] = t[q];
          at[3].x = __uint_as_float(j);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const float4* t = s_tri[wave][0];
#pragma unroll 2
        for (uint32_t i = 0; i < n_all; i++, t += 4) measure(reinterpret_cast<const float*>(t), __float_as_uint(t[3].x));
        for (; todo; todo &= todo - 1ull, t += 4) {
          const int l = __ffsll((unsigned long long)todo) - 1;
          auto of = [&](float v) { return __uint_as_float(uint32_t(__builtin_amdgcn_readlane(int(__float_as_uint(v)), l))); };
          const float low = of(hd[k]) + of(hx[k]) * (px - wcx) + of(hy[k]) * (py - wcy) + of(hz[k]) * (pz - wcz) - of(hs[k]);
          if (__any(!(low > best))) measure(reinterpret_cast<const float*>(t), __float_as_uint(t[3].x));
        }
      }
    }
    count = 0;
  }
  if (m < nc) sdf[m] = valid ? (outer ? best : -best) : 1e9f;
}

// The pass over all triangles, for few of them (bounded null), or where most have no
// bound: what the bounds cost is then not made good.  It holds nothing but a cell's
// best, 8 waves a SIMD where the search has 4.  Whole calls on 256^3 cells with 1 / 12
// triangles: 469 / 664 us searched, 141 / 520 this way; 2000 of no height: 35 ms and 24.
constexpr uint32_t kMeshFew = 16;
template <bool EXACT>
__global__ __launch_bounds__(256) void k_mesh_all(const float* __restrict__ tris, const uint32_t* __restrict__ bounded,
                                                  uint32_t n_tris, int rx, int ry, int rz, uint32_t nc,
                                                  uint32_t first_brick, float cs, float* __restrict__ sdf) {
#pragma clang fp contract(off)
  if (bounded != nullptr && !mesh_mostly_unbounded(*bounded, n_tris)) return;
  constexpr uint32_t kStage = 256;
  __shared__ float4 s_tri[kStage * 3];
  const uint32_t m = first_brick * kMeshThreads + blockIdx.x * 256u + threadIdx.x;
  const int ix = int(morton_compact(m)), iy = int(morton_compact(m >> 1)), iz = int(morton_compact(m >> 2));
  const bool valid = m < nc && ix < rx && iy < ry && iz < rz;
  const float px = (float(ix) + 0.5f) * cs, py = (float(iy) + 0.5f) * cs, pz = (float(iz) + 0.5f) * cs;
  float best = 1e9f;
  bool outer = true;
  if (__syncthreads_or(valid)) {
    for (uint32_t t0 = 0; t0 < n_tris; t0 += kStage) {
      const uint32_t nt = min(kStage, n_tris - t0);
      __syncthreads();
      for (uint32_t e = threadIdx.x; e < nt * 3u; e += 256u)
        s_tri[e] = reinterpret_cast<const float4*>(tris + size_t(t0) * 12)[e];
      __syncthreads();
      if (!valid) continue;
      for (uint32_t j = 0; j < nt; j++) {
        const float* t = reinterpret_cast<const float*>(s_tri) + 12 * j;
        const float3 q = tri_closest<EXACT>(t, px, py, pz);
        const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
        const float d = sqrtf((dx * dx + dy * dy) + dz * dz);
        if (d < best) {
          best = d;
          outer = (dx * t[0] + dy * t[1]) + dz * t[2] >= 0.f;
        }
      }
    }
  }
  if (m < nc) sdf[m] = valid ? (outer ? best : -best) : 1e9f;
}

void launch_mesh_sdf(const float* tris, void* scratch, uint32_t n_tris, const int32_t res[3], uint32_t cube, float cs,
                     bool exact, float* sdf, hipStream_t s) {
  const uint32_t nc = cube * cube * cube, bricks = cdiv(nc, kMeshThreads);
  float4* sph = static_cast<float4*>(scratch);
  float* err = reinterpret_cast<float*>(sph + n_tris);
  uint32_t* bounded = reinterpret_cast<uint32_t*>(err + n_tris);
  const bool few = n_tris <= kMeshFew;
  if (!few) {
    k_zero<<<1, 256, 0, s>>>(bounded, 1u);
    k_mesh_spheres<<<cdiv(n_tris, 256), 256, 0, s>>>(tris, n_tris, sph, err, bounded);
  }
  // so that no launch runs long on a large mesh: at most 2^31 triangle tests
  // (a brick against a triangle) to a launch
  const uint32_t step = std::max(1u, uint32_t((uint64_t(1) << 31) / std::max(n_tris, 1u)));
  for (uint32_t b0 = 0; b0 < bricks; b0 += step) {
    const uint32_t nb = std::min(step, bricks - b0);
#define NB_MESH(EX)                                                                                                   \
  if (!few)                                                                                                           \
    k_mesh_sdf<EX><<<nb, kMeshThreads, 0, s>>>(tris, sph, err, bounded, n_tris, res[0], res[1], res[2], nc, b0, cs, sdf); \
  k_mesh_all<EX><<<nb * (kMeshThreads / 256u), 256, 0, s>>>(tris, few ? nullptr : bounded, n_tris, res[0], res[1],     \
                                                            res[2], nc, b0, cs, sdf)
    if (exact) {
      NB_MESH(true);
    } else {
      NB_MESH(false);
    }
#undef NB_MESH
  }
}

void launch_sdf_sphere(float* sdf, const SubParams& p, float r, float cx, float cy, float cz, hipStream_t s) {
  const uint32_t nc = p.cube_res * p.cube_res * p.cube_res;
  k_sdf_sphere<<<cdiv(nc, 256), 256, 0, s>>>(sdf, p, r, cx, cy, cz);
}

void launch_fill_identity(uint32_t* a, uint32_t rows, uint32_t n, hipStream_t s) {
  for (uint32_t r = 0; r < rows; r += 32768u)
    k_fill_identity<<<dim3(cdiv(n, 256), std::min(rows - r, 32768u)), 256, 0, s>>>(a + size_t(r) * n, n);
}

void launch_soa_to_aos(const DevState& d, const SubParams& p, bool count, hipStream_t s) {
  if (!p.n) return;
  FieldPtrs f;
  for (int i = 0; i < NB_NUM_FIELDS; i++) f.f[i] = d.field[i];
  const uint32_t g = cdiv(p.n, 256);
  if (!count) k_soa_to_aos<false, false><<<g, 256, 0, s>>>(p, f, d.rec, p.n, nullptr, nullptr, nullptr);
  else if (p.n_scenes > 0) k_soa_to_aos<true, true><<<g, 256, 0, s>>>(p, f, d.rec, p.n, d.keys, d.rank, d.tile_cnt);
  else k_soa_to_aos<true, false><<<g, 256, 0, s>>>(p, f, d.rec, p.n, d.keys, d.rank, d.tile_cnt);
}

void launch_aos_to_soa(const DevState& d, uint32_t n, hipStream_t s) {
  if (!n) return;
  FieldPtrs f;
  for (int i = 0; i < NB_NUM_FIELDS; i++) f.f[i] = d.field[i];
  k_aos_to_soa<<<cdiv(n, 256), 256, 0, s>>>(d.rec, f, n);
}

void launch_soa_to_aos_ptrs(const FieldPtrs& f, float4* rec, uint32_t n, hipStream_t s) {
  if (n) k_soa_to_aos<false, false><<<cdiv(n, 256), 256, 0, s>>>(SubParams{}, f, rec, n, nullptr, nullptr, nullptr);
}
void launch_aos_to_soa_ptrs(const float4* rec, const FieldPtrs& f, uint32_t n, hipStream_t s) {
  if (n) k_aos_to_soa<<<cdiv(n, 256), 256, 0, s>>>(rec, f, n);
}

void launch_copy(float4* dst, const float4* src, uint64_t n4, hipStream_t s) {
  k_copy<<<8192, 256, 0, s>>>(dst, src, n4);
}

void launch_init_particles(const DevState& d, uint32_t first, uint32_t count, hipStream_t s) {
  if (!count) return;
  k_init_FB<<<cdiv(count, 256), 256, 0, s>>>(d.field[2], d.field[3], d.field[4], d.field[5], d.field[6], d.field[7],
                                             first, count);
}

}  // namespace nb
