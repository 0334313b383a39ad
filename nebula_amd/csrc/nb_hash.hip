// nb_hash.hip — the spatial hash of the reference's position-based engines
// (PBF fluid, cloth self-collision) behind nb_hash_build (include/nebula_hash.h).
//
// The reference records six dispatches (zero_cells, hash_count,
// hash_scan_local, hash_scan_global, hash_add_base, hash_sort) over
// engine-owned buffers.  Here:
//   k_hash_clear      zero cell_count (and the scratch counter)
//   k_hash_count      cell of every particle, one atomic count per run of lanes (in
//                     few cells: per cell of a wave)
//   k_hash_chunk_sums / k_hash_chunk_scan / k_hash_offsets
//                     exclusive prefix of the counts in two levels (4096 cells
//                     per block; no group-count limit; the scan kernel only
//                     beyond 4096 blocks) -> START offsets
//   k_hash_place      END offsets less the place the count gave each particle;
//                     without room for the places k_hash_scatter: slot =
//                     atomicAdd(START of the cell) -> cell_offset ends as END
//                     offsets, as after hash_sort
//   k_hash_stabilize  every cell's slice of `sorted` put in ascending particle
//                     order: cells of <= 16 in registers by a sorting network, of
//                     <= 512 by a wave (in larger hashes, many: listed), more
//                     crowded ones left for k_hash_crowded
//   k_hash_crowded    listed cells of <= 512 by a wave each, larger ones by a
//                     block each: bitonic sort in LDS (up to 16384 particles) or
//                     in place in global memory
// Per-particle work reads the 16-byte predP (and typeFlag).  The result does not depend on the order of the
// atomics, so it is deterministic.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/nebula_hash.h"
#include "../../include/nebula_mpm.h"
#include "nb_device_math.hpp"
#include "nb_engine.hpp"
#include "nb_kernel_util.hpp"

namespace nbh {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kItems = 16;                         // cells per thread in the scan
constexpr uint32_t kChunk = kThreads * kItems;          // cells per scan block
constexpr uint32_t kMaxChunks = NB_HASH_MAX_CELLS / kChunk;
constexpr uint32_t kSmall = 16;                         // cells up to this size: sorted by their thread
constexpr uint32_t kLdsSort = 16384;                    // crowded cells up to this size: sorted in LDS
constexpr uint32_t kCrowdThreads = 512;
constexpr uint32_t kSumChunks = 4096;                   // up to this many chunks: no scan kernel
constexpr uint32_t kWaveSort = 512;                     // crowded cells up to this size: sorted by one wave
constexpr uint32_t kWaveCells = 4;                      // so many of them the wave that meets them sorts at once
constexpr uint32_t kBigStep = 256;                      // every cell of more than kWaveSort has a multiple of it
constexpr uint32_t kCrowdCap = 65536;                   // listed crowded cells; beyond: a dense sweep
// scratch layout (uint32 words)
constexpr uint32_t kOffCrowdCount = kMaxChunks;         // after the chunk sums
constexpr uint32_t kOffCrowdList = kMaxChunks + 64;
constexpr uint32_t kScratchWords = kOffCrowdList + kCrowdCap;

struct Geo {
  float wmin[3];
  float h;
  float gmax[3];  // grid_res - 1
};

// cellId (shaders/common.glsl:100-105): IEEE quotient, clamp to
// [0, gridRes - 1] (NaN maps to 0: fmaxf returns the other operand), truncation
__device__ __forceinline__ uint32_t hash_cell(const Geo& g, const float4 p) {
  const float lx = fminf(fmaxf((p.x - g.wmin[0]) / g.h, 0.f), g.gmax[0]);
  const float ly = fminf(fmaxf((p.y - g.wmin[1]) / g.h, 0.f), g.gmax[1]);
  const float lz = fminf(fmaxf((p.z - g.wmin[2]) / g.h, 0.f), g.gmax[2]);
  return nb::morton3(uint32_t(lx), uint32_t(ly), uint32_t(lz));
}

// Adds one per valid lane to counters[key]; returns the value before the lane's
// atomic's add plus the lane's place among the lanes it covers.  Call from uniform
// control flow.
// One atomic per run of equal keys in neighbouring lanes: particles stored in no
// spatial order have 64 runs a wave, and a loop that groups all equal keys takes a turn
// for each (94 us for the count of 2,000,003 such particles in 256 x 128 x 200 cells
// and 148 for their scatter, against 83 and 128 by runs, bound by the cells' lines
// then, one moved by each atomic; 32,768 in 64^3 cells: 11 and 12 us against 4.6 and
// 5.1).  In few cells the atomics themselves meet: 200,000 particles in 4^3 cells took
// 287 us by runs and 63 in groups.  Equal keys in different runs tell the two apart,
// looked for at four of the wave's lanes (32,768 particles in 8^3 cells: 11 and 15 us;
// two waves in five find a pair there, nearly all do in 4^3 cells).
__device__ __forceinline__ uint32_t wave_add(uint32_t* __restrict__ counters, uint32_t key, bool valid) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t k = valid ? key : 0xFFFFFFFFu;  // no cell has this key
  const uint32_t before = uint32_t(__shfl_up(int(k), 1));
  const uint64_t heads = __ballot(lane == 0u || before != k);
  auto in_runs = [&](int l) {
    const uint32_t kl = uint32_t(__builtin_amdgcn_readlane(int(k), l));
    const uint64_t peers = __ballot(k == kl) & heads;
    return kl != 0xFFFFFFFFu && (peers & (peers - 1ull)) != 0ull;
  };
  uint32_t leader, place, count = 0, base = 0;
  if (!(in_runs(0) || in_runs(16) || in_runs(32) || in_runs(48))) {
    leader = 63u - uint32_t(__clzll((long long)(heads & (below | (1ull << lane)))));
    place = lane - leader;
    const uint64_t after = heads & ~(below | (1ull << lane));
    count = (after ? uint32_t(__ffsll((unsigned long long)after)) - 1u : 64u) - lane;
  } else {
    leader = lane;
    place = 0;
    uint64_t pending = __ballot(valid);
    while (pending) {
      const int l = __ffsll((unsigned long long)pending) - 1;
      const bool mine = k == uint32_t(__builtin_amdgcn_readlane(int(k), l));
      const uint64_t peers = __ballot(mine);
      if (mine) {
        leader = uint32_t(l);
        place = uint32_t(__popcll(peers & below));
        count = uint32_t(__popcll(peers));
      }
      pending &= ~peers;
    }
  }
  if (valid && leader == lane) base = atomicAdd(&counters[key], count);
  return uint32_t(__shfl(int(base), int(leader))) + place;
}

__global__ __launch_bounds__(kThreads) void k_hash_clear(uint32_t* __restrict__ cell_count, uint32_t nc,
                                                         uint32_t* __restrict__ scratch) {
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if ((reinterpret_cast<uintptr_t>(cell_count) & 15u) == 0u) {
    uint4* c4 = reinterpret_cast<uint4*>(cell_count);
    for (uint32_t i = t; i < nc / 4u; i += stride) c4[i] = make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t i = (nc & ~3u) + t; i < nc; i += stride) cell_count[i] = 0u;
  } else {
    for (uint32_t i = t; i < nc; i += stride) cell_count[i] = 0u;
  }
  if (t == 0 && scratch != nullptr) scratch[kOffCrowdCount] = 0u;
}

// RANKED: keeps each particle's place in its cell
template <bool RANKED>
__global__ __launch_bounds__(kThreads) void k_hash_count(Geo g, const float4* __restrict__ pred,
                                                         const uint32_t* __restrict__ type_flag, uint32_t n,
                                                         uint32_t* __restrict__ cell_count,
                                                         uint32_t* __restrict__ rank) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  bool valid = i < n;
  uint32_t key = 0;
  if (valid) {
    if (type_flag != nullptr && type_flag[i] == NB_HASH_TYPE_UNUSED) valid = false;
    else key = hash_cell(g, pred[i]);
  }
  const uint32_t r = wave_add(cell_count, key, valid);
  if (RANKED && valid) rank[i] = r;
}

// the kItems counts of thread t in chunk b (zeros past nc)
__device__ __forceinline__ void load_items(const uint32_t* __restrict__ c, uint32_t nc, uint32_t first,
                                           uint32_t (&v)[kItems]) {
  if (first + kItems <= nc && (reinterpret_cast<uintptr_t>(c + first) & 15u) == 0u) {
    const uint4* c4 = reinterpret_cast<const uint4*>(c + first);
#pragma unroll
    for (uint32_t q = 0; q < kItems / 4u; q++) {
      const uint4 a = c4[q];
      v[4 * q + 0] = a.x; v[4 * q + 1] = a.y; v[4 * q + 2] = a.z; v[4 * q + 3] = a.w;
    }
  } else {
#pragma unroll
    for (uint32_t k = 0; k < kItems; k++) v[k] = first + k < nc ? c[first + k] : 0u;
  }
}

// The chunk's sum into out[b], or (OWN) for each later chunk j into out[j kChunk + b]:
// out is then cell_offset, and the sums that a block of k_hash_offsets reads lie in the
// part that it alone writes.
template <bool OWN>
__global__ __launch_bounds__(kThreads) void k_hash_chunk_sums(const uint32_t* __restrict__ cell_count, uint32_t nc,
                                                              uint32_t* __restrict__ out) {
  __shared__ uint32_t s_wave[kThreads / 64 + 1];
  uint32_t v[kItems];
  load_items(cell_count, nc, blockIdx.x * kChunk + threadIdx.x * kItems, v);
  uint32_t s = 0;
#pragma unroll
  for (uint32_t k = 0; k < kItems; k++) s += v[k];
  uint32_t tot;
  (void)nb::block_exclusive_scan<kThreads>(s, s_wave, tot);
  if (OWN) {
    for (uint32_t j = blockIdx.x + 1u + threadIdx.x; j < gridDim.x; j += kThreads) out[size_t(j) * kChunk + blockIdx.x] = tot;
  } else if (threadIdx.x == 0) {
    out[blockIdx.x] = tot;
  }
}

// exclusive scan of the chunk sums in place, one block of 1024 threads
__global__ __launch_bounds__(1024) void k_hash_chunk_scan(uint32_t* __restrict__ scratch, uint32_t nchunks) {
  __shared__ uint32_t s_wave[1024 / 64 + 1];
  const uint32_t per = (nchunks + 1023u) / 1024u;
  const uint32_t lo = min(threadIdx.x * per, nchunks), hi = min(lo + per, nchunks);
  uint32_t s = 0;
  for (uint32_t i = lo; i < hi; i++) s += scratch[i];
  uint32_t tot;
  uint32_t run = nb::block_exclusive_scan<1024>(s, s_wave, tot);
  for (uint32_t i = lo; i < hi; i++) {
    const uint32_t x = scratch[i];
    scratch[i] = run;
    run += x;
  }
}

// START offsets (END: END offsets): the chunk's base plus the prefix inside the chunk.
// SUMS: scratch holds the chunks' sums and each block adds up those before its
// own, which saves the scan's launch (a whole kernel is 2-5 us of stream time)
// and reads at most kSumChunks words a block; OWN: these sums stand in the block's
// own part of cell_off; SCAN: scratch holds the sums' scan.
enum class Base { SCAN, SUMS, OWN };
template <Base FROM, bool END>
__global__ __launch_bounds__(kThreads) void k_hash_offsets(const uint32_t* __restrict__ cell_count, uint32_t nc,
                                                           const uint32_t* __restrict__ scratch,
                                                           uint32_t* __restrict__ cell_off) {
  __shared__ uint32_t s_wave[kThreads / 64 + 1];
  const uint32_t first = blockIdx.x * kChunk + threadIdx.x * kItems;
  uint32_t v[kItems];
  load_items(cell_count, nc, first, v);
  uint32_t s = 0;
#pragma unroll
  for (uint32_t k = 0; k < kItems; k++) s += v[k];
  uint32_t tot;
  uint32_t base;
  if (FROM != Base::SCAN) {
    uint32_t b = 0;
    for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kThreads)
      b += FROM == Base::OWN ? cell_off[size_t(blockIdx.x) * kChunk + i] : scratch[i];
    (void)nb::block_exclusive_scan<kThreads>(b, s_wave, base);  // its barriers part these reads from the writes below
  } else {
    base = scratch[blockIdx.x];
  }
  uint32_t run = base + nb::block_exclusive_scan<kThreads>(s, s_wave, tot);
#pragma unroll
  for (uint32_t k = 0; k < kItems; k++) {
    const uint32_t x = v[k];
    v[k] = END ? run + x : run;
    run += x;
  }
  if (first + kItems <= nc && (reinterpret_cast<uintptr_t>(cell_off + first) & 15u) == 0u) {
    uint4* o4 = reinterpret_cast<uint4*>(cell_off + first);
#pragma unroll
    for (uint32_t q = 0; q < kItems / 4u; q++) o4[q] = make_uint4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
  } else {
#pragma unroll
    for (uint32_t k = 0; k < kItems; k++)
      if (first + k < nc) cell_off[first + k] = v[k];
  }
}

__global__ __launch_bounds__(kThreads) void k_hash_scatter(Geo g, const float4* __restrict__ pred,
                                                           const uint32_t* __restrict__ type_flag, uint32_t n,
                                                           uint32_t* __restrict__ cell_off, uint32_t* __restrict__ sorted) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  bool valid = i < n;
  uint32_t key = 0;
  if (valid) {
    if (type_flag != nullptr && type_flag[i] == NB_HASH_TYPE_UNUSED) valid = false;
    else key = hash_cell(g, pred[i]);
  }
  const uint32_t slot = wave_add(cell_off, key, valid);
  if (valid) sorted[slot] = i;
}

// The scatter of particles whose places in their cells are kept, into END offsets:
// a read of the cell's line where k_hash_scatter's atomic moves it there and back.
// For builds that take scratch from the allocator anyway (4 bytes a particle more):
// whole builds of 2,000,003 particles in no order in 256 x 128 x 200 cells 282 -> 215
// us, 1,000,000 in 128^3 146 -> 110, 300,000 67 -> 59, 100,000 48 -> 47;
// in the order of their cells 148 -> 137, 66 -> 59, 200,000 50 -> 53.
__global__ __launch_bounds__(kThreads) void k_hash_place(Geo g, const float4* __restrict__ pred,
                                                         const uint32_t* __restrict__ type_flag, uint32_t n,
                                                         const uint32_t* __restrict__ cell_off,
                                                         const uint32_t* __restrict__ rank, uint32_t* __restrict__ sorted) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= n || (type_flag != nullptr && type_flag[i] == NB_HASH_TYPE_UNUSED)) return;
  sorted[cell_off[hash_cell(g, pred[i])] - 1u - rank[i]] = i;
}

// ascending sort of the first W of v by odd-even transposition (W even)
template <uint32_t W>
__device__ __forceinline__ void sort_net(uint32_t (&v)[kSmall]) {
#pragma unroll
  for (uint32_t r = 0; r < W; r++) {
#pragma unroll
    for (uint32_t k = r & 1u; k + 1 < W; k += 2) {
      const uint32_t a = v[k], b = v[k + 1];
      v[k] = min(a, b);
      v[k + 1] = max(a, b);
    }
  }
}

template <uint32_t W>
__device__ __forceinline__ void sort_small(uint32_t* __restrict__ seg, uint32_t cnt) {
  uint32_t v[kSmall];
#pragma unroll
  for (uint32_t k = 0; k < W; k++) v[k] = k < cnt ? seg[k] : 0xFFFFFFFFu;
  sort_net<W>(v);
#pragma unroll
  for (uint32_t k = 0; k < W; k++)
    if (k < cnt) seg[k] = v[k];
}

// a crowded cell of up to kWaveSort particles, by its wave
__device__ __forceinline__ void wave_sort_cell_of(uint32_t* __restrict__ seg, uint32_t cnt) {
  if (cnt <= 64u) nb::group_sort_segment<64, 1>(seg, cnt);
  else if (cnt <= 256u) nb::group_sort_segment<64, 4>(seg, cnt);
  else nb::group_sort_segment<64, 8>(seg, cnt);
}

// Without a list the crowded cells are found from `sorted` itself: a cell of more than
// `step` particles has some at a multiple of step, the first of which is its own, so
// one lane a multiple looks its particle's cell up.  That deals the cells out by the
// particles they hold, whatever part of the grid is crowded.  (A place read while its
// cell is being sorted holds some particle of the same cell.)  Count, cell and start of
// the cell whose first multiple of step the place `at` is, else 0.
__device__ __forceinline__ uint32_t crowded_at(const Geo& g, const float4* __restrict__ pred,
                                               const uint32_t* __restrict__ cell_count,
                                               const uint32_t* __restrict__ cell_off, const uint32_t* sorted,
                                               uint64_t at, uint32_t used, uint32_t step, uint32_t& c, uint32_t& start) {
  c = start = 0u;
  if (at >= used) return 0u;
  c = hash_cell(g, pred[sorted[at]]);
  const uint32_t cnt = cell_count[c];
  start = cell_off[c] - cnt;
  return at - start < step ? cnt : 0u;
}
// the cells of kSmall to kWaveSort at the lanes' places, one after the other by the wave
__device__ __forceinline__ void sort_crowded_at(const Geo& g, const float4* __restrict__ pred,
                                                const uint32_t* __restrict__ cell_count,
                                                const uint32_t* __restrict__ cell_off, uint32_t* sorted, uint64_t at,
                                                uint32_t used) {
  uint32_t c, start;
  const uint32_t cnt = crowded_at(g, pred, cell_count, cell_off, sorted, at, used, kSmall, c, start);
  uint64_t mid = __ballot(cnt > kSmall && cnt <= kWaveSort);
  while (mid) {
    const int l = __ffsll((unsigned long long)mid) - 1;
    mid &= mid - 1ull;
    wave_sort_cell_of(sorted + uint32_t(__builtin_amdgcn_readlane(int(start), l)),
                      uint32_t(__builtin_amdgcn_readlane(int(cnt), l)));
  }
}

// One thread per cell, or per V = 4 consecutive cells where most are empty:
// the counts then come in 16-byte loads and the offsets are read only beside a
// cell that needs them.  Crowded cells of up to kWaveSort particles: with a list, a
// wave sorts the few it meets itself, one after the other, and lists more; without, the
// waves of the launch's first find_blocks blocks find them, `lanes` lanes of each at a
// multiple of kSmall.  (Sorted by the wave that meets them, however many: 165 us for
// 200,000 particles of which the cells hold 37 each, 120 for 8^3 cells of 64, 64 for
// 2,000 particles in 4^3 cells.)
template <uint32_t V, bool LIST>
__global__ __launch_bounds__(kThreads) void k_hash_stabilize(Geo g, const float4* __restrict__ pred,
                                                             const uint32_t* __restrict__ cell_count,
                                                             const uint32_t* __restrict__ cell_off, uint32_t nc,
                                                             uint32_t* sorted, uint32_t* __restrict__ scratch,
                                                             uint32_t find_blocks, uint32_t lanes) {
  if (!LIST && blockIdx.x < find_blocks) {
    const uint32_t lane = threadIdx.x & 63u, wave = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    const uint64_t at = lane < lanes ? (uint64_t(wave) * lanes + lane) * kSmall : ~0ull;
    sort_crowded_at(g, pred, cell_count, cell_off, sorted, at, cell_off[nc - 1u]);
    return;
  }
  const uint32_t c0 = ((LIST ? blockIdx.x : blockIdx.x - find_blocks) * kThreads + threadIdx.x) * V;
  uint32_t n[V];
  if (V == 4u && c0 + 4u <= nc && (reinterpret_cast<uintptr_t>(cell_count) & 15u) == 0u) {
    const uint4 q = *reinterpret_cast<const uint4*>(cell_count + c0);
    n[0] = q.x; n[V > 1 ? 1 : 0] = q.y; n[V > 2 ? 2 : 0] = q.z; n[V > 3 ? 3 : 0] = q.w;
  } else {
#pragma unroll
    for (uint32_t k = 0; k < V; k++) n[k] = c0 + k < nc ? cell_count[c0 + k] : 0u;
  }
#pragma unroll
  for (uint32_t k = 0; k < V; k++) {
    const uint32_t cnt = n[k];
    if (!__any(cnt >= 2u)) continue;
    const uint32_t start = cnt >= 2u ? cell_off[c0 + k] - cnt : 0u;
    if (LIST) {
      uint64_t mid = __ballot(cnt > kSmall && cnt <= kWaveSort);
      const bool few = uint32_t(__popcll(mid)) <= kWaveCells / V;
      const bool listed = cnt > kWaveSort || (!few && cnt > kSmall);
      const uint64_t list = __ballot(listed);
      if (list) {
        const uint32_t lane = threadIdx.x & 63u, first = uint32_t(__ffsll((unsigned long long)list)) - 1u;
        uint32_t at = 0;
        if (lane == first) at = atomicAdd(&scratch[kOffCrowdCount], uint32_t(__popcll(list)));
        at = uint32_t(__builtin_amdgcn_readlane(int(at), int(first))) + uint32_t(__popcll(list & ((1ull << lane) - 1ull)));
        if (listed && at < kCrowdCap) scratch[kOffCrowdList + at] = c0 + k;
      }
      while (few && mid) {
        const int l = __ffsll((unsigned long long)mid) - 1;
        mid &= mid - 1ull;
        wave_sort_cell_of(sorted + uint32_t(__builtin_amdgcn_readlane(int(start), l)),
                          uint32_t(__builtin_amdgcn_readlane(int(cnt), l)));
      }
    }
    const bool small = cnt >= 2u && cnt <= kSmall;
    // network width: the widest small cell of the wave
    const bool w8 = __any(small && cnt > 4u), w16 = __any(small && cnt > 8u);
    if (small) {
      uint32_t* seg = sorted + start;
      if (w16) sort_small<16>(seg, cnt);
      else if (w8) sort_small<8>(seg, cnt);
      else sort_small<4>(seg, cnt);
    }
  }
}

__device__ void sort_crowded(uint32_t* __restrict__ sorted, const uint32_t* __restrict__ cell_count,
                             const uint32_t* __restrict__ cell_off, uint32_t c, uint32_t* s_buf) {
  const uint32_t cnt = cell_count[c];
  uint32_t* seg = sorted + (cell_off[c] - cnt);
  uint32_t P = 1;
  while (P < cnt) P <<= 1;
  if (cnt <= kLdsSort) {
    for (uint32_t k = threadIdx.x; k < P; k += blockDim.x) s_buf[k] = k < cnt ? seg[k] : 0xFFFFFFFFu;
    __syncthreads();
    nb::block_bitonic(s_buf, P, P);
    for (uint32_t k = threadIdx.x; k < cnt; k += blockDim.x) seg[k] = s_buf[k];
  } else {
    nb::block_bitonic(seg, cnt, P);
  }
  __syncthreads();
}

// The crowded cells that are left.  LIST: those k_hash_stabilize listed, up to
// kWaveSort particles one per wave, larger ones one per block.  Without a list the
// larger ones alone, and all of them when the list overflowed: a block takes a stretch
// of places and the cells that crowded_at finds there.
template <bool LIST>
__global__ __launch_bounds__(kCrowdThreads) void k_hash_crowded(Geo g, const float4* __restrict__ pred,
                                                                const uint32_t* __restrict__ cell_count,
                                                                const uint32_t* __restrict__ cell_off, uint32_t nc,
                                                                uint32_t* sorted, const uint32_t* __restrict__ scratch) {
  __shared__ uint32_t s_buf[kLdsSort];
  __shared__ uint32_t s_list[kCrowdThreads];
  __shared__ uint32_t s_n;
  static_assert(kWaveSort >= kBigStep && kBigStep % kSmall == 0u, "a multiple of the step in each");
  if (LIST) {
    const uint32_t m = scratch[kOffCrowdCount];
    if (m <= kCrowdCap) {
      for (uint32_t e = blockIdx.x + (threadIdx.x >> 6) * gridDim.x; e < m; e += (kCrowdThreads / 64) * gridDim.x) {
        const uint32_t c = uint32_t(__builtin_amdgcn_readfirstlane(int(scratch[kOffCrowdList + e]))), cnt = cell_count[c];
        if (cnt <= kWaveSort) wave_sort_cell_of(sorted + (cell_off[c] - cnt), cnt);
      }
      for (uint32_t e = blockIdx.x; e < m; e += gridDim.x) {
        const uint32_t c = scratch[kOffCrowdList + e];
        if (cell_count[c] > kWaveSort) sort_crowded(sorted, cell_count, cell_off, c, s_buf);
      }
      return;
    }
  }
  const uint32_t used = cell_off[nc - 1u];
  const uint32_t steps = used / kBigStep + (used % kBigStep ? 1u : 0u), per = (steps + gridDim.x - 1u) / gridDim.x;
  const uint64_t first = uint64_t(blockIdx.x) * per * kBigStep;
  if (LIST) {
    for (uint64_t x = threadIdx.x & ~63u; x < uint64_t(per) * (kBigStep / kSmall); x += kCrowdThreads) {
      const uint64_t y = x + (threadIdx.x & 63u);
      sort_crowded_at(g, pred, cell_count, cell_off, sorted,
                      y < uint64_t(per) * (kBigStep / kSmall) ? first + y * kSmall : ~0ull, used);
    }
  }
  for (uint32_t w = 0; w < per; w += kCrowdThreads) {
    if (threadIdx.x == 0u) s_n = 0u;
    __syncthreads();
    uint32_t c, start;
    const uint32_t v = w + threadIdx.x;
    const uint32_t cnt = crowded_at(g, pred, cell_count, cell_off, sorted, v < per ? first + uint64_t(v) * kBigStep : ~0ull,
                                    used, kBigStep, c, start);
    if (cnt > kWaveSort) s_list[atomicAdd(&s_n, 1u)] = c;
    __syncthreads();
    const uint32_t k = s_n;
    for (uint32_t e = 0; e < k; e++) sort_crowded(sorted, cell_count, cell_off, s_list[e], s_buf);
    __syncthreads();
  }
}

}  // namespace nbh

namespace nb {

uint32_t hash_scratch_words() { return nbh::kScratchWords; }

// Checks the arguments of a hash build (no device work); NB_OK or an error.
int validate_hash_build(const nb_hash_grid* grid, const float* pred_pos4, uint32_t n, const uint32_t* cell_count,
                        const uint32_t* cell_offset, const uint32_t* sorted) {
  if (!grid) return set_error(NB_ERR_ARG, "nb_hash_build: null grid");
  uint32_t maxr = 1;
  for (int a = 0; a < 3; a++) {
    if (grid->grid_res[a] == 0u || grid->grid_res[a] > 1024u)
      return set_error(NB_ERR_ARG, "nb_hash_build: grid_res[%d] = %u is outside [1, 1024]", a, grid->grid_res[a]);
    maxr = grid->grid_res[a] > maxr ? grid->grid_res[a] : maxr;
  }
  uint32_t cube = 1;
  while (cube < maxr) cube <<= 1;
  const uint64_t nc64 = uint64_t(cube) * cube * cube;
  if (uint64_t(grid->hash_cells) != nc64)
    return set_error(NB_ERR_ARG, "nb_hash_build: hash_cells = %u, expected %llu (the Morton cube of grid_res)",
                     grid->hash_cells, (unsigned long long)nc64);
  if (!(grid->cell_size > 0.f)) return set_error(NB_ERR_ARG, "nb_hash_build: cell_size must be positive");
  if (!cell_count || !cell_offset || (n && (!pred_pos4 || !sorted)))
    return set_error(NB_ERR_ARG, "nb_hash_build: null buffer");
  if (reinterpret_cast<uintptr_t>(pred_pos4) & 15u)
    return set_error(NB_ERR_ARG, "nb_hash_build: pred_pos4 must be 16-byte aligned (float4)");
  return NB_OK;
}

// Whether a build needs no scratch: the chunks' sums stand in cell_offset until the
// offsets do (at most 64 of them, and a chunk that has another before it is whole,
// hash_cells being a power of two), and the crowded pass finds its cells by itself (its
// counts, 1 MB at most, stay in the L2s).  Taking scratch from the stream-ordered
// allocator and giving it back costs 25 us of host time, as much as all of a
// small build: 32,768 particles in 64^3 cells took 48 us with it and take
// 27 without.
bool hash_needs_no_scratch(const nb_hash_grid* grid) { return grid->hash_cells <= (1u << 18); }

// Enqueues a validated hash build with the given scratch (hash_scratch_words()
// uint32 of device memory; null when hash_needs_no_scratch) and, or null, n words
// for the particles' places in their cells.
int enqueue_hash_build(const nb_hash_grid* grid, const float* pred_pos4, const uint32_t* type_flag, uint32_t n,
                       uint32_t* cell_count, uint32_t* cell_offset, uint32_t* sorted, uint32_t* scratch,
                       uint32_t* rank, hipStream_t s) {
  using namespace nbh;
  const uint32_t nc = grid->hash_cells;
  Geo g{};
  for (int a = 0; a < 3; a++) {
    g.wmin[a] = grid->world_min[a];
    g.gmax[a] = float(grid->grid_res[a]) - 1.f;
  }
  g.h = grid->cell_size;
  const float4* pred = reinterpret_cast<const float4*>(pred_pos4);
  const uint32_t nchunks = (nc + kChunk - 1u) / kChunk;
  const uint32_t pblocks = uint32_t((uint64_t(n) + kThreads - 1u) / kThreads);
  const bool sums = nchunks <= kSumChunks;
  // four cells a thread where most cells are empty and their counts are
  // bandwidth (16.8 M cells, 2 M particles: 22 us against 38); in a small hash
  // the four turns of a thread are latency (262,144 cells, 32,768 particles: 9.8
  // against 4.6)
  const uint32_t vec = nc / 4u > n && nc >= (1u << 22) ? 4u : 1u;
  const uint32_t cblocks = (nc + vec * kThreads - 1u) / (vec * kThreads);
  hipLaunchKernelGGL(k_hash_clear, dim3(std::min<uint32_t>((nc / 4u + kThreads - 1u) / kThreads + 1u, 8192u)),
                     dim3(kThreads), 0, s, cell_count, nc, scratch);
  if (n && rank)
    hipLaunchKernelGGL(k_hash_count<true>, dim3(pblocks), dim3(kThreads), 0, s, g, pred, type_flag, n, cell_count, rank);
  else if (n)
    hipLaunchKernelGGL(k_hash_count<false>, dim3(pblocks), dim3(kThreads), 0, s, g, pred, type_flag, n, cell_count, rank);
  if (scratch)
    hipLaunchKernelGGL(k_hash_chunk_sums<false>, dim3(nchunks), dim3(kThreads), 0, s, cell_count, nc, scratch);
  else if (nchunks > 1u)
    hipLaunchKernelGGL(k_hash_chunk_sums<true>, dim3(nchunks), dim3(kThreads), 0, s, cell_count, nc, cell_offset);
  if (!sums) hipLaunchKernelGGL(k_hash_chunk_scan, dim3(1), dim3(1024), 0, s, scratch, nchunks);
#define NB_OFFSETS(FR, EN)                                                                                            \
  hipLaunchKernelGGL((k_hash_offsets<Base::FR, EN>), dim3(nchunks), dim3(kThreads), 0, s, cell_count, nc, scratch, \
                     cell_offset)
  if (!scratch) {
    NB_OFFSETS(OWN, false);
  } else if (sums) {
    if (rank) NB_OFFSETS(SUMS, true); else NB_OFFSETS(SUMS, false);
  } else {
    if (rank) NB_OFFSETS(SCAN, true); else NB_OFFSETS(SCAN, false);
  }
#undef NB_OFFSETS
  if (n) {
    if (rank)
      hipLaunchKernelGGL(k_hash_place, dim3(pblocks), dim3(kThreads), 0, s, g, pred, type_flag, n, cell_offset, rank,
                         sorted);
    else
      hipLaunchKernelGGL(k_hash_scatter, dim3(pblocks), dim3(kThreads), 0, s, g, pred, type_flag, n, cell_offset, sorted);
    // few lanes a wave while there are waves to spare
    const uint32_t lanes = n <= (1u << 16) ? 4u : (n <= (1u << 18) ? 16u : 64u);
    const uint32_t find_blocks = scratch ? 0u : (n - 1u) / (nbh::kThreads / 64u * lanes * kSmall) + 1u;
#define NB_STABILIZE(VC, LI)                                                                                           \
  hipLaunchKernelGGL((k_hash_stabilize<VC, LI>), dim3(cblocks + find_blocks), dim3(kThreads), 0, s, g, pred, cell_count, \
                     cell_offset, nc, sorted, scratch, find_blocks, lanes)
    // 64 KB of LDS a block: two fit a CU, so 512 blocks run at once; twice as many
    // where most cells are large, so that each is alone in a block's stretch (2,000,003
    // particles in 8^3 cells: 102 us against 150; else the empty ones cost 2 us)
    const uint32_t crowd_blocks = std::min((n - 1u) / kWaveSort + 1u, !scratch && n / kWaveSort >= nc ? 1024u : 512u);
#define NB_CROWDED(LI)                                                                                              \
  hipLaunchKernelGGL(k_hash_crowded<LI>, dim3(crowd_blocks), dim3(kCrowdThreads), 0, s, g, pred, cell_count,        \
                     cell_offset, nc, sorted, scratch)
    if (!scratch) {
      NB_STABILIZE(1, false);
      NB_CROWDED(false);
    } else {
      if (vec == 4u) NB_STABILIZE(4, true); else NB_STABILIZE(1, true);
      NB_CROWDED(true);
    }
#undef NB_STABILIZE
#undef NB_CROWDED
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(NB_ERR_HIP, "nb_hash_build: launch failed: %s", hipGetErrorString(e));
  return NB_OK;
}

}  // namespace nb

extern "C" int nb_hash_build(const nb_hash_grid* grid, const float* pred_pos4, const uint32_t* type_flag, uint32_t n,
                             uint32_t* cell_count, uint32_t* cell_offset, uint32_t* sorted, void* hip_stream) {
  const int v = nb::validate_hash_build(grid, pred_pos4, n, cell_count, cell_offset, sorted);
  if (v != NB_OK) return v;
  hipStream_t s = static_cast<hipStream_t>(hip_stream);
  if (nb::hash_needs_no_scratch(grid))
    return nb::enqueue_hash_build(grid, pred_pos4, type_flag, n, cell_count, cell_offset, sorted, nullptr, nullptr, s);
  void* scratch = nullptr;
  // with room for the particles' places in their cells, or, where there is none,
  // without
  bool ranked = n != 0u;
  hipError_t e = hipMallocAsync(&scratch, (size_t(nb::hash_scratch_words()) + n) * 4u, s);
  if (e != hipSuccess && ranked) {
    (void)hipGetLastError();
    ranked = false;
    e = hipMallocAsync(&scratch, size_t(nb::hash_scratch_words()) * 4u, s);
  }
  if (e != hipSuccess) return nb::set_error(NB_ERR_HIP, "nb_hash_build: hipMallocAsync failed: %s", hipGetErrorString(e));
  const int rc = nb::enqueue_hash_build(grid, pred_pos4, type_flag, n, cell_count, cell_offset, sorted,
                                        static_cast<uint32_t*>(scratch),
                                        ranked ? static_cast<uint32_t*>(scratch) + nb::hash_scratch_words() : nullptr, s);
  e = hipFreeAsync(scratch, s);
  if (rc != NB_OK) return rc;
  if (e != hipSuccess) return nb::set_error(NB_ERR_HIP, "nb_hash_build: hipFreeAsync failed: %s", hipGetErrorString(e));
  return NB_OK;
}

// ---- nb_hash_build_noalloc: the same build on a file-scope scratch array ----
// The array lives in every GPU's copy of this code object.  Host code never
// passes its name to a kernel (on the host the name is a stand-in, not a
// device address): the device address comes from hipGetSymbolAddress, once per
// device, with that device current, and is kept per device.
#include <mutex>

namespace nbh_noalloc {

static __device__ __align__(256) uint32_t scratch[nbh::kScratchWords];
static_assert(sizeof(uint32_t) * nbh::kScratchWords == NB_HASH_NOALLOC_SCRATCH_BYTES,
              "NB_HASH_NOALLOC_SCRATCH_BYTES must equal the scratch the build uses");

constexpr int kMaxDevices = 64;
static std::mutex g_mu;
static uint32_t* g_ptr[kMaxDevices] = {};

// The current device's address of `scratch` into *out (looked up on the
// device's first use); NB_OK or an error code with the message set.
static int device_scratch(uint32_t** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess)
    return nb::set_error(NB_ERR_HIP, "nb_hash_build_noalloc: hipGetDevice failed: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return nb::set_error(NB_ERR_RANGE, "nb_hash_build_noalloc: device %d is beyond the %d this library serves", dev,
                         kMaxDevices);
  std::lock_guard<std::mutex> lock(g_mu);
  if (!g_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return nb::set_error(NB_ERR_HIP, "nb_hash_build_noalloc: hipGetSymbolAddress of the scratch array failed: %s",
                           hipGetErrorString(e));
    g_ptr[dev] = static_cast<uint32_t*>(p);
  }
  *out = g_ptr[dev];
  return NB_OK;
}

}  // namespace nbh_noalloc

extern "C" int nb_hash_build_noalloc(const nb_hash_grid* grid, const float* pred_pos4, const uint32_t* type_flag,
                                     uint32_t n, uint32_t* cell_count, uint32_t* cell_offset, uint32_t* sorted,
                                     void* hip_stream) {
  // validate_hash_build refuses any hash_cells other than the Morton cube of
  // a grid of at most 1024 per axis, so hash_cells <= NB_HASH_MAX_CELLS, the
  // largest hash the array's chunk sums cover; checked again here because the
  // array's size depends on it.
  const int v = nb::validate_hash_build(grid, pred_pos4, n, cell_count, cell_offset, sorted);
  if (v != NB_OK) return v;
  if (grid->hash_cells > NB_HASH_MAX_CELLS)
    return nb::set_error(NB_ERR_ARG, "nb_hash_build_noalloc: hash_cells = %u exceeds the scratch array's %u",
                         grid->hash_cells, NB_HASH_MAX_CELLS);
  if (nb::hash_needs_no_scratch(grid))
    return nb::enqueue_hash_build(grid, pred_pos4, type_flag, n, cell_count, cell_offset, sorted, nullptr, nullptr,
                                  static_cast<hipStream_t>(hip_stream));
  uint32_t* s = nullptr;
  const int rc = nbh_noalloc::device_scratch(&s);
  if (rc != NB_OK) return rc;
  return nb::enqueue_hash_build(grid, pred_pos4, type_flag, n, cell_count, cell_offset, sorted, s, nullptr,
                                static_cast<hipStream_t>(hip_stream));
}
