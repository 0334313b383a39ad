// nb_kernel_util.hpp — device helpers shared by the substep kernels
// (mpm_kernels.hip) and their adjoints (mpm_adjoint.hip): tile coordinates,
// block scans, the XCD-aware chunk map, cell keys, the per-axis B-spline
// stencil, and the SDF / analytic-collider boundary functions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nb_device_math.hpp"
#include "nb_engine.hpp"

namespace nb {

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ void tile_coords(uint32_t T, int& tx, int& ty, int& tz) {
  tx = int(morton_compact(T));
  ty = int(morton_compact(T >> 1));
  tz = int(morton_compact(T >> 2));
}

// Exclusive scan across a block of BS threads (BS a multiple of 64) of a
// 32- or 64-bit unsigned value.  s_wave must hold BS/64 + 1 values.  Returns
// the exclusive prefix; *total is the block sum.  Contains barriers: call from
// uniform control flow.
template <int BS, class T>
__device__ __forceinline__ T block_exclusive_scan(T v, T* s_wave, T& total) {
  constexpr int NW = BS / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  T x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    T y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) s_wave[wave] = x;
  __syncthreads();
  if (wave == 0) {
    T w = lane < NW ? s_wave[lane] : T(0);
    T ws = w;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      T y = __shfl_up(ws, d);
      if (lane >= d) ws += y;
    }
    if (lane < NW) s_wave[lane] = ws - w;
    if (lane == NW - 1) s_wave[NW] = ws;
  }
  __syncthreads();
  T excl = x - v + s_wave[wave];
  total = s_wave[NW];
  __syncthreads();
  return excl;
}

// Three 64-bit scans with one set of barriers; s must hold 3 (BS/64 + 1) values.
template <int BS>
__device__ __forceinline__ void block_exclusive_scan3(const uint64_t (&v)[3], uint64_t* s, uint64_t (&excl)[3],
                                                      uint64_t (&total)[3]) {
  constexpr int NW = BS / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t x[3] = {v[0], v[1], v[2]};
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
    for (int q = 0; q < 3; q++) {
      const uint64_t y = __shfl_up(x[q], d);
      if (lane >= d) x[q] += y;
    }
  }
  if (lane == 63) {
#pragma unroll
    for (int q = 0; q < 3; q++) s[q * (NW + 1) + wave] = x[q];
  }
  __syncthreads();
  if (wave < 3) {  // wave q scans the waves' sums of value q
    uint64_t* w = s + wave * (NW + 1);
    const uint64_t own = lane < NW ? w[lane] : 0u;
    uint64_t run = own;
#pragma unroll
    for (int d = 1; d < NW; d <<= 1) {
      const uint64_t y = __shfl_up(run, d);
      if (lane >= d) run += y;
    }
    if (lane < NW) w[lane] = run - own;
    if (lane == NW - 1) w[NW] = run;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 3; q++) {
    excl[q] = x[q] - v[q] + s[q * (NW + 1) + wave];
    total[q] = s[q * (NW + 1) + NW];
  }
}

// Ascending sort of seg[0, cnt), cnt <= G E, by G neighbouring lanes (a power of two),
// E registers each: value e in register e / G of the group's lane e % G.  Bitonic: a step
// of G or more pairs values of one lane.  All groups of a wave call it together (cnt 0:
// none).
template <uint32_t G, uint32_t E>
__device__ __forceinline__ void group_sort_segment(uint32_t* seg, uint32_t cnt) {
  const uint32_t lane = threadIdx.x & (G - 1u);
  uint32_t v[E];
#pragma unroll
  for (uint32_t e = 0; e < E; e++) v[e] = G * e + lane < cnt ? seg[G * e + lane] : 0xFFFFFFFFu;
#pragma unroll
  for (uint32_t k = 2; k <= G * E; k <<= 1) {
#pragma unroll
    for (uint32_t j = k >> 1; j >= 1u; j >>= 1) {
#pragma unroll
      for (uint32_t e = 0; e < E; e++) {
        const uint32_t at = G * e + lane;
        const bool up = (at & k) == 0u;
        if (j >= G) {
          const uint32_t f = e ^ (j / G);
          if (f > e) {
            const uint32_t lo = min(v[e], v[f]), hi = max(v[e], v[f]);
            v[e] = up ? lo : hi;
            v[f] = up ? hi : lo;
          }
        } else {
          const uint32_t o = uint32_t(__shfl_xor(int(v[e]), int(j)));
          v[e] = up == ((at & j) == 0u) ? min(v[e], o) : max(v[e], o);
        }
      }
    }
  }
#pragma unroll
  for (uint32_t e = 0; e < E; e++)
    if (G * e + lane < cnt) seg[G * e + lane] = v[e];
}

// Bitonic sort (ascending) of a[0, cnt) over the padded length P (a power of
// two >= cnt), every merge in its "flip" form so that all compare-exchanges put
// the smaller value first: partners at or past cnt hold +inf and are skipped.
// Block-cooperative; a is LDS or global memory of this block alone.
__device__ __forceinline__ void compare_exchange(uint32_t* a, uint32_t i, uint32_t l, uint32_t cnt) {
  if (l < cnt) {
    const uint32_t x = a[i], y = a[l];
    if (x > y) {
      a[i] = y;
      a[l] = x;
    }
  }
}
__device__ inline void block_bitonic(uint32_t* a, uint32_t cnt, uint32_t P) {
  const uint32_t half = P >> 1;
  for (uint32_t k = 2; k <= P; k <<= 1) {
    const uint32_t hk = k >> 1;
    for (uint32_t t = threadIdx.x; t < half; t += blockDim.x) {
      const uint32_t b = (t / hk) * k, o = t % hk;
      compare_exchange(a, b + o, b + k - 1u - o, cnt);
    }
    __syncthreads();
    for (uint32_t j = k >> 2; j >= 1u; j >>= 1) {
      for (uint32_t t = threadIdx.x; t < half; t += blockDim.x) {
        const uint32_t i = (t / j) * (2u * j) + (t % j);
        compare_exchange(a, i, i + j, cnt);
      }
      __syncthreads();
    }
  }
}

// Workgroups are dealt to the 8 XCDs (each with its own L2) round-robin by
// id.  Block b is given chunk xcd_chunk(b, nb) of the work, so that each XCD
// walks one contiguous eighth of the chunks: neighbouring particles, and the
// grid nodes they share, stay in one L2.  A bijection of [0, nb).
constexpr uint32_t kXCDs = 8;
__device__ __forceinline__ uint32_t xcd_chunk(uint32_t b, uint32_t nb) {
  const uint32_t x = b % kXCDs, i = b / kXCDs, q = nb / kXCDs, r = nb % kXCDs;
  return x < r ? x * (q + 1u) + i : r * (q + 1u) + (x - r) * q + i;
}

// ---- scene geometry ----
// the plain engine's one scene, from the kernel arguments (stays in scalar registers)
__device__ __forceinline__ SceneGeo geo_of(const SubParams& p) {
  SceneGeo g;
  g.h = p.h;
  g.inv_h = 1.f / p.h;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    g.wmin[a] = p.wmin[a];
    g.wmax[a] = p.wmax[a];
    g.grid_res[a] = p.grid_res[a];
  }
  g.cube_res = p.cube_res;
  g.tile_dim = p.tile_dim;
  g.key_base = 0u;
  g.h_pow2 = p.h_pow2;
  g.pad = 0u;
  return g;
}
// the scene of tile T (uniform across a block) and of particle q
template <bool BATCH>
__device__ __forceinline__ SceneGeo tile_geo(const SubParams& p, uint32_t T) {
  if constexpr (BATCH) return p.scenes[p.tile_scene[T]];
  else return geo_of(p);
}
template <bool BATCH>
__device__ __forceinline__ SceneGeo particle_geo(const SubParams& p, uint32_t q) {
  if constexpr (BATCH) return p.scenes[p.pscene[q]];
  else return geo_of(p);
}
// tile coordinates within the scene's cube, and the tile id of coordinates
__device__ __forceinline__ void tile_coords(const SceneGeo& g, uint32_t T, int& tx, int& ty, int& tz) {
  tile_coords(T - (g.key_base >> kTileBits), tx, ty, tz);
}
__device__ __forceinline__ uint32_t tile_id(const SceneGeo& g, int tx, int ty, int tz) {
  return (g.key_base >> kTileBits) + morton3(uint32_t(tx), uint32_t(ty), uint32_t(tz));
}
// The nodes of the grid, tile by occupied tile.  A node lies in some particle's
// stencil when an occupied tile's 10^3 box covers it.  The block of an occupied
// tile takes its tile's 512 nodes (thread t the t-th in Morton order), then those
// of the 488 nodes around them whose own tile is not occupied and that no occupied
// tile before it (z, y, x ascending) covers: each covered node once.  A block per
// tile that any box reaches spent most of its threads on nodes that none covers, and
// read the covering boxes one after the other.  Now bound by the latency of
// a tile's list entries and boxes, then by memory: 43 -> 20 us for the 1,279
// occupied tiles of 64 small scenes, 47 -> 36 for 2,385 of a terrain (4.19 M
// particles), 18 -> 12 for 300 of 16 scenes (backward 20 -> 11).  Up to
// kGridSplitTiles tiles, where blocks are few, a tile's own nodes and those around
// it are two blocks: 7.6 -> 6.2 us at 128 tiles, even at 1,279 (20.3 / 21.5), 36 ->
// 40 at 2,385.
constexpr uint32_t kGridSplitTiles = 512;
struct NeighbourTiles {
  int32_t act[27];  // index of the occupied tile, -1: not occupied, -2: outside the cube
  uint32_t open;    // some neighbour is not occupied
};

// Called by the whole block; n is in LDS.
__device__ __forceinline__ void load_neighbours(const SceneGeo& g, int tx, int ty, int tz,
                                                const int32_t* __restrict__ tile_act, NeighbourTiles& n) {
  __syncthreads();
  if (threadIdx.x < 64u) {
    int32_t v = -2;
    if (threadIdx.x < 27u) {
      const int e = int(threadIdx.x), td = int(g.tile_dim);
      const int sx = tx + e % 3 - 1, sy = ty + (e / 3) % 3 - 1, sz = tz + e / 9 - 1;
      if (uint32_t(sx) < uint32_t(td) && uint32_t(sy) < uint32_t(td) && uint32_t(sz) < uint32_t(td))
        v = max(tile_act[tile_id(g, sx, sy, sz)], -1);
      n.act[e] = v;
    }
    const bool open = __any(v == -1);
    if (threadIdx.x == 0u) n.open = open;
  }
  __syncthreads();
}

// Box coordinates of the node this thread takes: its tile's own (shell = false) or
// one around it; false when it takes none.
__device__ __forceinline__ bool box_node(bool shell, int& bx, int& by, int& bz) {
  const int t = int(threadIdx.x);
  if (!shell) {
    bx = int(morton_compact(threadIdx.x)) + 1;
    by = int(morton_compact(threadIdx.x >> 1)) + 1;
    bz = int(morton_compact(threadIdx.x >> 2)) + 1;
    return true;
  }
  if (t < 200) {  // the layers z = 0 and z = 9
    bz = t < 100 ? 0 : 9;
    by = (t % 100) / 10;
    bx = t % 10;
    return true;
  }
  const int r = (t - 200) % 36;  // the rings between them
  bz = 1 + (t - 200) / 36;
  by = r < 10 ? 0 : (r < 20 ? 9 : 1 + (r - 20) % 8);
  bx = r < 20 ? r % 10 : (r < 28 ? 0 : 9);
  return t < 488;
}

// Sum of the boxes that cover the node at box coordinates (bx, by, bz) of the tile
// whose neighbours are n, tile by tile (z, y, x ascending); false when the node is
// another block's.  The boxes' loads are independent: all are in flight together.
__device__ __forceinline__ bool sum_boxes(const NeighbourTiles& n, bool shell, int bx, int by, int bz,
                                          const float4* __restrict__ boxes, float4& sum) {
  const int b[3] = {bx, by, bz};
  int lo[3], own = 13;
  bool two[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {  // covered by the tiles lo and, near a face, lo + 1 of the axis
    lo[a] = b[a] <= 1 ? -1 : 0;
    two[a] = b[a] <= 1 || b[a] >= 8;
    own += (b[a] == 0 ? -1 : (b[a] == 9 ? 1 : 0)) * (a == 0 ? 1 : (a == 1 ? 3 : 9));
  }
  bool mine = !shell || n.act[own] == -1;
  float4 q[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    q[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    const bool in = (!(k & 1) || two[0]) && (!(k & 2) || two[1]) && (!(k & 4) || two[2]);
    const int ox = lo[0] + (k & 1), oy = lo[1] + ((k >> 1) & 1), oz = lo[2] + (k >> 2);
    const int32_t a = in ? n.act[(oz + 1) * 9 + (oy + 1) * 3 + ox + 1] : -1;
    if (a >= 0) {
      // a tile before this one covers the node
      if (shell && (oz < 0 || (oz == 0 && (oy < 0 || (oy == 0 && ox < 0))))) mine = false;
      if (mine) q[k] = boxes[size_t(a) * kBoxNodes + ((bz - 8 * oz) * kBox + by - 8 * oy) * kBox + bx - 8 * ox];
    }
  }
  sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    sum.x += q[k].x; sum.y += q[k].y; sum.z += q[k].z; sum.w += q[k].w;
  }
  return mine;
}
// With turbulence or noise the nodes of a block share lattice points (tile_forces).
// ROLES = 1: a block takes a tile's own nodes, or those around it, one a thread.
// ROLES = 4: a quarter of its own (8 x 4 x 4), or one face of those around it, four
// threads a node: ten blocks a tile, for scenes of few.  The unit's node t (box
// coordinates, false: none) and the corners of the box its nodes lie in.
constexpr uint32_t kNoiseThreads = 512;
// A tile of a small scene has four quarters and about one face with nodes on it: five
// blocks, on 256 CUs 51 tiles.  Frames of 20 substeps with ROLES 1 / 4, us: 8 tiles
// 1777 / 1558, 12 tiles 1861 / 1653, 48 tiles (57,001 particles) 2116 / 1924, 64 tiles
// 2316 / 2249 and, full, 2644 / 2874, 216 tiles 3881 / 4780.
constexpr uint32_t kNoiseSplitTiles = 51;
template <uint32_t ROLES>
constexpr uint32_t noise_units() { return ROLES == 1u ? 2u : 10u; }
template <uint32_t ROLES>
__device__ __forceinline__ bool noise_shell(uint32_t unit) { return unit >= (ROLES == 1u ? 1u : 4u); }
template <uint32_t ROLES>
__device__ __forceinline__ bool noise_unit_node(uint32_t unit, int t, int (&n)[3], int (&first)[3], int (&last)[3]) {
  if (ROLES == 1u) {
    const bool shell = unit != 0u;
    first[0] = first[1] = first[2] = shell ? 0 : 1;
    last[0] = last[1] = last[2] = shell ? 9 : 8;
    return box_node(shell, n[0], n[1], n[2]);
  }
  if (unit < 4u) {
    const uint32_t m = unit * 128u + uint32_t(t);
    const int hy = 4 * int(unit & 1u), hz = 4 * int(unit >> 1);
    n[0] = int(morton_compact(m)) + 1; n[1] = int(morton_compact(m >> 1)) + 1; n[2] = int(morton_compact(m >> 2)) + 1;
    first[0] = 1; first[1] = 1 + hy; first[2] = 1 + hz;
    last[0] = 8; last[1] = 4 + hy; last[2] = 4 + hz;
    return true;
  }
  const int side = (unit & 1u) ? 9 : 0;
  if (unit < 6u) {  // z = 0, 9
    n[0] = t % 10; n[1] = t / 10; n[2] = side;
    first[0] = first[1] = 0; first[2] = last[2] = side; last[0] = last[1] = 9;
    return t < 100;
  }
  if (unit < 8u) {  // y = 0, 9 between them
    n[0] = t % 10; n[1] = side; n[2] = 1 + t / 10;
    first[0] = 0; first[1] = last[1] = side; first[2] = 1; last[0] = 9; last[2] = 8;
    return t < 80;
  }
  n[0] = side; n[1] = 1 + t % 8; n[2] = 1 + t / 8;  // x = 0, 9 between those
  first[0] = last[0] = side; first[1] = first[2] = 1; last[1] = last[2] = 8;
  return t < 64;
}

// index of node (x, y, z) of the scene in the Morton-ordered node arrays
__device__ __forceinline__ uint32_t node_id(const SceneGeo& g, uint32_t x, uint32_t y, uint32_t z) {
  return g.key_base + morton3(x, y, z);
}

// (x - wmin[a]) / h, the IEEE quotient the reference's cell index takes
// (shaders/mpm_common.glsl:190-195, mpm_g2p.comp:78).  When h is a power of
// two the product with 1/h is the same number (an exact scaling), one
// instruction instead of the division's sequence.
__device__ __forceinline__ float cell_coord(const SceneGeo& g, float x, int a) {
  const float d = x - g.wmin[a];
  if (g.h_pow2) return d * g.inv_h;
  return d / g.h;
}

// cell key of a position: shaders/mpm_common.glsl:190-195 (IEEE quotient,
// clamp to [0, gridRes-1], truncation; NaN maps to 0 as fmaxf returns the
// non-NaN operand), offset by the scene's key base
__device__ __forceinline__ uint32_t cell_key(const SceneGeo& g, float x, float y, float z) {
  float lx = fminf(fmaxf(cell_coord(g, x, 0), 0.f), float(g.grid_res[0]) - 1.f);
  float ly = fminf(fmaxf(cell_coord(g, y, 1), 0.f), float(g.grid_res[1]) - 1.f);
  float lz = fminf(fmaxf(cell_coord(g, z, 2), 0.f), float(g.grid_res[2]) - 1.f);
  return g.key_base + morton3(uint32_t(lx), uint32_t(ly), uint32_t(lz));
}


// Per-axis stencil data of a particle relative to the three nodes c-1, c, c+1.
struct Axis3 {
  float w[3], g[3], dx[3];  // weight, weight derivative / h, x_node - x_p
};

// smallest positive entry (+inf if none)
__device__ __forceinline__ float min_positive3(const float w[3]) {
  const float a = w[0] > 0.f ? w[0] : INFINITY, b = w[1] > 0.f ? w[1] : INFINITY, c = w[2] > 0.f ? w[2] : INFINITY;
  return fminf(a, fminf(b, c));
}

// Quadratic B-spline weight and derivative (shaders/mpm_common.glsl:198-210),
// evaluated with selects instead of branches; inv_h = 1/h replaces the
// division of the derivative by h.
__device__ __forceinline__ void axis_stencil_f(float f, float xp, float wmin, float h, float inv_h, int first_node,
                                               Axis3& a) {
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float nf = float(first_node + i) + 0.5f;
    const float d = f - nf;
    const float ad = fabsf(d);
    const float t = 1.5f - ad;
    const bool in = ad < 0.5f, mid = ad < 1.5f;
    a.w[i] = in ? 0.75f - ad * ad : (mid ? 0.5f * t * t : 0.f);
    a.g[i] = (in ? -2.f * d : (mid ? (d > 0.f ? -t : t) : 0.f)) * inv_h;
    a.dx[i] = nf * h + wmin - xp;
  }
}
// The same stencil for a particle known to lie in cell c (c - 1 the first
// node): when f is in [c, c+1) and c >= 1, the differences f - (c + i - 0.5)
// are exact and fall in [0.5, 1.5), [-0.5, 0.5) and [-1.5, -0.5), so each
// node's piece of the B-spline is fixed and the weights and derivatives come
// out with the bits axis_stencil_f gives, without its compares and selects
// (at the ends of the ranges both pieces give the same values: the spline
// is C1).  Returns false when f is not in that range; a is then not valid.
__device__ __forceinline__ bool axis_stencil_cell(float f, float xp, float wmin, float h, float inv_h, int c,
                                                  Axis3& a) {
  const float n0 = float(c - 1) + 0.5f, n1 = float(c) + 0.5f, n2 = float(c + 1) + 0.5f;
  const float d0 = f - n0, d1 = f - n1, d2 = f - n2;
  const float t0 = 1.5f - d0, t2 = 1.5f + d2;  // 1.5 - |d|
  a.w[0] = 0.5f * t0 * t0;
  a.g[0] = -t0 * inv_h;
  a.w[1] = 0.75f - d1 * d1;
  a.g[1] = (-2.f * d1) * inv_h;
  a.w[2] = 0.5f * t2 * t2;
  a.g[2] = t2 * inv_h;
  a.dx[0] = n0 * h + wmin - xp;
  a.dx[1] = n1 * h + wmin - xp;
  a.dx[2] = n2 * h + wmin - xp;
  return (c >= 1) & (f >= float(c)) & (f < float(c + 1));
}
// f = (x - wmin) / h, the IEEE quotient the cell keys use
__device__ __forceinline__ void axis_stencil(float xp, float wmin, float h, float inv_h, int first_node, Axis3& a) {
  axis_stencil_f((xp - wmin) / h, xp, wmin, h, inv_h, first_node, a);
}

// the dense SDF (plain engine only: Morton order over its cube)
__device__ __forceinline__ float sample_sdf(const float* sdf, const SceneGeo& g, int x, int y, int z) {
  if (x < 0 || y < 0 || z < 0 || x >= g.grid_res[0] || y >= g.grid_res[1] || z >= g.grid_res[2]) return 1e6f;
  return sdf[morton3(x, y, z)];
}

// position of node (nx, ny, nz)
__device__ __forceinline__ float3 node_pos(const SceneGeo& g, int nx, int ny, int nz) {
  return make_float3(fmaf(float(nx) + 0.5f, g.h, g.wmin[0]), fmaf(float(ny) + 0.5f, g.h, g.wmin[1]),
                     fmaf(float(nz) + 0.5f, g.h, g.wmin[2]));
}

__device__ __forceinline__ float len3(float x, float y, float z) { return sqrtf(x * x + y * y + z * z); }

// ---- procedural noise of the turbulence and noise forces ----
// shaders/force_noise.glsl:7-84 with GLSL's fract(x) = x - floor(x),
// mix(a, b, t) = a + (b - a) t and dot summed left to right.  The hash
// fract(sin(a) 43758.5453) turns one rounding step of a into a different
// value, so these functions are compiled without FMA contraction, every
// product and sum rounded as written.  GLSL leaves sin's accuracy to the
// driver; here the hash's sin is the correctly rounded FP32 sine, taken as
// sin in FP64 rounded once to FP32 (any two FP64 sines within an ulp round
// to the same float unless the value lies within 2^-29 ulp of a rounding
// boundary), so every platform that does the same gets the same hash.
__device__ __forceinline__ float hash_sin(float a) { return float(sin(double(a))); }
__device__ __forceinline__ float gl_fract(float x) { return x - floorf(x); }
__device__ __forceinline__ float gl_mix(float a, float b, float t) { return a + (b - a) * t; }
// WIDE: the three sines side by side; else one after the other, in fewer registers
template <bool WIDE>
__device__ __forceinline__ float3 noise_hash33(float x, float y, float z) {  // force_noise.glsl:7-12
#pragma clang fp contract(off)
  const float a = x * 127.1f + y * 311.7f + z * 74.7f;
  const float b = x * 269.5f + y * 183.3f + z * 246.1f;
  const float c = x * 113.5f + y * 271.9f + z * 124.6f;
  if (WIDE)
    return make_float3(-1.f + 2.f * gl_fract(hash_sin(a) * 43758.5453123f),
                       -1.f + 2.f * gl_fract(hash_sin(b) * 43758.5453123f),
                       -1.f + 2.f * gl_fract(hash_sin(c) * 43758.5453123f));
  float h[3];
#pragma unroll 1
  for (int k = 0; k < 3; k++) {
    const float v = -1.f + 2.f * gl_fract(hash_sin(k == 0 ? a : (k == 1 ? b : c)) * 43758.5453123f);
    h[0] = k == 0 ? v : h[0];
    h[1] = k == 1 ? v : h[1];
    h[2] = v;
  }
  return make_float3(h[0], h[1], h[2]);
}
// value noise at (px, py, pz); grad(ox, oy, oz) is the gradient at the corner
// (floor p) + (ox, oy, oz), o in {0, 1}
template <class Grad>
__device__ __forceinline__ float noise_value3_of(float px, float py, float pz, Grad grad) {  // force_noise.glsl:14-37
#pragma clang fp contract(off)
  const float fx = gl_fract(px), fy = gl_fract(py), fz = gl_fract(pz);
  const float ux = fx * fx * (3.f - 2.f * fx), uy = fy * fy * (3.f - 2.f * fy), uz = fz * fz * (3.f - 2.f * fz);
  float n[8];
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const float ox = float(c & 1), oy = float((c >> 1) & 1), oz = float((c >> 2) & 1);
    const float3 g = grad(c & 1, (c >> 1) & 1, (c >> 2) & 1);
    n[c] = g.x * (fx - ox) + g.y * (fy - oy) + g.z * (fz - oz);
  }
  const float nx00 = gl_mix(n[0], n[1], ux), nx10 = gl_mix(n[2], n[3], ux);
  const float nx01 = gl_mix(n[4], n[5], ux), nx11 = gl_mix(n[6], n[7], ux);
  return gl_mix(gl_mix(nx00, nx10, uy), gl_mix(nx01, nx11, uy), uz);
}
// (a call: inlined, its 24 sines would fill the instruction cache of the kernels that
// have it for the lattice ranges that no table holds.  Its sines are side by side, the
// kernels' blocks having the registers: with one after the other six substeps of 65,536
// particles in turbulence of four octaves at 1.25 of a node's spacing took 2.88 ms, and
// take 2.39; of 4,096 strewn over 330 tiles 6.80 and 5.56.)
__device__ __attribute__((noinline)) float noise_value3(float px, float py, float pz) {
#pragma clang fp contract(off)
  const float ix = floorf(px), iy = floorf(py), iz = floorf(pz);
  return noise_value3_of(px, py, pz, [&](int ox, int oy, int oz) {
    return noise_hash33<true>(ix + float(ox), iy + float(oy), iz + float(oz));
  });
}
// The grid's force block (src/core/ForceShaderCompiler.cpp:72-93 for the MPM
// grid, typeFlag 0; Force.h:136-256): gravity and constant wind add
// dir strength dt, turbulence its curl noise, noise its fBm along dir; the
// z clamp constrains positions only and does nothing here.  This form is for
// force lists without turbulence and noise; tile_forces below takes them
// all (its registers would otherwise cost every launch occupancy).
__device__ inline void apply_forces(float& vx, float& vy, float& vz, const nb_force* forces, uint32_t count, float dt) {
  for (uint32_t fi = 0; fi < count; fi++) {
    const nb_force f = forces[fi];
    const uint32_t mask = f.affect_mask;
    if (mask != 0u && (mask & 1u) == 0u) continue;
    if (f.type == NB_FORCE_GRAVITY || f.type == NB_FORCE_CONSTANT_WIND) {
      const float s = f.data[3];
      vx += (f.data[0] * s) * dt;
      vy += (f.data[1] * s) * dt;
      vz += (f.data[2] * s) * dt;
    }
  }
}

// ---- turbulence and noise over a tile of nodes ----
// Noise at a node needs the hashed gradients of the 8 lattice points around
// each point it is taken at: 12 points (the curl's central differences) times
// the octaves, and each hash three correctly rounded sines (taken in FP64).
// Evaluated node by node that is 864 FP64 sines per node for three octaves
// and bounds the whole grid update.  The 512 nodes of a tile share their
// lattice points, though: a tile spans few lattice cells (8 nodes of spacing
// h * frequency, times two per octave).  So the block hashes each lattice
// point its nodes can reach once, into LDS, and the nodes interpolate from
// there; the hash of a lattice point depends on its integer coordinates only,
// so every value has the bits the node-by-node form gives.  An octave whose
// lattice range does not fit the table (a high frequency on a coarse grid)
// is hashed node by node.  On 57,001 sand particles (96^3, turbulence of three
// octaves and noise of two) the grid update went from 233 to 39 us, and to 29 with the
// sines one after the other and the hashing of nodes out of line (38 registers spilled
// and code beyond the instruction cache before).  What was left is a chain per node,
// 38 values of noise: four threads share a node, one for each of the curl's four
// points (ROLES = 4), and all forces' lattice points are hashed at once: 29 -> 19 us.
constexpr uint32_t kNoiseTab = 2048;    // lattice points held at a time
constexpr uint32_t kNoisePhases = 32;   // (group of points, octave) pairs with a place in the table
constexpr uint32_t kForcePhases = 16;   // of one force
struct NoisePhase {
  float lo[3];       // first lattice point of the range
  int dim[3];        // lattice points per axis (0: not in the table)
  uint32_t off;      // place of its first gradient
};
struct NoiseLds {
  float4 grad[kNoiseTab];
  NoisePhase ph[kNoisePhases];
  uint32_t size[kNoisePhases];
  float part[3][4][kNoiseThreads];  // the curl's potentials: group, point, node
  float end[2][3];   // world position of the block's first and last node
  uint32_t total, upto;
};

// noise at p in a phase's lattice range (or hashed at once when it has none)
__device__ __forceinline__ float noise_value3_tab(float px, float py, float pz, const NoisePhase& ph, const float4* grad) {
#pragma clang fp contract(off)
  if (ph.dim[0] == 0) return noise_value3(px, py, pz);
  const int ix = min(max(int(floorf(px) - ph.lo[0]), 0), ph.dim[0] - 2);
  const int iy = min(max(int(floorf(py) - ph.lo[1]), 0), ph.dim[1] - 2);
  const int iz = min(max(int(floorf(pz) - ph.lo[2]), 0), ph.dim[2] - 2);
  const int at = int(ph.off) + (iz * ph.dim[1] + iy) * ph.dim[0] + ix;
  return noise_value3_of(px, py, pz, [&](int ox, int oy, int oz) {
    const float4 g = grad[at + (oz * ph.dim[1] + oy) * ph.dim[0] + ox];
    return make_float3(g.x, g.y, g.z);
  });
}

// A force's noise: groups 0 for none
struct NoiseForm {
  bool turb;
  float fr, sd;
  uint32_t oct, groups, phases;  // phases: octave by octave, the groups within
};
__device__ __forceinline__ NoiseForm noise_form(const nb_force& f) {
  NoiseForm n;
  n.turb = f.type == NB_FORCE_TURBULENCE;  // data: strength, frequency, octaves bits, seed; noise: dir xyz before them
  n.fr = n.turb ? f.data[1] : f.data[4];
  n.sd = n.turb ? f.data[3] : f.data[6];
  const uint32_t oct = __float_as_uint(n.turb ? f.data[2] : f.data[5]);
  n.oct = oct > 1u ? oct : 1u;
  const bool on = (f.affect_mask == 0u || (f.affect_mask & 1u) != 0u) && (n.turb || f.type == NB_FORCE_NOISE);
  n.groups = on ? (n.turb ? 3u : 1u) : 0u;
  n.phases = on ? min(n.oct, kForcePhases / n.groups) * n.groups : 0u;
  return n;
}

// apply_forces for a block of kNoiseThreads, ROLES a node: thread t holds node
// t % (kNoiseThreads / ROLES); of the curl's four points it takes all (ROLES = 1) or
// number t / (kNoiseThreads / ROLES) (ROLES = 4).  The nodes lie in the box from first to last (their
// positions); (x, y, z) is the thread's node, live whether its velocity is wanted;
// role 0 holds the velocity.  Every thread of the block calls it.
template <uint32_t ROLES>
__device__ inline void tile_forces(float& vx, float& vy, float& vz, float x, float y, float z, bool live, float3 first,
                                   float3 last, const nb_force* forces, uint32_t count, float dt, NoiseLds& L) {
#pragma clang fp contract(off)
  constexpr float kEps = 0.1f;                            // step of the curl's differences
  constexpr float kShift[3] = {19.1f, 47.3f, 71.7f};      // of the curl's three potentials, each along its own axis
  constexpr uint32_t kNodes = kNoiseThreads / ROLES;
  const uint32_t node = threadIdx.x % kNodes, role = threadIdx.x / kNodes;
  if (threadIdx.x == 0u) {
    L.end[0][0] = first.x; L.end[0][1] = first.y; L.end[0][2] = first.z;
    L.end[1][0] = last.x; L.end[1][1] = last.y; L.end[1][2] = last.z;
  }
  // as many forces at a time as the phases and the table hold
  for (uint32_t from = 0; from < count;) {
    __syncthreads();  // the ends are there; the last table is done with
    if (threadIdx.x < 64u) {
      static_assert(kNoisePhases <= 64u && kForcePhases <= kNoisePhases, "a lane a phase");
      uint32_t upto = from, used = 0u, mine = count, idx = 0u;
      for (; upto < count; upto++) {
        const uint32_t np = noise_form(forces[upto]).phases;
        if (used + np > kNoisePhases) break;
        if (threadIdx.x >= used && threadIdx.x < used + np) {
          mine = upto;
          idx = threadIdx.x - used;
        }
        used += np;
      }
      NoisePhase ph;
      ph.lo[0] = ph.lo[1] = ph.lo[2] = 0.f;
      ph.dim[0] = ph.dim[1] = ph.dim[2] = 0;
      uint32_t size = 0u;
      if (mine < count) {
        const NoiseForm f = noise_form(forces[mine]);
        const uint32_t grp = idx % f.groups;
        float freq = 1.f;
        for (uint32_t o = 0; o < idx / f.groups; o++) freq *= 2.f;
        float vol = 1.f;
        bool ok = true;
        for (int a = 0; a < 3; a++) {
          // the nodes' coordinates lie between the ends', and rounding keeps
          // that order through every step
          const float p0 = L.end[0][a] * f.fr + f.sd, p1 = L.end[1][a] * f.fr + f.sd;
          float lo = fminf(p0, p1), hi = fmaxf(p0, p1);
          if (f.turb) {
            if (uint32_t(a) == grp) {
              lo = lo + kShift[a];
              hi = hi + kShift[a];
            } else {
              lo = lo - kEps;
              hi = hi + kEps;
            }
          }
          lo = floorf(lo * freq);
          hi = floorf(hi * freq);
          ok = ok && lo > -4194304.f && hi < 4194304.f && hi - lo < float(kNoiseTab);  // false for NaN too
          ph.lo[a] = lo;
          const float d = ok ? hi - lo + 2.f : 0.f;
          ph.dim[a] = int(d);
          vol *= d;
        }
        ok = ok && vol <= float(kNoiseTab);
        if (!ok) ph.dim[0] = ph.dim[1] = ph.dim[2] = 0;
        size = ok ? uint32_t(vol) : 0u;
      }
      // places in the table, force by force; a force that does not fit beside
      // those before it waits for the next table
      uint32_t at = 0u, slot = 0u;
      for (uint32_t f = from; f < upto; f++) {
        const uint32_t np = noise_form(forces[f]).phases;
        uint32_t sum = 0u;
        for (uint32_t i = 0; i < np; i++) sum += uint32_t(__shfl(int(size), int(slot + i)));
        if (f > from && at + sum > kNoiseTab) {
          upto = f;
          break;
        }
        for (uint32_t i = 0; i < np; i++, slot++) {
          uint32_t n = uint32_t(__shfl(int(size), int(slot)));
          const bool fits = at + n <= kNoiseTab;
          if (threadIdx.x == slot) {
            if (!fits) {
              ph.dim[0] = 0;
              size = 0u;
            }
            ph.off = at;
          }
          at += fits ? n : 0u;
        }
      }
      if (threadIdx.x < slot) {
        L.ph[threadIdx.x] = ph;
        L.size[threadIdx.x] = size;
      }
      if (threadIdx.x == 0u) {
        L.total = at;
        L.upto = upto;
      }
    }
    __syncthreads();
    const uint32_t total = L.total, upto = L.upto;
    for (uint32_t e = threadIdx.x; e < total; e += blockDim.x) {
      uint32_t i = 0;
      while (e >= L.ph[i].off + L.size[i]) i++;
      const uint32_t j = e - L.ph[i].off, dx = uint32_t(L.ph[i].dim[0]), dy = uint32_t(L.ph[i].dim[1]);
      const float3 g = noise_hash33<false>(L.ph[i].lo[0] + float(j % dx), L.ph[i].lo[1] + float((j / dx) % dy),
                                    L.ph[i].lo[2] + float(j / (dx * dy)));
      L.grad[e] = make_float4(g.x, g.y, g.z, 0.f);
    }
    __syncthreads();
    NoisePhase none;
    none.dim[0] = 0;
    uint32_t base = 0u;  // of the force's phases
    for (uint32_t fi = from; fi < upto; fi++) {
      const nb_force f = forces[fi];
      const uint32_t mask = f.affect_mask;
      if (mask != 0u && (mask & 1u) == 0u) continue;
      if (f.type == NB_FORCE_GRAVITY || f.type == NB_FORCE_CONSTANT_WIND) {
        const float s = f.data[3];
        vx += (f.data[0] * s) * dt;
        vy += (f.data[1] * s) * dt;
        vz += (f.data[2] * s) * dt;
        continue;
      }
      const NoiseForm nf = noise_form(f);
      if (nf.groups == 0u) continue;
      const float px = x * nf.fr + nf.sd, py = y * nf.fr + nf.sd, pz = z * nf.fr + nf.sd;
      // fBm (force_noise.glsl:40-50), octave by octave
      if (nf.turb) {
        // the curl (force_noise.glsl:54-82): group g holds the potential shifted
        // along axis g, at +-eps along the two other axes
        if (live) {
#pragma unroll 1
          for (uint32_t g = 0; g < 3u; g++) {
            const float qx = g == 0u ? px + kShift[0] : px, qy = g == 1u ? py + kShift[1] : py;
            const float qz = g == 2u ? pz + kShift[2] : pz;
            // first other axis: y, x, x; second: z, z, y
            const float ax = g == 0u ? 0.f : kEps, ay = g == 0u ? kEps : 0.f;
            const float bz = g == 2u ? 0.f : kEps, by = g == 2u ? kEps : 0.f;
            float s[4 / ROLES] = {};
            float amp = 0.5f, freq = 1.f;
#pragma unroll 1
            for (uint32_t o = 0; o < nf.oct; o++) {
              const uint32_t i = o * 3u + g;
              const NoisePhase ph = i < nf.phases ? L.ph[base + i] : none;
#pragma unroll
              for (uint32_t j = 0; j < 4u / ROLES; j++) {
                const uint32_t k = ROLES == 1u ? j : role;
                float ux = qx, uy = qy, uz = qz;
                if (k == 0u) { ux = qx + ax; uy = qy + ay; }
                if (k == 1u) { ux = qx - ax; uy = qy - ay; }
                if (k == 2u) { uy = qy + by; uz = qz + bz; }
                if (k == 3u) { uy = qy - by; uz = qz - bz; }
                s[j] += amp * noise_value3_tab(ux * freq, uy * freq, uz * freq, ph, L.grad);
              }
              freq *= 2.f;
              amp *= 0.5f;
            }
#pragma unroll
            for (uint32_t j = 0; j < 4u / ROLES; j++) L.part[g][ROLES == 1u ? j : role][node] = s[j];
          }
        }
        __syncthreads();
        if (live && role == 0u) {
          float d[3][2];  // differences of group g along its first and second other axis
#pragma unroll
          for (int g = 0; g < 3; g++) {
            d[g][0] = L.part[g][0][node] - L.part[g][1][node];
            d[g][1] = L.part[g][2][node] - L.part[g][3][node];
          }
          const float s2 = 2.f * kEps;
          const float cx = d[2][1] / s2 - d[1][1] / s2, cy = d[0][1] / s2 - d[2][0] / s2, cz = d[1][0] / s2 - d[0][0] / s2;
          vx += (cx * f.data[0]) * dt;
          vy += (cy * f.data[0]) * dt;
          vz += (cz * f.data[0]) * dt;
        }
        __syncthreads();
      } else if (live && role == 0u) {
        float s = 0.f, amp = 0.5f, freq = 1.f;
#pragma unroll 1
        for (uint32_t o = 0; o < nf.oct; o++) {
          const NoisePhase ph = o < nf.phases ? L.ph[base + o] : none;
          s += amp * noise_value3_tab(px * freq, py * freq, pz * freq, ph, L.grad);
          freq *= 2.f;
          amp *= 0.5f;
        }
        const float k = (s * f.data[3]) * dt;
        vx += f.data[0] * k;
        vy += f.data[1] * k;
        vz += f.data[2] * k;
      }
      base += nf.phases;
    }
    from = upto;
  }
}

// Whether a block's nodes are wanted, known by role 0 (live), for all roles; any: of
// the block.
template <uint32_t ROLES>
__device__ __forceinline__ bool noise_live(bool live, uint64_t* s_live, bool& any) {
  constexpr uint32_t kWaves = kNoiseThreads / ROLES / 64u;
  any = __syncthreads_or(live);
  if (ROLES == 1u) return live;
  const uint64_t b = __ballot(live);
  if (threadIdx.x < kWaves * 64u && (threadIdx.x & 63u) == 0u) s_live[threadIdx.x >> 6] = b;
  __syncthreads();
  return (s_live[(threadIdx.x >> 6) % kWaves] >> (threadIdx.x & 63u)) & 1u;
}

// applyColliderBC — shaders/collider_common.glsl:62-73
__device__ __forceinline__ void collider_bc(float& vx, float& vy, float& vz, float nx, float ny, float nz,
                                            const nb_collider& c) {
  float rx = vx - c.vx, ry = vy - c.vy, rz = vz - c.vz;
  float vn = rx * nx + ry * ny + rz * nz;
  if (vn < 0.f) {
    float nvx = vn * nx, nvy = vn * ny, nvz = vn * nz;
    float tx = rx - nvx, ty = ry - nvy, tz = rz - nvz;
    float tl = len3(tx, ty, tz);
    if (tl > 1e-8f) {
      float sc = fmaxf(0.f, 1.f - c.friction * fabsf(vn) / tl);
      tx *= sc; ty *= sc; tz *= sc;
    }
    vx = c.vx + tx - c.restitution * nvx;
    vy = c.vy + ty - c.restitution * nvy;
    vz = c.vz + tz - c.restitution * nvz;
  }
}

// analytic SDFs — shaders/collider_common.glsl:22-58; returns sdf, writes normal
__device__ __forceinline__ float collider_sdf(const nb_collider& c, float x, float y, float z, float& nx, float& ny,
                                              float& nz) {
  if (c.type == NB_COLL_SPHERE) {
    float dx = x - c.px, dy = y - c.py, dz = z - c.pz;
    float dist = len3(dx, dy, dz);
    if (dist > 1e-8f) { nx = dx / dist; ny = dy / dist; nz = dz / dist; } else { nx = 0.f; ny = 1.f; nz = 0.f; }
    return dist - c.radius;
  } else if (c.type == NB_COLL_BOX) {
    float rx = x - c.px, ry = y - c.py, rz = z - c.pz;
    float qx = fabsf(rx) - c.nx, qy = fabsf(ry) - c.ny, qz = fabsf(rz) - c.nz;
    float px = fmaxf(qx, 0.f), py = fmaxf(qy, 0.f), pz = fmaxf(qz, 0.f);
    float ql = len3(px, py, pz);
    float sdf = ql + fminf(fmaxf(qx, fmaxf(qy, qz)), 0.f);
    if (sdf < 0.f) {
      float ex = c.nx - fabsf(rx), ey = c.ny - fabsf(ry), ez = c.nz - fabsf(rz);
      nx = ny = nz = 0.f;
      if (ex < ey && ex < ez) nx = glsl_sign(rx + 1e-8f);
      else if (ey < ez) ny = glsl_sign(ry + 1e-8f);
      else nz = glsl_sign(rz + 1e-8f);
    } else {
      float sx = glsl_sign(rx + 1e-8f), sy = glsl_sign(ry + 1e-8f), sz = glsl_sign(rz + 1e-8f);
      float ux, uy, uz;
      if (ql > 1e-8f) { ux = px * sx; uy = py * sy; uz = pz * sz; } else { ux = sx; uy = sy; uz = sz; }
      float ul = len3(ux, uy, uz);
      nx = ux / ul; ny = uy / ul; nz = uz / ul;
    }
    return sdf;
  } else if (c.type == NB_COLL_CAPSULE) {
    float al = len3(c.nx, c.ny, c.nz);
    float adx, ady, adz;
    if (al > 1e-8f) { adx = c.nx / al; ady = c.ny / al; adz = c.nz / al; } else { adx = 0.f; ady = 1.f; adz = 0.f; }
    float t = fminf(fmaxf((x - c.px) * adx + (y - c.py) * ady + (z - c.pz) * adz, 0.f), al);
    float dx = x - (c.px + t * adx), dy = y - (c.py + t * ady), dz = z - (c.pz + t * adz);
    float dist = len3(dx, dy, dz);
    if (dist > 1e-8f) { nx = dx / dist; ny = dy / dist; nz = dz / dist; } else { nx = 0.f; ny = 1.f; nz = 0.f; }
    return dist - c.radius;
  }
  // plane
  float l = len3(c.nx, c.ny, c.nz);
  nx = c.nx / l; ny = c.ny / l; nz = c.nz / l;
  return (x - c.px) * nx + (y - c.py) * ny + (z - c.pz) * nz;
}

}  // namespace nb
