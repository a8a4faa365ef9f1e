// Kernels and launchers of the README step on gfx950 (shared by the forward
// entry points in transfer.hip and the adjoint in adjoint.hip): tile binning,
// deterministic P2G, fused grid update, G2P.  Reference: README.md:66-87; @P2G lowering
// src/Transfer/p2g.jl:145-178 (hoisting :272-307), grid-node half :377-395;
// @G2P lowering src/Transfer/g2p.jl:110-157; deferred weights
// src/Transfer/runtime.jl:21-24,55-130.
//
// Data flow of one P2G (no global float atomics; the lanes of a wave add to
// distinct nodes in LDS, so the sums follow a fixed order):
//   k_bin_keys      particle -> tile whose footprint holds its support window
//   radix sort      stable (tile, particle id) order -> perm
//   k_tile_counts / k_tab_reduce / k_tab_scan   tile ranges + slots, node blocks
//                   touched by some footprint (binning.hip)
//   k_p2g_tile      a few waves per tile: lanes own the 64 window-start classes of
//                   the tile, accumulate their particles' contributions in
//                   registers and add them into an LDS tile of the
//                   (BW+3)^dim footprint (distinct targets per instruction),
//                   then store the tile to a per-tile partial buffer
//   k_gather_grid   one workgroup per node block: each node sums the <= 2^dim
//                   tile partials covering it in a fixed order, then applies
//                   the grid-node half (Float64 m⁻¹, vⁿ, v, gravity, slip walls)
// G2P: k_g2p_tile stages the footprint's vⁿ, v in LDS and updates the tile's
// particles; k_g2p_outside handles particles outside the mesh (empty window).
// @G2P2G: the G2P kernel, then the P2G kernels at the kept positions; or, on
// request, k_g2p2g_fast: the G2P half and the P2G half's tile partials in one
// sweep over the particles, then k_gather_grid as for P2G.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <string>
#include <vector>

#include "tess_correct.hpp"
#include "tess_device.hpp"
#include "tess_internal.hpp"

namespace tess {
namespace {

// Tile geometry: 64 window-start classes per tile in both dimensions.
template <int D>
struct Geo;
template <>
struct Geo<3> {
  static constexpr int LT = 2, BW = 4, TS = 7, NFOOT = 343, NCLASS = 64, GNODES = 64;
  // padded LDS footprint, one array per component: node (x, y, z) at
  // x + PY*y + PZ*z.  For the 64 class lanes (4x4x4) at any stencil offset
  // the 64 addresses fall in distinct banks of a 64-bank LDS (two per bank
  // with 32 banks), which the unpadded pitches 7/49 do not give.
  static constexpr int PY = 12, PZ = 80, PSZ = TS * PZ;
};
template <>
struct Geo<2> {
  static constexpr int LT = 3, BW = 8, TS = 11, NFOOT = 121, NCLASS = 64, GNODES = 64;
  static constexpr int PY = 24, PZ = 0, PSZ = TS * PY;  // 8x8 class lanes, as in 3D
};

// padded LDS index of footprint node (x, y[, z])
template <int D>
__device__ __forceinline__ constexpr int pad_node(int x, int y, int z) {
  return x + Geo<D>::PY * y + Geo<D>::PZ * z;
}

template <int N, int E>
struct Pow;

// A tile's P2G partial in HBM: the nodes its classes reach, E = BW + SW - 1
// per axis from the footprint origin, x fastest, NV values per node
// (m, mv[D], f[D]).
template <int D, int SW>
struct Part {
  static constexpr int E = Geo<D>::BW + SW - 1;
  static constexpr int NV = 1 + 2 * D;
  static constexpr int NODES = Pow<E, D>::v;
  static constexpr int SIZE = NODES * NV;
};

template <int N, int E>
struct Pow {
  static constexpr int v = N * Pow<N, E - 1>::v;
};

template <int N>
struct Pow<N, 0> {
  static constexpr int v = 1;
};

// the lane counters (zero between their reports)
inline uint32_t* lane_counters(tess_ctx* ctx) {
  return ctx->lanes.as<uint32_t>(size_t(LANE_GROUPS) * LANES * LANE_STRIDE);
}
__device__ __forceinline__ uint32_t* lane_of(uint32_t* lanes, int group) {
  return lanes + (group * LANES + int(blockIdx.x) % LANES) * LANE_STRIDE;
}
enum { ERR_GIMP_LENGTH = 1, ERR_WINDOW = 2, ERR_INACTIVE = 4 };

template <typename T, int D>
struct SceneRec;

template <typename T, int D>
struct Args {
  DMesh<T, D> mesh;
  DField<T> x, v, V, gradv, F, sigma, l, logE;
  // where G2P writes the updated state, and at which index the particle at each
  // sorted position (nullptr: its own); the fields above unless a reorder moves
  // the particles to other arrays
  DField<T> ox, ov, oV, ogradv, oF, osigma;
  const uint32_t* dest;
  DField<T> gm, gmv, gf, gvn, gv;
  const int64_t* window;
  DField<T> w, gw;
  // a particle's stored weights, and its Vec and Mat fields, are contiguous (Julia layout)
  int32_t w_rows, p_rows;
  // corrected basis of deferred weights (0: the plain kernel) and its node filter
  int32_t corr;
  const uint8_t* filter;
  const uint32_t* perm;
  const uint32_t* tile_start;
  const uint32_t* tile_end;
  const uint32_t* active;
  const uint32_t* tile_flag;
  const uint32_t* tile_slot;
  const uint32_t* nb_list;
  const uint32_t* nb_flag;
  T* partials;
  // node blocks the last call on the grid wrote (zeroed unless written again)
  const uint32_t* stale_list;
  int64_t n_stale;
  // when set, G2P also writes each particle's position before the update here
  // (dense, D per particle): the positions the P2G half of a @G2P2G pass reads
  T* x_keep;
  // SpGrid: block numbering (nullptr for a dense grid), block_size_log2, blocks per axis
  const int32_t* numbering;
  int32_t spL;
  int32_t nblk[D];
  uint32_t* p2g_err;
  // batches of scenes: per-scene records and the first global tile / particle
  // of each scene (nscenes+1 entries); nullptr for a single scene
  const SceneRec<T, D>* scenes;
  const int64_t* scene_toff;
  const int64_t* scene_poff;
  const uint32_t* tile_scene;  // scene of each global tile
  int32_t nscenes;
  int64_t n, n_inside, n_active, n_nb;
  int32_t ntiles[D];
  T mp, dt;
  double lambda, mu, V0;
  T gravity[D];
  int32_t slip;
};

// G2P writes in place: the state fields are its outputs.
template <typename T, int D>
__host__ __device__ __forceinline__ void write_in_place(Args<T, D>& a) {
  a.ox = a.x;
  a.ov = a.v;
  a.oV = a.V;
  a.ogradv = a.gradv;
  a.oF = a.F;
  a.osigma = a.sigma;
  a.dest = nullptr;
}

// One scene of a batch: what differs between scenes in Args, plus where the
// scene's tiles and particles start in the batch-wide index spaces.
template <typename T, int D>
struct SceneRec {
  DMesh<T, D> mesh;
  DField<T> x, v, V, gradv, F, sigma, l, logE;
  DField<T> gm, gmv, gf, gvn, gv;
  T mp, dt;
  double lambda, mu, V0;
  T gravity[D];
  int32_t slip;
  int32_t ntiles[D];
  int64_t toff, poff, n, nnodes;
};

// Largest s with off[s] <= g (off ascending, off[0] = 0).
__device__ __forceinline__ int scene_of(const int64_t* __restrict__ off, int ns, int64_t g) {
  int lo = 0, hi = ns - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (off[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// The same for lanes whose places lie close together: one search by scalar loads
// for the wave's first lane, which nearly every lane shares.
__device__ __forceinline__ int scene_near(const int64_t* __restrict__ off, int ns, int64_t g) {
  const int64_t g0 = (int64_t(__builtin_amdgcn_readfirstlane(int(g >> 32))) << 32) |
                     int64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(g)))));
  const int s = scene_of(off, ns, g0);
  return off[s] <= g && g < off[s + 1] ? s : scene_of(off, ns, g);
}

// Replace the scene-dependent part of a by scene s of the batch.
template <typename T, int D>
__device__ __forceinline__ const SceneRec<T, D>& bind_scene(Args<T, D>& a, int s) {
  const SceneRec<T, D>& r = a.scenes[s];
  a.mesh = r.mesh;
  a.x = r.x;
  a.v = r.v;
  a.V = r.V;
  a.gradv = r.gradv;
  a.F = r.F;
  a.sigma = r.sigma;
  a.l = r.l;
  a.logE = r.logE;
  write_in_place(a);
  a.gm = r.gm;
  a.gmv = r.gmv;
  a.gf = r.gf;
  a.gvn = r.gvn;
  a.gv = r.gv;
  a.mp = r.mp;
  a.dt = r.dt;
  a.lambda = r.lambda;
  a.mu = r.mu;
  a.V0 = r.V0;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    a.gravity[d] = r.gravity[d];
    a.ntiles[d] = r.ntiles[d];
  }
  a.slip = r.slip;
  return r;
}

// A tile kernel's tile: in a batch, binds the scene holding global tile gtile
// and returns the scene-local tile, with the scene's first particle in poff.
template <bool BATCH, typename T, int D>
__device__ __forceinline__ uint32_t bind_tile(Args<T, D>& a, uint32_t gtile, uint32_t& poff) {
  poff = 0;
  if constexpr (!BATCH) {
    return gtile;
  } else {
    const SceneRec<T, D>& r = bind_scene(a, int(a.tile_scene[gtile]));
    poff = uint32_t(r.poff);
    return gtile - uint32_t(r.toff);
  }
}

// Workgroup i -> logical index; consecutive logical indices stay on one XCD
// (workgroups are dealt to the 8 XCDs round-robin).
__device__ __forceinline__ int64_t xcd_remap(int64_t i, int64_t N) {
  const int64_t per = (N + 7) >> 3;
  return (i & 7) * per + (i >> 3);
}
inline unsigned xcd_grid(int64_t N) { return unsigned(((N + 7) >> 3) << 3); }

// Workgroup i -> work item of the tile kernels.  One scene: xcd_remap (each
// XCD on a contiguous run of tiles, which share node blocks in its L2).  A
// batch (TESS_BATCH_SPREAD): consecutive items, dealt round-robin to the XCDs,
// since one scene's tiles carry loads that differ from the next scene's by
// orders of magnitude and contiguous runs would leave XCDs with unequal work.
#ifndef TESS_BATCH_SPREAD
#define TESS_BATCH_SPREAD 1
#endif
template <bool BATCH>
__device__ __forceinline__ int64_t item_of(int64_t i, int64_t N) {
  if constexpr (BATCH && TESS_BATCH_SPREAD) return i;
  return xcd_remap(i, N);
}

template <int D>
__device__ __forceinline__ void unlin(int64_t l, const int32_t* dims, int* I) {
#pragma unroll
  for (int d = 0; d < D; ++d) {
    I[d] = int(l % dims[d]);
    l /= dims[d];
  }
}

// Element of grid node I in the caller's grid arrays: the column-major node
// index of a dense grid, or on an SpGrid the SpArray storage index
// (k-1)*2^(L*dim) + local of its block's number k (src/Grids/spindices.jl:89,
// 96-102, 133-140), -1 when the block is inactive.
template <typename T, int D>
__device__ __forceinline__ int64_t grid_slot(const Args<T, D>& a, const int* I) {
  if (a.numbering == nullptr) return a.mesh.lin(I);
  const int L = a.spL;
  int64_t b = 0, loc = 0;
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    b = b * a.nblk[d] + (I[d] >> L);
    loc = (loc << L) | (I[d] & ((1 << L) - 1));
  }
  const int32_t k = a.numbering[b];
  return k > 0 ? (int64_t(k - 1) << (L * D)) + loc : int64_t(-1);
}

// SpGrid: every node of a class window [lo, lo+sw-1] (clipped to the mesh)
// must lie in an active block, the reference's "inactive SpGrid support node"
// check (src/Transfer/runtime.jl:155-161).  The class window contains the
// window of every particle of the class.
template <typename T, int D, int SW>
__device__ __forceinline__ void check_sparse_support(const Args<T, D>& a, const int* origin, const int* ccoord,
                                                     int ccount) {
  if (a.p2g_err == nullptr || ccount == 0) return;
  const int L = a.spL;
  int blo[D], ext[D], tot = 1;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int lo = max(origin[d] + ccoord[d], 0);  // a class holding particles has lo >= 0
    const int hi = min(lo + SW - 1, int(a.mesh.dims[d]) - 1);
    blo[d] = lo >> L;
    ext[d] = (hi >> L) - blo[d] + 1;
    tot *= ext[d];
  }
  bool bad = false;
  for (int k = 0; k < tot; ++k) {
    int r = k;
    int64_t b = 0, mul = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      b += int64_t(blo[d] + r % ext[d]) * mul;
      r /= ext[d];
      mul *= a.nblk[d];
    }
    bad = bad || a.numbering[b] == 0;
  }
  if (bad) atomicOr(a.p2g_err, uint32_t(ERR_INACTIVE));
}

// Particle window (0-based, clamped) from its position (deferred weights) or
// from stored weights; false if the window is empty.
template <typename T, int D, int BASIS, bool STORED>
__device__ __forceinline__ bool particle_window(const Args<T, D>& a, int64_t p, T* x, T& l, int* lo, int* hi,
                                                uint32_t* err) {
#pragma unroll
  for (int d = 0; d < D; ++d) x[d] = a.x(p, d);
  l = T(0);
  if constexpr (BASIS == TESS_UGIMP) {
    l = a.l(p) / a.mesh.h;  // _normalized_particle_length, gimp.jl:25
  }
  if constexpr (STORED) {
    bool ok = true, bad = false;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      lo[d] = int(a.window[p * 2 * D + 2 * d]) - 1;
      hi[d] = int(a.window[p * 2 * D + 2 * d + 1]) - 1;
      ok = ok && hi[d] >= lo[d];
      bad = bad || hi[d] - lo[d] >= support_width(BASIS) || lo[d] < 0 || hi[d] > a.mesh.dims[d] - 1;
    }
    if (ok && bad) {
      if (err) atomicOr(err, uint32_t(ERR_WINDOW));
      return false;
    }
    return ok;
  } else {
    T xi[D];
#pragma unroll
    for (int d = 0; d < D; ++d) xi[d] = (x[d] - a.mesh.xmin[d]) * a.mesh.h_inv;
    if (!inside_xi<T, D>(xi, a.mesh)) return false;
    if constexpr (BASIS == TESS_UGIMP) {
      if (!(T(0) <= l && l <= T(1)) && err) atomicOr(err, uint32_t(ERR_GIMP_LENGTH));
    }
#pragma unroll
    for (int d = 0; d < D; ++d) axis_window<T, BASIS>(xi[d], l, a.mesh.dims[d], lo[d], hi[d]);
    return true;
  }
}

// key = tile * 64 + class: the tile whose footprint [BW*t-1, BW*t+BW+1] holds
// the particle's window, and the window start relative to the footprint
// origin; ntiles*64 for particles with an empty window.
template <typename T, int D, int BASIS, bool STORED>
__device__ __forceinline__ uint32_t particle_key(const Args<T, D>& a, int64_t p, uint32_t ntiles, uint32_t* err) {
  T x[D], l;
  int lo[D], hi[D];
  if (!particle_window<T, D, BASIS, STORED>(a, p, x, l, lo, hi, err)) return ntiles * 64u;
  uint32_t t = 0, c = 0;
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    t = t * uint32_t(a.ntiles[d]) + uint32_t((lo[d] + 1) >> Geo<D>::LT);
    c = c * uint32_t(Geo<D>::BW) + uint32_t((lo[d] + 1) & (Geo<D>::BW - 1));
  }
  return t * 64u + c;
}

// The same key from a position and particle length held in registers
// (deferred weights); equals particle_key of the stored position.
template <typename T, int D, int BASIS>
__device__ __forceinline__ uint32_t key_of_position(const Args<T, D>& a, const T* x, T l, uint32_t ntiles) {
  T xi[D];
#pragma unroll
  for (int d = 0; d < D; ++d) xi[d] = (x[d] - a.mesh.xmin[d]) * a.mesh.h_inv;
  if (!inside_xi<T, D>(xi, a.mesh)) return ntiles * 64u;
  uint32_t t = 0, c = 0;
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    int lo, hi;
    axis_window<T, BASIS>(xi[d], l, a.mesh.dims[d], lo, hi);
    t = t * uint32_t(a.ntiles[d]) + uint32_t((lo + 1) >> Geo<D>::LT);
    c = c * uint32_t(Geo<D>::BW) + uint32_t((lo + 1) & (Geo<D>::BW - 1));
  }
  return t * 64u + c;
}

template <typename T, int D, int BASIS, bool STORED, bool BATCH = false>
__global__ __launch_bounds__(256) void k_bin_keys(Args<T, D> a, uint32_t* __restrict__ keys, uint32_t ntiles,
                                                  uint32_t* __restrict__ counters) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= a.n) return;
  if constexpr (BATCH) {  // batch: scene-local key, shifted to the scene's first global tile
    const SceneRec<T, D>& r = bind_scene(a, scene_near(a.scene_poff, a.nscenes, p));
    uint32_t nl = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) nl *= uint32_t(r.ntiles[d]);
    const uint32_t k = particle_key<T, D, BASIS, STORED>(a, p - r.poff, nl, counters + CNT_ERR);
    keys[p] = k == nl * 64u ? ntiles * 64u : k + uint32_t(r.toff) * 64u;
    return;
  }
  keys[p] = particle_key<T, D, BASIS, STORED>(a, p, ntiles, counters + CNT_ERR);
}

// ---- re-binning ----------------------------------------------------------------
// New keys are taken in the previous sorted order; the new order is the stable
// sort of that order by the new keys (the merge of binning.hip).

// The counters of a workgroup that computes its tile's next keys.
struct TileMoves {
  uint32_t leave, moved, out;  // out: those that leave the mesh, where next_key counts them (OWN)
};

// A leaver's rank among the arrivals of tile `to`: a wave draws the ranks of those
// that enter the tile of its first leaver with one atomic.  Where many leave in one
// step they mostly go to one place, and an atomic each on the one word takes 5.6 ns.
__device__ __forceinline__ uint32_t arrival_rank(const MoveOut& mo, uint32_t to) {
  const bool mine = to == uint32_t(__builtin_amdgcn_readfirstlane(int(to)));
  const uint64_t same = __ballot(mine);
  const uint32_t below = uint32_t(__popcll(same & ((uint64_t(1) << (threadIdx.x & 63)) - 1)));
  uint32_t r = 0;
  if (!mine || below == 0) r = atomicAdd(&mo.tin[to], mine ? uint32_t(__popcll(same)) : 1u);
  const uint32_t first = uint32_t(__builtin_amdgcn_readfirstlane(int(r)));
  return mine ? first + below : r;
}

// One particle's next key at sorted position jj of the tile whose run starts at
// `start`: written out, counted, and listed with its rank among the arrivals
// when it enters another tile (or leaves the mesh: tile ntiles).  OWN: of those
// that leave the mesh the rank is the workgroup's own, until tile_moves_end makes
// it global.  WAVE: the ranks by arrival_rank.
// k_rekey does both (8 M particles put outside: 1.7 ms by the wave, 0.54 so).  G2P
// draws by the wave but in 3D Float64, whose registers are full (the Taylor rod, five
// steps: 2,590 and 2,690 us by the wave, 2,570 and 2,580 us OWN).  Five steps whose
// first takes every particle out of the mesh, an atomic each and now: 2 M 3D Float32
// 24.8 and 2.7 ms, Float64 25.4 and 3.3 ms, 800 k 2D Float32 9.8 and 0.97 ms.
template <bool OWN, bool WAVE>
__device__ __forceinline__ void next_key(const MoveOut& mo, uint32_t key, uint32_t old_key, uint32_t jj, uint32_t tile,
                                         uint32_t start, uint32_t ntiles, TileMoves* s_mv, uint32_t& moved) {
  mo.nk[jj] = key;
  if (key != old_key) {
    ++moved;
    const uint32_t to = key >> 6;
    if (to != tile) {
      uint32_t r;
      if (OWN && to == ntiles)
        r = atomicAdd(&s_mv->out, 1u);
      else if constexpr (WAVE)
        r = arrival_rank(mo, to);
      else
        r = atomicAdd(&mo.tin[to], 1u);
      mo.out[start + atomicAdd(&s_mv->leave, 1u)] = make_uint2(jj, r);
    }
  }
}

// The tile's counts, and its ranks outside the mesh, by every thread of the
// workgroup after its last key.
__device__ __forceinline__ void tile_moves_end(const MoveOut& mo, uint32_t tile, uint32_t start, int cnt,
                                               uint32_t ntiles, TileMoves* s_mv, uint32_t moved) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) moved += __shfl_xor(moved, off, 64);
  if ((threadIdx.x & 63) == 0 && moved) atomicAdd(&s_mv->moved, moved);
  __syncthreads();
  const uint32_t leave = s_mv->leave, out = s_mv->out;
  if (threadIdx.x == 0) {
    mo.stay[tile] = uint32_t(cnt) - leave;
    if (s_mv->moved) atomicAdd(lane_of(mo.lanes, LANE_MOVED), s_mv->moved);
  }
  if (out == 0) return;  // uniform
  __syncthreads();
  if (threadIdx.x == 0) s_mv->out = atomicAdd(&mo.tin[ntiles], out);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < leave; i += blockDim.x) {
    uint2& o = mo.out[start + i];
    if ((mo.nk[o.x] >> 6) == ntiles) o.y += s_mv->out;
  }
}

// Next keys from the positions: one workgroup per active tile of the previous
// binning (whose keys may belong to other positions, or another particle set
// of the same size).
template <typename T, int D, int BASIS, bool STORED>
__global__ __launch_bounds__(256) void k_rekey(Args<T, D> a, const uint32_t* __restrict__ skeys, uint32_t ntiles,
                                               MoveOut mo, uint32_t* __restrict__ counters) {
  __shared__ TileMoves s_mv;
  const int64_t j = xcd_remap(blockIdx.x, a.n_active);
  if (j >= a.n_active) return;
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  if (threadIdx.x == 0) s_mv = TileMoves{0u, 0u, 0u};
  __syncthreads();
  uint32_t moved = 0;
  auto key_at = [&](int i) {
    return particle_key<T, D, BASIS, STORED>(a, a.perm[start + uint32_t(i)], ntiles, counters + CNT_ERR);
  };
  auto take = [&](int i) {
    const uint32_t jj = start + uint32_t(i), key = key_at(i);
    next_key<true, true>(mo, key, skeys[jj], jj, tile, start, ntiles, &s_mv, moved);
    return (key >> 6) != tile;
  };
  int i = int(threadIdx.x);
  const bool left = i < cnt && take(i);
  i += 256;
  if (cnt > 256 && __popcll(__ballot(left)) >= 48) {
    // particles put elsewhere altogether: once an eighth of the waves has lost
    // three quarters of its first 64, the others leave the ranks to the sort and
    // the tables to a count of the sorted keys (8 M particles spread anew, one
    // atomic each on 2,200 words: 2.11 ms, so 1.63 ms)
    uint32_t before = 0u;
    if ((threadIdx.x & 63) == 0) before = atomicAdd(counters + CNT_SCATTERED, 1u);
    if (int64_t(__builtin_amdgcn_readfirstlane(int(before))) >= a.n_active / 2) {
      if ((threadIdx.x & 63) == 0) atomicOr(counters + CNT_RESORT, uint32_t(RESORT_RECOUNT));
      for (; i < cnt; i += 256) {
        const uint32_t jj = start + uint32_t(i), key = key_at(i);
        mo.nk[jj] = key;
        moved += key != skeys[jj] ? 1u : 0u;
      }
    }
  }
  for (; i < cnt; i += 256) take(i);
  tile_moves_end(mo, tile, start, cnt, ntiles, &s_mv, moved);
}

// A workgroup's changed keys into its lane, by every thread of the workgroup.
__device__ __forceinline__ void count_moved(uint32_t* lanes, bool moved) {
  const int k = __syncthreads_count(moved);
  if (threadIdx.x == 0 && k > 0) atomicAdd(lane_of(lanes, LANE_MOVED), uint32_t(k));
}

// Next keys from the positions where some tile is too full for one workgroup: one
// particle per thread, no per-tile counts.
template <typename T, int D, int BASIS, bool STORED>
__global__ __launch_bounds__(256) void k_rekey_flat(Args<T, D> a, const uint32_t* __restrict__ skeys, uint32_t ntiles,
                                                    MoveOut mo, uint32_t* __restrict__ counters) {
  const int64_t jj = int64_t(blockIdx.x) * 256 + threadIdx.x;
  bool moved = false;
  if (jj < a.n) {
    const uint32_t key = particle_key<T, D, BASIS, STORED>(a, a.perm[jj], ntiles, counters + CNT_ERR);
    mo.nk[jj] = key;
    moved = key != skeys[jj];
  }
  count_moved(mo.lanes, moved);
}

// The same for the particles that were outside the mesh; one that came back is
// reported (the caller then sorts every key and counts the tiles again).
template <typename T, int D, int BASIS, bool STORED>
__global__ __launch_bounds__(256) void k_rekey_outside(Args<T, D> a, uint32_t ntiles, MoveOut mo,
                                                       uint32_t* __restrict__ counters) {
  const int64_t jj = a.n_inside + int64_t(blockIdx.x) * 256 + threadIdx.x;
  bool back = false;
  if (jj < a.n) {
    const uint32_t key = particle_key<T, D, BASIS, STORED>(a, a.perm[jj], ntiles, counters + CNT_ERR);
    mo.nk[jj] = key;
    back = (key >> 6) != ntiles;
  }
  count_moved(mo.lanes, back);
  if (__syncthreads_or(back) && threadIdx.x == 0) {
    const uint32_t marked = __atomic_load_n(counters + CNT_RESORT, __ATOMIC_RELAXED);
    if (!(marked & RESORT_RECOUNT)) atomicOr(counters + CNT_RESORT, uint32_t(RESORT_RECOUNT));
  }
}

template <typename T, int D>
__device__ __forceinline__ void zero_node(const Args<T, D>& a, int64_t i) {
  a.gm(i) = T(0);
#pragma unroll
  for (int c = 0; c < D; ++c) {
    a.gmv(i, c) = T(0);
    a.gf(i, c) = T(0);
    a.gvn(i, c) = T(0);
    a.gv(i, c) = T(0);
  }
}

template <typename T, int D>
__global__ __launch_bounds__(256) void k_zero_grid(Args<T, D> a, int64_t nnodes) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < nnodes) zero_node(a, i);
}

// Every node of every scene of a batch (blockIdx.y = scene).
template <typename T, int D>
__global__ __launch_bounds__(256) void k_zero_grid_batch(Args<T, D> a) {
  const SceneRec<T, D>& r = bind_scene(a, int(blockIdx.y));
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < r.nnodes) zero_node(a, i);
}

// Zero the nodes of node block B, touched by the last call, unless this call
// touches it (one thread per node).
template <typename T, int D, bool BATCH = false>
__device__ __forceinline__ void zero_stale_block(Args<T, D>& a, const uint32_t B) {
  using G = Geo<D>;
  if (a.nb_flag[B]) return;
  uint32_t poff;
  const uint32_t Bl = bind_tile<BATCH>(a, B, poff);
  int Bi[D], I[D];
  unlin<D>(Bl, a.ntiles, Bi);
  int r = threadIdx.x;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    I[d] = Bi[d] * G::BW + r % G::BW;
    r /= G::BW;
    if (I[d] >= a.mesh.dims[d]) return;
  }
  const int64_t i = grid_slot(a, I);
  if (i >= 0) zero_node(a, i);
}
template <typename T, int D, bool BATCH = false>
__global__ __launch_bounds__(64) void k_zero_stale(Args<T, D> a, const uint32_t* __restrict__ prev_list,
                                                    int64_t n_prev) {
  if (int64_t(blockIdx.x) < n_prev) zero_stale_block<T, D, BATCH>(a, prev_list[blockIdx.x]);
}

template <typename T, int D, int BASIS>
__device__ __forceinline__ void axis_jets(T xd, int lo_local, const T* s_nodex, T l, T hinv, T* val, T* der) {
  constexpr int SW = support_width(BASIS);
#pragma unroll
  for (int a = 0; a < SW; ++a) {
    const T xi = (xd - s_nodex[lo_local + a]) * hinv;  // separable_nodal_basis_jet, basis_weight.jl:49-60
    piecewise_jet<T, BASIS>(xi, l, val[a], der[a]);
  }
}

// Corrected deferred weights of one particle inside a tile kernel: the axis
// jets (nodewise values at the footprint's node coordinates) become the
// corrected ones, or the general fit is prepared (src/Transfer/runtime.jl:55-80
// with the deferred states of wls.jl:131-163, kernelcorrection.jl:41-63).
// ext = window extent - 1 per axis, ccoord = window start in the footprint.
template <typename T, int D, int BASIS>
__device__ __forceinline__ void correct_jets(const Args<T, D>& a, const T* x, const int* lo, const int* ext,
                                             const int* ccoord, const T (*s_nodex)[Geo<D>::TS],
                                             Corrected<T, D, support_width(BASIS)>& cs,
                                             T (&val)[D][support_width(BASIS)], T (&der)[D][support_width(BASIS)]) {
  constexpr int SW = support_width(BASIS);
  int cnt[D];
  T xi[D][SW];
#pragma unroll
  for (int d = 0; d < D; ++d) {
    cnt[d] = ext[d] + 1;
#pragma unroll
    for (int k = 0; k < SW; ++k) xi[d][k] = (x[d] - s_nodex[d][ccoord[d] + k]) * a.mesh.h_inv;
  }
  cs.prepare(a.corr, BASIS, false, a.filter, a.mesh.dims, lo, cnt, xi, val, der);
}

// The footprint's node coordinates per axis into LDS, by the workgroup's first
// threads.  The axes are unrolled: an axis taken from the thread's number indexes
// the mesh at run time, which keeps a batch's whole argument block (880 bytes per
// lane, rewritten per scene) in scratch memory (8 scenes of 125 k 3D Float32
// particles in no order: P2G 760 and 139 us, G2P 1006 and 186 us).
template <typename T, int D>
__device__ __forceinline__ void stage_nodes(const DMesh<T, D>& mesh, const int* origin, T (*s_nodex)[Geo<D>::TS]) {
  constexpr int TS = Geo<D>::TS;
  static_assert(D * TS <= 64, "one thread per coordinate in the smallest workgroup");
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const int k = int(threadIdx.x) - d * TS;
    if (k >= 0 && k < TS) s_nodex[d][k] = mesh.node(d, origin[d] + k);
  }
}

// ---- P2G -------------------------------------------------------------------

__device__ __forceinline__ uint64_t lanemask_lt64() { return (uint64_t(1) << (threadIdx.x & 63)) - 1; }

// Per-class counts of one tile from its slice of the sorted keys (class = low 6
// bits), by wave-level matching; lane c gets count and offset of class c.
// sorted slots per tile whose particle ids the transfer kernels stage in LDS
constexpr int PID_CAP = 1024;
// G2P's own: a 3D tile of 27 particles per cell holds 1728
template <int D>
constexpr int G2P_PID_CAP = D == 3 ? 2048 : 1024;

template <int NW = 1>
// With s_pid, also stages the particle ids (perm - poff) of the tile's first
// `cap` sorted slots in LDS, and with s_key their sort keys: the transfer
// kernels then address their particle loads through LDS reads instead of
// global loads that the memory counter would drain behind earlier traffic.
__device__ __forceinline__ void tile_class_counts(const uint32_t* __restrict__ skeys, uint32_t start, int cnt,
                                                  uint32_t* s_cnt, int& ccount, int& coff, int& maxcnt,
                                                  const uint32_t* __restrict__ perm = nullptr, uint32_t poff = 0,
                                                  uint32_t* s_pid = nullptr, uint32_t* s_key = nullptr,
                                                  int cap = 0) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));  // uniform: scalar branches
  // one chunk of 64 sorted slots: stage ids and keys, count the classes
  auto chunk = [&](int i, uint32_t key, uint32_t pid) {
    const bool valid = i < cnt;
    const uint32_t c = key & 63u;
    if (s_pid && valid && i < cap) {
      s_pid[i] = pid - poff;
      if (s_key) s_key[i] = key;
    }
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const bool bit = (c >> b) & 1u;
      const uint64_t m = __ballot(valid && bit);
      peers &= bit ? m : ~m;
    }
    if (valid && (peers & lanemask_lt64()) == 0) atomicAdd(&s_cnt[c], uint32_t(__popcll(peers)));
  };
  // the keys and ids of a wave's first CC chunks are loaded together, before
  // the barrier (it waits only on LDS operations), so one memory round trip
  // serves them (and whatever the caller has in flight)
  constexpr int CC = 4;
  uint32_t kk[CC], pp[CC];
#pragma unroll
  for (int r = 0; r < CC; ++r) {
    const int i = wave * 64 + r * 64 * NW + lane;
    kk[r] = i < cnt ? skeys[start + i] : 0u;
    pp[r] = (s_pid && i < cnt && i < cap) ? perm[start + i] : 0u;
  }
  if (wave == 0) s_cnt[lane] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < CC; ++r) {
    const int i = wave * 64 + r * 64 * NW + lane;
    if (wave * 64 + r * 64 * NW < cnt) chunk(i, kk[r], pp[r]);  // uniform
  }
  for (int base = wave * 64 + CC * 64 * NW; base < cnt; base += 64 * NW) {
    const int i = base + lane;
    const bool valid = i < cnt;
    chunk(i, valid ? skeys[start + i] : 0u, (s_pid && valid && i < cap) ? perm[start + i] : 0u);
  }
  __syncthreads();
  ccount = int(s_cnt[lane]);
  int incl = ccount;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(incl, off, 64);
    if (lane >= off) incl += u;
  }
  coff = incl - ccount;
  maxcnt = ccount;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) maxcnt = max(maxcnt, __shfl_xor(maxcnt, off, 64));
}

// Layered-order contiguity of one layer (the estimator of
// block_ordered_particle_contiguity, src/Parallel/cpu_block_strategy.jl:222-246):
// a lane holding a particle (bit set in `has`) is paired with the next lower
// such lane, the lowest one with the last particle of the previous layer
// (`last`, updated here); returns 1 where the pair is not consecutive in
// storage.  Called by every lane of the wave; the tile's first particle has
// no pair.
__device__ __forceinline__ uint32_t broken_pair(uint64_t has, int k, uint32_t pid, uint32_t& last) {
  const uint64_t below = has & lanemask_lt64();
  const uint32_t pl = __shfl(pid, below ? 63 - __clzll(below) : 0, 64);
  const bool mine = (has >> (threadIdx.x & 63)) & 1u;
  const uint32_t r = (mine && (below || k > 0) && pid != (below ? pl : last) + 1u) ? 1u : 0u;
  last = __shfl(pid, 63 - __clzll(has), 64);
  return r;
}

// NC components of particle p; where they are contiguous (the Julia layout) as
// 16-byte words: the particles of a wave lie 64 places apart, and the address
// unit takes one request per lane and instruction.
template <typename T, int NC>
__device__ __forceinline__ void get_row(bool rows, const DField<T>& f, int64_t p, T (&v)[NC]) {
  if (rows) {
    __builtin_memcpy(v, f.p + p * NC, sizeof(v));
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = f(p, c);
  }
}
template <typename T, int NC>
__device__ __forceinline__ void put_row(bool rows, const DField<T>& f, int64_t p, const T (&v)[NC]) {
  if (rows) {
    __builtin_memcpy(f.p + p * NC, v, sizeof(v));
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c) f(p, c) = v[c];
  }
}

// N of a particle's stored weights from offset o0 on, likewise.
template <typename T, int D, int NOFF, int N>
__device__ __forceinline__ void stored_weights(const Args<T, D>& a, uint32_t pid, int o0, T (&w)[N], T (&g)[N][D]) {
  const int64_t e0 = int64_t(o0) + int64_t(NOFF) * pid;
  if (a.w_rows) {
    __builtin_memcpy(w, a.w.p + e0, sizeof(w));
    __builtin_memcpy(g, a.gw.p + e0 * D, sizeof(g));
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      w[i] = a.w(e0 + i);
#pragma unroll
      for (int c = 0; c < D; ++c) g[i][c] = a.gw(e0 + i, c);
    }
  }
}

// Stored and general corrected weights.  The sort key orders each tile's
// particles by class (window start relative to the footprint origin), so lane c
// owns class c: it walks its particles, accumulates their contributions to the
// sw^dim nodes of the class window in registers, and adds them into the LDS
// tile.  Lanes hold distinct classes, so the adds of one offset touch each node at
// most once; the waves add in turn, so the order of the adds is fixed.
//
// A tile has WP x NK waves: wave w accumulates the offsets of the passes w % WP,
// w % WP + WP, ... over every NK-th particle of each class (WP is NPASS, or 1).
// What bounds it is the latency of the particle loads (each waits for its id) and,
// for particles in no order, the lines they touch.  168k particles at random
// places, 2D Float64 quadratic with stored weights, about 250 and up to 1400
// particles per tile: one wave per tile 58 and 239 us; four, ids in LDS, 58 and
// 106 us; with the weights in 16-byte words 46 and 67 us; with the adds below 38 us
// (the first).
//
// The waves add by reading, adding and writing back: LDS add instructions made the
// four waves' adds the longest part in Float32 (1.44 M ordered 2D particles, stored
// quadratic: 408 us with them, 361 us for one wave with them, 149 us so).
template <int D, int NPASS>
constexpr int P2G_TILE_SPLIT = NPASS == 1 ? 4 : (D == 2 ? 2 : 1);  // NK

// A general corrected basis in Float64 fills the registers of a SIMD with one or
// two waves.  Where the tiles alone fill the chip, a tile takes one wave per pass
// (2D), or one wave for its three passes (3D: three waves leave every fourth SIMD
// idle).  WLS quadratic, random places, split and so: 2D 57.6 k particles (400
// tiles) 68 and 70 us, 360 k (2,500) 160 and 116, 1.44 M 459 and 276; 3D 64 k (500
// tiles) 181 and 182 us, 125 k (730) 257 and 193, 1 M 1225 and 651.
template <typename T, int D, int NPASS>
constexpr bool P2G_TILE_SOLO = sizeof(T) == 8 && (D == 2 || NPASS == 3);
constexpr int64_t P2G_SOLO_TILES = 512;

template <typename T, int D, int BASIS, bool STORED, int NPASS, bool CORR = false, int WP = NPASS,
          int NK = P2G_TILE_SPLIT<D, NPASS>>
__global__ __launch_bounds__((64 * WP * NK)) void k_p2g_tile(
    Args<T, D> a, const uint32_t* __restrict__ skeys, uint32_t* __restrict__ misplaced) {
  using G = Geo<D>;
  constexpr int SW = support_width(BASIS);
  constexpr int NV = 1 + 2 * D;
  constexpr int NOFF = Pow<SW, D>::v;
  constexpr int NSL = NOFF / NPASS;  // offsets per pass (NPASS is 1 or SW)
  constexpr int NW = WP * NK;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int part = wave / WP;
  const int64_t j = xcd_remap(blockIdx.x, a.n_active);
  if (j >= a.n_active) return;
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  int tI[D], origin[D];
  unlin<D>(tile, a.ntiles, tI);
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = tI[d] * G::BW - 1;

  __shared__ __align__(16) T s_tile[G::NFOOT][8];
  __shared__ T s_nodex[D][G::TS];
  __shared__ uint32_t s_cnt[64];
  __shared__ uint32_t s_pid[PID_CAP];
  for (int q = int(threadIdx.x); q < 8 * G::NFOOT; q += 64 * NW) (&s_tile[0][0])[q] = T(0);
  stage_nodes<T, D>(a.mesh, origin, s_nodex);
  int ccount, coff, maxcnt;
  tile_class_counts<NW>(skeys, start, cnt, s_cnt, ccount, coff, maxcnt, a.perm, 0, s_pid, nullptr, PID_CAP);
  auto id_at = [&](int i) { return cnt <= PID_CAP ? s_pid[i] : a.perm[start + uint32_t(i)]; };
  int ccoord[D];
  {
    int r = lane;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      ccoord[d] = r % G::BW;
      r /= G::BW;
    }
  }
  if (wave == 0) check_sparse_support<T, D, SW>(a, origin, ccoord, ccount);
  // neighbours in the layered order (k-th particle of every class, classes
  // ascending, then the next k) whose storage indices are not consecutive
  if (misplaced && wave == NW - 1) {
    uint32_t bad = 0, last = 0;
    for (int k = 0; k < maxcnt; ++k) {
      const uint64_t has = __ballot(k < ccount);
      const uint32_t pid = k < ccount ? id_at(coff + k) : 0u;
      bad += broken_pair(has, k, pid, last);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) bad += __shfl_xor(bad, off, 64);
    if (lane == 0 && bad) atomicAdd(lane_of(misplaced, LANE_BROKEN), bad);
  }
  const T mp = a.mp, hinv = a.mesh.h_inv;
  for (int pass = wave % WP; pass < NPASS; pass += WP) {
    T acc[NSL][NV];
#pragma unroll
    for (int s2 = 0; s2 < NSL; ++s2)
#pragma unroll
      for (int v = 0; v < NV; ++v) acc[s2][v] = T(0);
    for (int k = part; k < maxcnt; k += NK) {
      if (k >= ccount) continue;
      const uint32_t pid = id_at(coff + k);
      T x[D], l;
      int lo[D], hi[D];
      particle_window<T, D, BASIS, STORED>(a, pid, x, l, lo, hi, nullptr);
      int ext[D];
#pragma unroll
      for (int d = 0; d < D; ++d) ext[d] = hi[d] - lo[d];
      // hoisted particle factors (p2g.jl:272-307): mₚ*v[p] and (-V[p])*σ[p]
      T mv[D], A[D * D];
      get_row(a.p_rows, a.v, pid, mv);
      get_row(a.p_rows, a.sigma, pid, A);
      const T negV = -a.V(pid);
#pragma unroll
      for (int d = 0; d < D; ++d) mv[d] = mp * mv[d];
#pragma unroll
      for (int q = 0; q < D * D; ++q) A[q] = negV * A[q];
      T val[D][SW], der[D][SW];
      constexpr int NCH = D == 3 ? SW : NSL;  // weights in registers at a time: 3D a row, 2D the pass's
      T sw[STORED ? NCH : 1], sg[STORED ? NCH : 1][D];
      if constexpr (!STORED) {
#pragma unroll
        for (int d = 0; d < D; ++d) axis_jets<T, D, BASIS>(x[d], ccoord[d], s_nodex[d], l, hinv, val[d], der[d]);
      }
      Corrected<T, D, SW> cs;
      if constexpr (CORR) correct_jets<T, D, BASIS>(a, x, lo, ext, ccoord, s_nodex, cs, val, der);
#pragma unroll
      for (int s2 = 0; s2 < NSL; ++s2) {
        const int o = pass * NSL + s2;
        if constexpr (STORED) {
          if (s2 % NCH == 0) stored_weights<T, D, NOFF>(a, pid, o, sw, sg);
        }
        int aa[D];
        int r = o;
        bool ok = true;
#pragma unroll
        for (int d = 0; d < D; ++d) {
          aa[d] = r % SW;
          r /= SW;
          ok = ok && aa[d] <= ext[d];
        }
        if (!ok) continue;
        T w, g[D];
        if constexpr (STORED) {
          w = sw[s2 % NCH];
#pragma unroll
          for (int c = 0; c < D; ++c) g[c] = sg[s2 % NCH][c];
        } else if (CORR && cs.mode == CORR_GENERAL) {
          cs.node(val, aa, filter_pass<D>(a.filter, a.mesh.dims, lo, aa), hinv, w, g);
        } else {
          // w = Π_d N_d (left-assoc), ∇w_c = (N'_c Π_{d≠c} N_d) h⁻¹
          w = val[0][aa[0]];
#pragma unroll
          for (int d = 1; d < D; ++d) w = w * val[d][aa[d]];
#pragma unroll
          for (int c = 0; c < D; ++c) {
            T gg = (c == 0) ? der[0][aa[0]] : val[0][aa[0]];
#pragma unroll
            for (int d = 1; d < D; ++d) gg = gg * ((d == c) ? der[d][aa[d]] : val[d][aa[d]]);
            g[c] = gg * hinv;
          }
        }
        acc[s2][0] += w * mp;
#pragma unroll
        for (int c = 0; c < D; ++c) acc[s2][1 + c] += w * mv[c];
#pragma unroll
        for (int r2 = 0; r2 < D; ++r2) {
          T f = A[r2] * g[0];
#pragma unroll
          for (int c = 1; c < D; ++c) f = f + A[r2 + D * c] * g[c];
          acc[s2][1 + D + r2] += f;
        }
      }
    }
    for (int turn = 0; turn < NW; ++turn) {
      if (wave == turn && ccount > part) {
#pragma unroll
      for (int s2 = 0; s2 < NSL; ++s2) {
        int r = pass * NSL + s2, q = 0, mul = 1;
#pragma unroll
        for (int d = 0; d < D; ++d) {
          q += (ccoord[d] + r % SW) * mul;
          r /= SW;
          mul *= G::TS;
        }
        T t[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) t[v] = s_tile[q][v];
#pragma unroll
        for (int v = 0; v < NV; ++v) s_tile[q][v] = t[v] + acc[s2][v];
        __asm__ volatile("" ::: "memory");  // the LDS executes one wave's accesses in order
      }
      }
      __syncthreads();
    }
  }
  using PT = Part<D, SW>;
  T* out = a.partials + int64_t(j) * PT::SIZE;
  for (int e = int(threadIdx.x); e < PT::SIZE; e += 64 * NW) {
    const int n = e / NV, v = e % NV;
    const int x = n % PT::E, y = (n / PT::E) % PT::E, z = D == 3 ? n / (PT::E * PT::E) : 0;
    out[e] = s_tile[x + G::TS * (y + G::TS * z)][v];
  }
}

template <typename T, int D>
__device__ __forceinline__ double det_d(const T* F) {
  if constexpr (D == 2) {
    return double(F[0]) * double(F[3]) - double(F[2]) * double(F[1]);
  } else {
    const double f11 = F[0], f21 = F[1], f31 = F[2], f12 = F[3], f22 = F[4], f32 = F[5], f13 = F[6], f23 = F[7],
                 f33 = F[8];
    return f11 * (f22 * f33 - f23 * f32) - f12 * (f21 * f33 - f23 * f31) + f13 * (f21 * f32 - f22 * f31);
  }
}

// Neo-Hookean Cauchy stress σ = (μ(FFᵀ-I) + λ lnJ I)/J and V = V0 J of the
// updated F (README.md:84-86), stiffness scaled by exp(logE) when has_logE.
// J = det F (cofactor expansion), ln J and 1/J are Float64 for both storage
// types, so a small or large J keeps its relative accuracy.  Float64 storage
// forms FFᵀ - I as written.  Float32 storage forms it from H = F - I as
// H + Hᵀ + HHᵀ in Float32: the difference of FFᵀ and I would lose the digits
// of a small strain, H itself is exact, and nothing in the sum cancels for F
// near I.  σ is written as sig[r + D*b].
template <typename T, int D>
__device__ __forceinline__ void neo_hookean(const T* Fn, double lam0, double mu0, double V0, bool has_logE, T logE,
                                            T* sig, T& Vout) {
  const double J = det_d<T, D>(Fn);
  double lam = lam0, mu = mu0;
  if (has_logE) {
    const double sc = exp(double(logE));
    lam *= sc;
    mu *= sc;
  }
  const double lnJ = log(J);
  const double invJ = 1.0 / J;
  if constexpr (sizeof(T) == 4) {
    const float muJ = float(mu * invJ);
    const float lamJ = float(lam * lnJ * invJ);
    float H[D * D];
#pragma unroll
    for (int b = 0; b < D; ++b)
#pragma unroll
      for (int r = 0; r < D; ++r) H[r + D * b] = Fn[r + D * b] - (r == b ? 1.0f : 0.0f);
#pragma unroll
    for (int b = 0; b < D; ++b)
#pragma unroll
      for (int r = 0; r < D; ++r) {
        float hh = H[r] * H[b];  // (HHᵀ)_rb = Σ_k H_rk H_bk
#pragma unroll
        for (int k = 1; k < D; ++k) hh = fmaf(H[r + D * k], H[b + D * k], hh);
        const float bp = (H[r + D * b] + H[b + D * r]) + hh;
        sig[r + D * b] = r == b ? fmaf(muJ, bp, lamJ) : muJ * bp;
      }
  } else {
#pragma unroll
    for (int b = 0; b < D; ++b)
#pragma unroll
      for (int r = 0; r < D; ++r) {
        double bb = 0.0;
#pragma unroll
        for (int k = 0; k < D; ++k) bb += double(Fn[r + D * k]) * double(Fn[b + D * k]);
        const double sg = mu * (bb - (r == b ? 1.0 : 0.0)) + (r == b ? lam * lnJ : 0.0);
        sig[r + D * b] = T(sg * invJ);
      }
  }
  Vout = T(V0 * J);
}

// ---- deferred-weight fast paths ------------------------------------------------
//
// Both transfer kernels below evaluate the basis on the fly.  Along an axis
// whose window is not truncated they use the reference's full-support
// polynomial (bspline.jl:90-100,146-170); truncated axes and uGIMP use the
// nodewise piecewise jet (basis_weight.jl:49-60,624-632).  Tensor-product sums
// are factored by axis (products of the y/z jets are formed once per (y,z)
// offset and reused along x); the results equal the reference's up to
// floating-point rounding.

// Loads component c of element e: Julia-native AoS fields (component stride 1,
// element stride NC) get compile-time strides so neighbouring components
// merge into vector loads.
template <typename T, int NC, bool AOS>
__device__ __forceinline__ T fld(const DField<T>& f, int64_t e, int c) {
  if constexpr (AOS) return f.p[e * NC + c];
  else return f(e, c);
}
template <typename T, int NC, bool AOS>
__device__ __forceinline__ T& fldw(const DField<T>& f, int64_t e, int c) {
  if constexpr (AOS) return f.p[e * NC + c];
  else return f(e, c);
}

// Stores of the G2P particle stream (v, ∇v, x, F, σ, V): non-temporal (NT)
// where the particles are known to lie in the layered order, so that a wave's
// stores fill whole lines.  Where they do not, the pieces of a line are written
// by different waves, and only the L2 can put them together: the block at 1.7 M
// particles in generation order took 355 us non-temporal and 132 us plain, the
// falling 13.4 M-particle block (contiguity 0.85-1) 884 and 840 us; the same
// block in layered order 805 us non-temporal and 843 us plain.
template <bool NT, typename T>
__device__ __forceinline__ void st_g2p(T& dst, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, &dst);
  else dst = v;
}

// 1-D jets at the window nodes lo..lo+SW-1 of one axis; entries past the
// (truncated) window are zero.  Derivatives are returned times h⁻¹.
template <typename T, int BASIS>
__device__ __forceinline__ void axis_jets_mixed(T xd, T xmin, int lo_local, int ext, const T* s_nodex, T l, T hinv,
                                                T* val, T* der) {
  constexpr int SW = support_width(BASIS);
  bool done = false;
  if constexpr (BASIS != TESS_UGIMP) {
    if (ext == SW - 1) {
      const T xi = (xd - xmin) * hinv;
      const T y = (degree_of(BASIS) % 2 == 1) ? xi : xi - T(0.5);
      bspline_local_jet<T, BASIS>(y - floor(y), val, der);
      done = true;
    }
  }
  if (!done) {
#pragma unroll
    for (int q = 0; q < SW; ++q) {
      T v0 = T(0), d0 = T(0);
      if (q <= ext) piecewise_jet<T, BASIS>((xd - s_nodex[lo_local + q]) * hinv, l, v0, d0);
      val[q] = v0;
      der[q] = d0;
    }
  }
#pragma unroll
  for (int q = 0; q < SW; ++q) der[q] *= hinv;
}

// Separable corrected bases in the fast kernels: KernelCorrection or WLS with
// Polynomial(MultiLinear()) over a quadratic or cubic B-spline and no filter
// (the reference's SeparableKernelCorrection and the MultiLinear WLS,
// kernelcorrection.jl:53-63, wls.jl:79-99, 166-189).  Every particle is either
// the plain kernel or a product of per-axis 1-D fits, so the fast kernels only
// swap the axis jets.
__host__ __device__ constexpr bool separable_correction(int corr, int basis, bool has_filter) {
  return (corr & TESS_POLY_MULTILINEAR) && (basis == TESS_BSPLINE_QUADRATIC || basis == TESS_BSPLINE_CUBIC) &&
         !has_filter;
}

// Whether a particle's axis jets are corrected: always for WLS, off a whole
// support for KernelCorrection (kernelcorrection.jl:55-63).
template <typename T, int D, int BASIS>
__device__ __forceinline__ bool sep_corrects(const Args<T, D>& a, const T* x) {
  if (!(a.corr & TESS_KERNEL_CORRECTION)) return true;
  bool full = true;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    int lo, hi;
    axis_window<T, BASIS>((x[d] - a.mesh.xmin[d]) * a.mesh.h_inv, T(0), a.mesh.dims[d], lo, hi);
    full = full && hi - lo == support_width(BASIS) - 1;
  }
  return !full;
}

// Axis jets of a separable corrected basis: the plain ones, or the 1-D fit of
// the nodewise values (der in world units, as axis_jets_mixed returns it).
template <typename T, int BASIS>
__device__ __forceinline__ void axis_jets_sep(T xd, T xmin, int lo_local, int ext, const T* s_nodex, T hinv,
                                              bool correct, T* val, T* der) {
  constexpr int SW = support_width(BASIS);
  if (!correct) {
    axis_jets_mixed<T, BASIS>(xd, xmin, lo_local, ext, s_nodex, T(0), hinv, val, der);
    return;
  }
  T dh[SW];
#pragma unroll
  for (int q = 0; q < SW; ++q) {
    const T xi = (xd - s_nodex[lo_local + q]) * hinv;
    T v0 = T(0), d0 = T(0);
    if (q <= ext) piecewise_jet<T, BASIS>(xi, T(0), v0, d0);
    val[q] = v0;
    dh[q] = -xi;
  }
  wls_axis<T, SW>(ext + 1, degree_of(BASIS), dh, val, der);
#pragma unroll
  for (int q = 0; q < SW; ++q) der[q] *= hinv;
}

// One particle's P2G inputs, loaded one iteration ahead of their use.
template <typename T, int D>
struct P2GIn {
  uint32_t pid;
  T x[D], v[D], V, S[D * D], l;
};

template <typename T, int D, int BASIS, bool AOS>
__device__ __forceinline__ void p2g_load(const Args<T, D>& a, uint32_t pid, P2GIn<T, D>& in) {
  in.pid = pid;
#pragma unroll
  for (int d = 0; d < D; ++d) in.x[d] = fldw<T, D, AOS>(a.x, pid, d);
#pragma unroll
  for (int d = 0; d < D; ++d) in.v[d] = fldw<T, D, AOS>(a.v, pid, d);
  in.V = a.V(pid);
#pragma unroll
  for (int q = 0; q < D * D; ++q) in.S[q] = fldw<T, D * D, AOS>(a.sigma, pid, q);
  in.l = T(0);
  if constexpr (BASIS == TESS_UGIMP) in.l = a.l(pid) / a.mesh.h;
}

// One layer of class lanes into the stencil offsets a wave owns, in
// registers: the KN offsets along the last axis from vl/dl (that axis's jets
// there), all SW along the others from val/der (axes 0..D-2).  mpe is the
// particle's mass (zero on a lane without a particle, whose jets are finite),
// mpv = mpe v and A = -V σ (column-major).  Offset o = ix + SW*(jy + SW*kz).
template <typename T, int D, int SW, int KN>
__device__ __forceinline__ void p2g_accumulate(const T (*val)[SW], const T (*der)[SW], const T* vl, const T* dl,
                                               const T mpe, const T* mpv, const T* A, T* am,
                                               T (*amv)[Pow<SW, D - 1>::v * KN], T (*af)[Pow<SW, D - 1>::v * KN]) {
  if constexpr (D == 3) {
#pragma unroll
    for (int kz = 0; kz < KN; ++kz) {
#pragma unroll
      for (int jy = 0; jy < SW; ++jy) {
        const T YZ = val[1][jy] * vl[kz];
        const T YdZ = der[1][jy] * vl[kz];
        const T YZd = val[1][jy] * dl[kz];
        const T cm = YZ * mpe;
        T cmv[3], U[3], Wv[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          cmv[c] = YZ * mpv[c];
          U[c] = A[c] * YZ;
          Wv[c] = A[c + 3] * YdZ + A[c + 6] * YZd;
        }
#pragma unroll
        for (int ix = 0; ix < SW; ++ix) {
          const int o = ix + SW * (jy + SW * kz);
          am[o] += val[0][ix] * cm;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            amv[c][o] += val[0][ix] * cmv[c];
            af[c][o] = fma(val[0][ix], Wv[c], fma(der[0][ix], U[c], af[c][o]));
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int jy = 0; jy < KN; ++jy) {
      const T Y = vl[jy], Yd = dl[jy];
      const T cm = Y * mpe;
      T cmv[2], U[2], Wv[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        cmv[c] = Y * mpv[c];
        U[c] = A[c] * Y;
        Wv[c] = A[c + 2] * Yd;
      }
#pragma unroll
      for (int ix = 0; ix < SW; ++ix) {
        const int o = ix + SW * jy;
        am[o] += val[0][ix] * cm;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          amv[c][o] += val[0][ix] * cmv[c];
          af[c][o] = fma(val[0][ix], Wv[c], fma(der[0][ix], U[c], af[c][o]));
        }
      }
    }
  }
}

// Adds one wave's stencil (offsets pass*KN .. pass*KN+KN-1 along the last
// axis) into the tile's node sums in LDS.  Lanes are distinct classes, so for
// one offset their target nodes are distinct; offsets are applied one after
// another (read, add, write: the LDS executes one wave's accesses in order).
template <typename T, int D, int SW, int KN>
__device__ __forceinline__ void p2g_stencil_to_lds(T (*s_tile)[Geo<D>::PSZ], const int* ccoord, int pass,
                                                   const T* am, const T (*amv)[Pow<SW, D - 1>::v * KN],
                                                   const T (*af)[Pow<SW, D - 1>::v * KN]) {
  constexpr int NV = 1 + 2 * D;
  constexpr int NSL = Pow<SW, D - 1>::v * KN;
#pragma unroll
  for (int o = 0; o < NSL; ++o) {
    int r = o, nI[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int off = (d == D - 1) ? pass * KN + r : r % SW;
      nI[d] = ccoord[d] + off;
      r /= SW;
    }
    const int q = pad_node<D>(nI[0], nI[1], nI[2]);
    T t[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) t[v] = s_tile[v][q];
    t[0] += am[o];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      t[1 + c] += amv[c][o];
      t[1 + D + c] += af[c][o];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) s_tile[v][q] = t[v];
    __asm__ volatile("" ::: "memory");  // keep the offsets in program order
  }
}

// The tile's compact partial (Part) from its node sums in LDS: the NT threads
// of the workgroup write one node's NV values each.
template <typename T, int D, int SW, int NT>
__device__ __forceinline__ void p2g_write_partial(const Args<T, D>& a, const int64_t j, T (*s_tile)[Geo<D>::PSZ]) {
  using PT = Part<D, SW>;
  constexpr int NV = 1 + 2 * D;
  T* out = a.partials + int64_t(j) * PT::SIZE;
  for (int n = int(threadIdx.x); n < PT::NODES; n += NT) {
    const int q = pad_node<D>(n % PT::E, (n / PT::E) % PT::E, D == 3 ? n / (PT::E * PT::E) : 0);
    T* o = out + int64_t(n) * NV;
#pragma unroll
    for (int v = 0; v < NV; ++v) o[v] = s_tile[v][q];
  }
}

// With several waves per tile, each owning KN offsets along the last axis,
// wave `pass` adds its stencil into a slab of its own: the PL = KN + BW - 1
// planes (last-axis node coordinates pass*KN ..) that its offsets reach, in
// the padded node order of Geo, one array of PL planes per component.  The
// waves fill their slabs at the same time; the partial is then the sum of the
// slabs in wave order (fixed per-node order, so the sums are deterministic).
template <typename T, int D, int SW, int KN>
struct Slab {
  static constexpr int PL = KN + Geo<D>::BW - 1;
  static constexpr int PITCH = D == 3 ? Geo<D>::PZ : Geo<D>::PY;  // words per plane
  static constexpr int VSTRIDE = PL * PITCH;                     // words per component
  static constexpr int SIZE = (1 + 2 * D) * VSTRIDE;             // words per wave
};

template <typename T, int D, int SW, int KN>
__device__ __forceinline__ void p2g_stencil_to_slab(T* slab, const int* ccoord, int pass, const T* am,
                                                    const T (*amv)[Pow<SW, D - 1>::v * KN],
                                                    const T (*af)[Pow<SW, D - 1>::v * KN]) {
  using SL = Slab<T, D, SW, KN>;
  constexpr int NV = 1 + 2 * D;
  constexpr int NSL = Pow<SW, D - 1>::v * KN;
#pragma unroll
  for (int o = 0; o < NSL; ++o) {
    int r = o, nI[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < D; ++d) {
      nI[d] = ccoord[d] + ((d == D - 1) ? r : r % SW);  // the last axis relative to the slab's first plane
      r /= SW;
    }
    const int q = pad_node<D>(nI[0], nI[1], nI[2]);
    T t[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) t[v] = slab[v * SL::VSTRIDE + q];
    t[0] += am[o];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      t[1 + c] += amv[c][o];
      t[1 + D + c] += af[c][o];
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) slab[v * SL::VSTRIDE + q] = t[v];
    __asm__ volatile("" ::: "memory");  // keep the offsets in program order
  }
}

// The tile's compact partial from the NPASS waves' slabs, summed in wave order;
// NT threads, one node each.
template <typename T, int D, int SW, int KN, int NPASS, int NT>
__device__ __forceinline__ void p2g_write_partial_slabs(const Args<T, D>& a, const int64_t j, const T* slabs) {
  using PT = Part<D, SW>;
  using SL = Slab<T, D, SW, KN>;
  constexpr int NV = 1 + 2 * D;
  T* out = a.partials + int64_t(j) * PT::SIZE;
  for (int n = int(threadIdx.x); n < PT::NODES; n += NT) {
    const int x = n % PT::E, y = (n / PT::E) % PT::E, z = D == 3 ? n / (PT::E * PT::E) : 0;
    const int last = D == 3 ? z : y;
    T sum[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) sum[v] = T(0);
#pragma unroll
    for (int w = 0; w < NPASS; ++w) {
      const int pl = last - w * KN;
      if (pl >= 0 && pl < SL::PL) {
        const int q = D == 3 ? pad_node<3>(x, y, pl) : pad_node<2>(x, pl, 0);
#pragma unroll
        for (int v = 0; v < NV; ++v) sum[v] += slabs[w * SL::SIZE + v * SL::VSTRIDE + q];
      }
    }
    T* o = out + int64_t(n) * NV;
#pragma unroll
    for (int v = 0; v < NV; ++v) o[v] = sum[v];
  }
}

// Float64 in 3D with three offsets per axis: one register set, the layer loaded
// as it is needed.  The set loaded ahead took the kernel to 298 registers, one
// wave per SIMD and one workgroup per CU, with nothing to run while it waits;
// without it two workgroups share a CU.  Taylor rod (1.48 M particles): 288 us
// with two sets, 319 us with one set and one wave per SIMD, 204 us with one set
// and two.  (Four offsets per axis spill hundreds of registers at two waves.)
template <typename T, int D, int BASIS>
constexpr bool p2g_single() {
  return sizeof(T) == 8 && D == 3 && support_width(BASIS) == 3;
}

// NPASS waves per tile: wave w accumulates the offsets w*KN .. w*KN+KN-1
// along the last axis for every class (the particles are read by each wave;
// the registers of one wave hold 1/NPASS of the stencil, which keeps several
// waves per SIMD resident).  The waves add their stencils into the LDS tile
// one after another, so the per-node order of the additions is fixed.
template <typename T, int D, int BASIS, int NPASS, bool AOS, bool BATCH, bool SEP>
__device__ __forceinline__ void k_p2g_fast_body(Args<T, D>& a, const uint32_t* __restrict__ skeys,
                                                          uint32_t* __restrict__ misplaced, const int64_t j) {
  using G = Geo<D>;
  constexpr int SW = support_width(BASIS);
  constexpr int NV = 1 + 2 * D;
  constexpr int KN = SW / NPASS;                       // last-axis offsets per pass
  constexpr int NSL = Pow<SW, D - 1>::v * KN;          // offsets per pass
  constexpr int NT = 64 * NPASS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));  // uniform: scalar branches
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  uint32_t poff;  // a batch's scene: local tile, first particle
  const uint32_t ltile = bind_tile<BATCH>(a, tile, poff);
  int tI[D], origin[D];
  unlin<D>(ltile, a.ntiles, tI);
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = tI[d] * G::BW - 1;

  // The tile's node sums m, mv[D], f[D].  One wave: one array per component
  // over the padded footprint (bank-conflict-free for the class lanes).
  // Several: one slab per wave (Slab), in LDS that the per-layer jet exchange
  // and the staged particle ids use before.
  constexpr bool SHJ = NPASS > 1;
  constexpr bool SINGLE = p2g_single<T, D, BASIS>();
  using SL = Slab<T, D, SW, KN>;
  constexpr int JET_WORDS = SHJ ? 2 * D * 2 * SW * 64 : 0;  // [layer parity][axis][val SW, der SW][lane]
  constexpr int PID_WORDS = PID_CAP * int(sizeof(uint32_t)) / int(sizeof(T));
  constexpr int SUM_WORDS = SHJ ? NPASS * SL::SIZE : NV * G::PSZ;
  constexpr int RAW_WORDS = SHJ ? (SUM_WORDS > JET_WORDS + PID_WORDS ? SUM_WORDS : JET_WORDS + PID_WORDS)
                                : SUM_WORDS + JET_WORDS + PID_WORDS;
  __shared__ __align__(16) T s_raw[RAW_WORDS];
  T* const s_sums = s_raw;
  T(*s_tile)[G::PSZ] = reinterpret_cast<T(*)[G::PSZ]>(s_raw);  // one wave
  T(*s_jet)[D][2 * SW][64] = reinterpret_cast<T(*)[D][2 * SW][64]>(s_raw + (SHJ ? 0 : SUM_WORDS));
  uint32_t* const s_pid = reinterpret_cast<uint32_t*>(s_raw + (SHJ ? JET_WORDS : SUM_WORDS + JET_WORDS));
  __shared__ T s_nodex[D][G::TS];
  __shared__ uint32_t s_cnt[64];
  static_assert(NV * G::PSZ * sizeof(T) % 16 == 0, "LDS tile in 16-byte words");
  static_assert(JET_WORDS * sizeof(T) % 16 == 0 && SUM_WORDS * sizeof(T) % 16 == 0, "16-byte LDS sections");
  if constexpr (!SHJ) {
    for (int q = int(threadIdx.x); q < int(NV * G::PSZ * sizeof(T) / 16); q += NT)
      reinterpret_cast<uint4*>(&s_tile[0][0])[q] = make_uint4(0u, 0u, 0u, 0u);
  }
  stage_nodes<T, D>(a.mesh, origin, s_nodex);
  int ccount, coff, maxcnt;
  tile_class_counts<NPASS>(skeys, start, cnt, s_cnt, ccount, coff, maxcnt, a.perm, poff, s_pid, nullptr,
                           PID_CAP);  // barrier after the staging
  int ccoord[D];
  {
    int r = lane;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      ccoord[d] = r % G::BW;
      r /= G::BW;
    }
  }
  if (wave == 0) check_sparse_support<T, D, SW>(a, origin, ccoord, ccount);
  const T mp = a.mp, hinv = a.mesh.h_inv;
  uint32_t bad = 0, last = 0;
  {
    const int pass = wave;
    T am[NSL], amv[D][NSL], af[D][NSL];
#pragma unroll
    for (int o = 0; o < NSL; ++o) {
      am[o] = T(0);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        amv[c][o] = T(0);
        af[c][o] = T(0);
      }
    }
    // two register sets that alternate between the layer being accumulated and
    // the one being loaded.  Lanes past their class's count compute on the
    // finite data they hold (zeros, or an earlier particle) with zero mass and
    // stress factors, so their contributions are exact zeros.
    P2GIn<T, D> pa, pb;
    std::memset(static_cast<void*>(&pa), 0, sizeof(pa));
    std::memset(static_cast<void*>(&pb), 0, sizeof(pb));
    // particle ids come from LDS (staged with the class counts), a layer ahead
    // of the loads they address
    auto pid_of = [&](int k, auto staged) {
      const int li = coff + k;
      if (k >= ccount) return 0u;
      if constexpr (decltype(staged)::value)
        return s_pid[li];
      else
        return a.perm[start + li] - poff;
    };
    // one layer: the accumulation runs on every lane (a branch around it made
    // the compiler copy all accumulators at each iteration)
    auto layer = [&](int k, const P2GIn<T, D>& cur, P2GIn<T, D>& nxt, uint32_t q_next, uint32_t& q_after,
                     auto staged) {
      if constexpr (!SINGLE) {
        q_after = pid_of(k + 2, staged);
        if (k + 1 < ccount) p2g_load<T, D, BASIS, AOS>(a, q_next, nxt);
      }
      const uint64_t has = __ballot(k < ccount);
      const bool act = k < ccount;
      if (misplaced && pass == 0) bad += broken_pair(has, k, act ? cur.pid : 0u, last);
      T x[D], mpv[D], A[D * D];
      const T mpe = act ? mp : T(0);
#pragma unroll
      for (int d = 0; d < D; ++d) x[d] = cur.x[d];
#pragma unroll
      for (int d = 0; d < D; ++d) mpv[d] = mpe * cur.v[d];  // hoisted mₚ*v[p]
      const T negV = act ? -cur.V : T(0);
#pragma unroll
      for (int q = 0; q < D * D; ++q) A[q] = negV * cur.S[q];  // hoisted (-V[p])*σ[p]
      const T l = cur.l;
      // jets of axes 0..D-2 at all SW offsets, of the last axis at this
      // wave's KN offsets (vl, dl)
      T val[D][SW], der[D][SW], vl[KN], dl[KN];
      auto axis_jets = [&](auto dc, T* jv, T* jd) {
        constexpr int d = decltype(dc)::value;
        const T xi = (x[d] - a.mesh.xmin[d]) * hinv;
        int lo, hi;
        axis_window<T, BASIS>(xi, l, a.mesh.dims[d], lo, hi);
        if constexpr (SEP)
          // inactive lanes carry zero mass and stress: they keep the plain jets, whose values are finite
          // whatever their position (a fit over a window that is not theirs can be singular)
          axis_jets_sep<T, BASIS>(x[d], a.mesh.xmin[d], ccoord[d], hi - lo, s_nodex[d], hinv,
                                  act && sep_corrects<T, D, BASIS>(a, x), jv, jd);
        else
          axis_jets_mixed<T, BASIS>(x[d], a.mesh.xmin[d], ccoord[d], hi - lo, s_nodex[d], l, hinv, jv, jd);
      };
      if constexpr (NPASS == 1) {
        axis_jets(std::integral_constant<int, 0>{}, val[0], der[0]);
        axis_jets(std::integral_constant<int, 1>{}, val[1], der[1]);
        if constexpr (D == 3) axis_jets(std::integral_constant<int, D - 1>{}, val[D - 1], der[D - 1]);
#pragma unroll
        for (int q = 0; q < KN; ++q) {
          vl[q] = val[D - 1][q];
          dl[q] = der[D - 1][q];
        }
      } else {
        // the waves hold the same particles: wave d % NPASS evaluates axis d
        // and shares it through LDS (double-buffered by layer, one barrier)
        const int buf = k & 1;
        auto share = [&](auto dc) {
          T jv[SW], jd[SW];
          axis_jets(dc, jv, jd);
#pragma unroll
          for (int q = 0; q < SW; ++q) {
            s_jet[buf][decltype(dc)::value][q][lane] = jv[q];
            s_jet[buf][decltype(dc)::value][SW + q][lane] = jd[q];
          }
        };
        if (wave == 0 % NPASS) share(std::integral_constant<int, 0>{});
        if (wave == 1 % NPASS) share(std::integral_constant<int, 1>{});
        if constexpr (D == 3) {
          if (wave == 2 % NPASS) share(std::integral_constant<int, D - 1>{});
        }
        __syncthreads();
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
#pragma unroll
          for (int q = 0; q < SW; ++q) {
            val[d][q] = s_jet[buf][d][q][lane];
            der[d][q] = s_jet[buf][d][SW + q][lane];
          }
#pragma unroll
        for (int q = 0; q < KN; ++q) {
          vl[q] = s_jet[buf][D - 1][pass * KN + q][lane];
          dl[q] = s_jet[buf][D - 1][SW + pass * KN + q][lane];
        }
      }
      p2g_accumulate<T, D, SW, KN>(val, der, vl, dl, mpe, mpv, A, am, amv, af);
    };
    auto walk = [&](auto staged) {
      if constexpr (SINGLE) {
        uint32_t qa = 0u, qb = 0u;
        for (int k = 0; k < maxcnt; ++k) {
          if (k < ccount) p2g_load<T, D, BASIS, AOS>(a, pid_of(k, staged), pa);
          layer(k, pa, pb, qa, qb, staged);
        }
        return;
      }
      uint32_t qa = pid_of(1, staged), qb = 0u;
      if (ccount > 0) p2g_load<T, D, BASIS, AOS>(a, pid_of(0, staged), pa);
      for (int k = 0; k < maxcnt; k += 2) {
        layer(k, pa, pb, qa, qb, staged);
        if (k + 1 < maxcnt) layer(k + 1, pb, pa, qb, qa, staged);
      }
    };
    if (cnt <= PID_CAP)
      walk(std::true_type{});
    else
      walk(std::false_type{});
    if constexpr (SHJ) {
      // the slabs take the LDS of the jet exchange and the ids: after every
      // wave's last layer.  Each wave zeroes and fills its own slab (the LDS
      // executes one wave's accesses in order)
      __syncthreads();
      T* const slab = s_sums + pass * SL::SIZE;
      static_assert(SL::SIZE * sizeof(T) % 16 == 0, "slabs in 16-byte words");
      for (int q = lane; q < int(SL::SIZE * sizeof(T) / 16); q += 64)
        reinterpret_cast<uint4*>(slab)[q] = make_uint4(0u, 0u, 0u, 0u);
      if (ccount > 0) p2g_stencil_to_slab<T, D, SW, KN>(slab, ccoord, pass, am, amv, af);
      __syncthreads();
    } else {
      // lanes are distinct classes, so for one offset their target nodes are
      // distinct; offsets are applied one after another (read, add, write: the
      // LDS executes one wave's accesses in order)
      if (ccount > 0) p2g_stencil_to_lds<T, D, SW, KN>(s_tile, ccoord, pass, am, amv, af);
      __syncthreads();
    }
  }
  if (misplaced && wave == 0) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) bad += __shfl_xor(bad, off, 64);
    if (lane == 0 && bad) atomicAdd(lane_of(misplaced, LANE_BROKEN), bad);
  }
  if constexpr (SHJ)
    p2g_write_partial_slabs<T, D, SW, KN, NPASS, NT>(a, j, s_sums);
  else
    p2g_write_partial<T, D, SW, NT>(a, j, s_tile);
}

template <typename T, int D, int BASIS, int NPASS, bool AOS, bool BATCH = false, bool SEP = false>
__global__ __launch_bounds__(64 * NPASS, (p2g_single<T, D, BASIS>() ? 2 : 1)) void k_p2g_fast(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                          uint32_t* __restrict__ misplaced) {
  const int64_t j = item_of<BATCH>(blockIdx.x, a.n_active);
  if (j < a.n_active) k_p2g_fast_body<T, D, BASIS, NPASS, AOS, BATCH, SEP>(a, skeys, misplaced, j);
}

// Forms whose item count is read on the device at `count` (launch sizes fixed
// in advance): one workgroup per possible item, those past the count ending
// at once (_grid), or a persistent grid sized to the device walking the items
// (_persist; a multiple of 8 workgroups keeps each XCD on a contiguous run of
// them, as xcd_remap does for one workgroup per item).
template <typename T, int D, int BASIS, int NPASS, bool AOS, bool BATCH = false, bool SEP = false>
__global__ __launch_bounds__(64 * NPASS) void k_p2g_fast_grid(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                          uint32_t* __restrict__ misplaced, const uint32_t* __restrict__ count) {
  const int64_t N = int64_t(*count), R = ((N + 7) >> 3) << 3;
  // xcd_remap is a bijection of [0, R) only: workgroups past R end here
  const int64_t j = item_of<BATCH>(blockIdx.x, N);
  if (int64_t(blockIdx.x) < R && j < N) k_p2g_fast_body<T, D, BASIS, NPASS, AOS, BATCH, SEP>(a, skeys, misplaced, j);
}
template <typename T, int D, int BASIS, int NPASS, bool AOS, bool BATCH = false, bool SEP = false>
__global__ __launch_bounds__(64 * NPASS) void k_p2g_fast_persist(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                          uint32_t* __restrict__ misplaced, const uint32_t* __restrict__ count) {
  const int64_t N = int64_t(*count), R = ((N + 7) >> 3) << 3;
  for (int64_t it = blockIdx.x; it < R; it += gridDim.x) {
    const int64_t j = item_of<BATCH>(it, N);
    if (j < N) k_p2g_fast_body<T, D, BASIS, NPASS, AOS, BATCH, SEP>(a, skeys, misplaced, j);
    __syncthreads();  // the next item reuses the workgroup's LDS
  }
}


// G2P with the footprint's v and v - vⁿ staged per node in LDS; the FLIP
// increment is formed from the node differences as the reference does.  NW
// waves share one tile: wave w walks the class-major order at k = w, w+NW, ...
// and prefetches its next particle while updating the current one.
template <typename T, int D, bool AOS>
struct G2PIn {
  uint32_t pid, cls, key;  // particle, window-start class in the tile, sort key at its slot
  uint32_t dst;            // index its updated state is written at
  T x[D], v[D], F[D * D], l;
};

template <typename T, int D, int BASIS, bool AOS>
__device__ __forceinline__ void g2p_load(const Args<T, D>& a, uint32_t pid, G2PIn<T, D, AOS>& in) {
  in.pid = pid;
#pragma unroll
  for (int c = 0; c < D; ++c) in.x[c] = fldw<T, D, AOS>(a.x, pid, c);
#pragma unroll
  for (int c = 0; c < D; ++c) in.v[c] = fldw<T, D, AOS>(a.v, pid, c);
#pragma unroll
  for (int q = 0; q < D * D; ++q) in.F[q] = fldw<T, D * D, AOS>(a.F, pid, q);
  in.l = T(0);
  if constexpr (BASIS == TESS_UGIMP) in.l = a.l(pid) / a.mesh.h;
}

// Stages a tile's footprint for G2P in two halves: g2p_stage_load issues the
// grid loads of v and vⁿ (zeros outside the grid) into registers, and
// g2p_stage_store writes v and v - vⁿ per component in the padded node order
// of Geo, with the footprint's node coordinates per axis; NT threads.  The
// loads stay in flight across the barriers in between (a barrier waits only on
// LDS operations), so the caller issues the tile's key and id loads before the
// grid values are needed, and one memory round trip serves both.  The caller
// synchronises after the store.
template <typename T, int D, int NT>
struct G2PStage {
  static constexpr int NPER = (Geo<D>::NFOOT + NT - 1) / NT;
  T v[NPER][D], vn[NPER][D];
};

template <typename T, int D, int NT>
__device__ __forceinline__ void g2p_stage_load(const Args<T, D>& a, const int* origin, G2PStage<T, D, NT>& st) {
  using G = Geo<D>;
#pragma unroll
  for (int u = 0; u < G2PStage<T, D, NT>::NPER; ++u) {
    const int q = int(threadIdx.x) + u * NT;
    int I[D], r = q;
    bool in = q < G::NFOOT;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      I[d] = origin[d] + r % G::TS;
      r /= G::TS;
      in = in && I[d] >= 0 && I[d] < a.mesh.dims[d];
    }
    const int64_t i = in ? grid_slot(a, I) : -1;
    in = i >= 0;
#pragma unroll
    for (int c = 0; c < D; ++c) {
      st.v[u][c] = in ? a.gv(i, c) : T(0);
      st.vn[u][c] = in ? a.gvn(i, c) : T(0);
    }
  }
}

template <typename T, int D, int NT>
__device__ __forceinline__ void g2p_stage_store(const Args<T, D>& a, const int* origin,
                                                const G2PStage<T, D, NT>& st, T (*s_n)[Geo<D>::PSZ],
                                                T (*s_nodex)[Geo<D>::TS]) {
  using G = Geo<D>;
#pragma unroll
  for (int u = 0; u < G2PStage<T, D, NT>::NPER; ++u) {
    const int q = int(threadIdx.x) + u * NT;
    if (q < G::NFOOT) {
      const int pq = pad_node<D>(q % G::TS, (q / G::TS) % G::TS, D == 3 ? q / (G::TS * G::TS) : 0);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        s_n[c][pq] = st.v[u][c];
        s_n[D + c][pq] = st.v[u][c] - st.vn[u][c];
      }
    }
  }
  stage_nodes<T, D>(a.mesh, origin, s_nodex);
}

// Writes of one field of NC components from a wave's particles through LDS, in
// storage order: lane l holds the components of the particle written at index
// dst, and the wave stores NC times 64 consecutive scalars of the sequence
// (particle of lane 0, 1, ...).  Where the particles of neighbouring lanes are
// neighbours in storage, each store instruction covers whole lines.
//
// A 3D particle's Mat is 9 scalars: stored straight from registers, every
// instruction touched 64 pieces of 8-16 bytes, each a write request of its own
// (6.3 requests per particle in Float32, 20 in Float64), and the address unit
// was busy throughout the kernel.
template <typename T, int NC>
struct RowStore {
  uint32_t off[NC];  // scalar offsets this lane writes, ~0: none
  // dst0: index * NC of the lane's particle; act: whether the lane has one
  __device__ __forceinline__ void prepare(uint32_t dst, bool act) {
    const int lane = int(threadIdx.x & 63);
    const uint32_t q = act ? uint32_t(NC) * (dst - uint32_t(lane)) : ~0u;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int w = i * 64 + lane;
      const uint32_t ql = uint32_t(__shfl(int(q), w / NC, 64));
      off[i] = ql == ~0u ? ~0u : ql + uint32_t(w);
    }
  }
  __device__ __forceinline__ void store(T* __restrict__ base, const T* v, T* s) const {
    const int lane = int(threadIdx.x & 63);
#pragma unroll
    for (int c = 0; c < NC; ++c) s[lane * NC + c] = v[c];
    __asm__ volatile("" ::: "memory");  // the LDS executes one wave's accesses in order
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const T t = s[i * 64 + lane];
      if (off[i] != ~0u) base[off[i]] = t;
    }
    __asm__ volatile("" ::: "memory");
  }
};

// One particle's G2P and update (README.md:81-86) from the tile's staged
// footprint (s_n: v and v - vⁿ per component; s_nodex: node coordinates): its
// axis jets at its class window, the axis-factored sums of Δv, ∇v and the x
// rate, the writes of v, ∇v, x, F, σ, V and, with mo.nk, of the next sort key
// at its sorted slot jj (next_key).  emit(val, der, v, σ, V) receives the
// jets and the updated state.  ROWS: called by the whole wave (act: the lane
// has a particle; a lane without one computes on what it holds and writes
// nothing), the Vec and Mat fields are written through s_row (64 D² scalars of
// the wave's own).
template <typename T, int D, int BASIS, bool AOS, bool SEP, bool ROWS, bool NT, typename Emit>
__device__ __forceinline__ void g2p_particle(const Args<T, D>& a, const G2PIn<T, D, AOS>& cur,
                                             const T (*s_n)[Geo<D>::PSZ], const T (*s_nodex)[Geo<D>::TS],
                                             const uint32_t jj, const uint32_t tile, const uint32_t ltile,
                                             const uint32_t start, const MoveOut& mo, TileMoves* s_mv,
                                             uint32_t& moved, const uint32_t ntiles, const bool act, T* s_row,
                                             Emit&& emit) {
  using G = Geo<D>;
  constexpr int SW = support_width(BASIS);
  const T hinv = a.mesh.h_inv, dt = a.dt;
  int cc[D];  // the particle's class coordinates (its window's offset in the footprint)
  {
    uint32_t r = cur.cls;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      cc[d] = int(r % G::BW);
      r /= G::BW;
    }
  }
  T val[D][SW], der[D][SW];
  T X[D], DV[D], L[D * D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    X[c] = T(0);
    DV[c] = T(0);
  }
#pragma unroll
  for (int q = 0; q < D * D; ++q) L[q] = T(0);
  // (a branch of its own: hoisted among the loads of the next particle and the
  // stores below, the gather's LDS reads took 175 registers to scratch)
  if (act) {
  bool corrects = false;
  if constexpr (SEP) corrects = sep_corrects<T, D, BASIS>(a, cur.x);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const T xi = (cur.x[d] - a.mesh.xmin[d]) * hinv;
    int lo, hi;
    axis_window<T, BASIS>(xi, cur.l, a.mesh.dims[d], lo, hi);
    if constexpr (SEP)
      axis_jets_sep<T, BASIS>(cur.x[d], a.mesh.xmin[d], cc[d], hi - lo, s_nodex[d], hinv, corrects, val[d],
                              der[d]);
    else
      axis_jets_mixed<T, BASIS>(cur.x[d], a.mesh.xmin[d], cc[d], hi - lo, s_nodex[d], cur.l, hinv, val[d],
                                der[d]);
  }
  // X = Σ w v_i, DV = Σ w (v_i - vⁿ_i), L = Σ v_i ⊗ ∇w, factored by axis
  if constexpr (D == 3) {
#pragma unroll
    for (int kz = 0; kz < SW; ++kz)
#pragma unroll
      for (int jy = 0; jy < SW; ++jy) {
        T S1[3] = {T(0), T(0), T(0)}, S2[3] = {T(0), T(0), T(0)}, Sd[3] = {T(0), T(0), T(0)};
#pragma unroll
        for (int ix = 0; ix < SW; ++ix) {
          const int q = pad_node<3>(cc[0] + ix, cc[1] + jy, cc[2] + kz);
          T nd[6];
#pragma unroll
          for (int u = 0; u < 6; ++u) nd[u] = s_n[u][q];
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            S1[c] += val[0][ix] * nd[c];
            S2[c] += der[0][ix] * nd[c];
            Sd[c] += val[0][ix] * nd[3 + c];
          }
        }
        const T YZ = val[1][jy] * val[2][kz];
        const T YdZ = der[1][jy] * val[2][kz];
        const T YZd = val[1][jy] * der[2][kz];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          X[c] += YZ * S1[c];
          DV[c] += YZ * Sd[c];
          L[c] += YZ * S2[c];
          L[c + 3] += YdZ * S1[c];
          L[c + 6] += YZd * S1[c];
        }
      }
  } else {
#pragma unroll
    for (int jy = 0; jy < SW; ++jy) {
      T S1[2] = {T(0), T(0)}, S2[2] = {T(0), T(0)}, Sd[2] = {T(0), T(0)};
#pragma unroll
      for (int ix = 0; ix < SW; ++ix) {
        const int q = pad_node<2>(cc[0] + ix, cc[1] + jy, 0);
        T nd[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) nd[u] = s_n[u][q];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          S1[c] += val[0][ix] * nd[c];
          S2[c] += der[0][ix] * nd[c];
          Sd[c] += val[0][ix] * nd[2 + c];
        }
      }
      const T Y = val[1][jy], Yd = der[1][jy];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        X[c] += Y * S1[c];
        DV[c] += Y * Sd[c];
        L[c] += Y * S2[c];
        L[c + 2] += Yd * S1[c];
      }
    }
  }
  }
  const uint32_t pid = cur.pid, dst = cur.dst;
  RowStore<T, D> rows;
  RowStore<T, D * D> mats;
  if constexpr (ROWS) {
    rows.prepare(dst, act);
    mats.prepare(dst, act);
  }
  auto put_vec = [&](const DField<T>& f, const T* v) {
    if constexpr (ROWS) {
      rows.store(f.p, v, s_row);
    } else {
#pragma unroll
      for (int c = 0; c < D; ++c) st_g2p<NT>(fldw<T, D, AOS>(f, dst, c), v[c]);
    }
  };
  auto put_mat = [&](const DField<T>& f, const T* v) {
    if constexpr (ROWS) {
      mats.store(f.p, v, s_row);
    } else {
#pragma unroll
      for (int q = 0; q < D * D; ++q) st_g2p<NT>(fldw<T, D * D, AOS>(f, dst, q), v[q]);
    }
  };
  // particle equations (README.md:81-86)
  T vn[D];
#pragma unroll
  for (int c = 0; c < D; ++c) vn[c] = cur.v[c] + DV[c];
  put_vec(a.ov, vn);
  put_mat(a.ogradv, L);
  T xn[D];
#pragma unroll
  for (int c = 0; c < D; ++c) xn[c] = cur.x[c] + X[c] * dt;
  put_vec(a.ox, xn);
  if (a.x_keep && act) {
#pragma unroll
    for (int c = 0; c < D; ++c) a.x_keep[int64_t(dst) * D + c] = cur.x[c];
  }
  if (mo.nk) {
    uint32_t nl = 1;  // the scene's tiles; in a batch its keys start at its first global tile
#pragma unroll
    for (int d = 0; d < D; ++d) nl *= uint32_t(a.ntiles[d]);
    const uint32_t kl = key_of_position<T, D, BASIS>(a, xn, cur.l, nl);
    const uint32_t key = kl == nl * 64u ? ntiles * 64u : kl + (tile - ltile) * 64u;
    constexpr bool OWN = D == 3 && sizeof(T) == 8;
    if (!ROWS || act) next_key<OWN, !OWN>(mo, key, cur.key, jj, tile, start, ntiles, s_mv, moved);
  }
  T Fn[D * D];
#pragma unroll
  for (int b = 0; b < D; ++b)
#pragma unroll
    for (int r = 0; r < D; ++r) {
      T t = L[r] * cur.F[D * b];  // (I + Δt∇v) F = F + Δt (∇v F)
#pragma unroll
      for (int kk = 1; kk < D; ++kk) t += L[r + D * kk] * cur.F[kk + D * b];
      Fn[r + D * b] = cur.F[r + D * b] + dt * t;
    }
  put_mat(a.oF, Fn);
  T sg[D * D], Vn;
  neo_hookean<T, D>(Fn, a.lambda, a.mu, a.V0, a.logE.p != nullptr, a.logE.p ? a.logE(pid) : T(0), sg, Vn);
  put_mat(a.osigma, sg);
  if (!ROWS || act) st_g2p<NT>(a.oV(dst), Vn);
  emit(val, der, vn, sg, Vn);
}

// With mo.nk != nullptr the kernel also writes, at each particle's sorted
// position, the sort key of its new position, and per tile what the next
// step's binning starts from (MoveOut).
// waves per SIMD the Float32 G2P is compiled for (VGPR budget 512 / n), and
// waves per tile of the single-scene G2P
#ifndef TESS_G2P_WAVES_PER_SIMD
#define TESS_G2P_WAVES_PER_SIMD 3
#endif
#ifndef TESS_G2P_WAVES_PER_TILE
#define TESS_G2P_WAVES_PER_TILE 4
#endif
template <typename T, int D, int BASIS, bool AOS, int NW, bool BATCH, bool SEP, bool NT>
__device__ __forceinline__ void k_g2p_fast_body(Args<T, D>& a, const uint32_t* __restrict__ skeys,
                                                       const MoveOut mo, uint32_t ntiles, const int64_t j) {
  using G = Geo<D>;
  constexpr int SW = support_width(BASIS);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));  // uniform: scalar branches
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  uint32_t poff;  // a batch's scene: local tile, first particle
  const uint32_t ltile = bind_tile<BATCH>(a, tile, poff);
  int tI[D], origin[D];
  unlin<D>(ltile, a.ntiles, tI);
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = tI[d] * G::BW - 1;
  // per component (v[D], then v-vⁿ[D]) the footprint in the padded
  // bank-conflict-free node order of Geo
  __shared__ T s_n[2 * D][G::PSZ];
  __shared__ T s_nodex[D][G::TS];
  __shared__ uint32_t s_cnt[64];
  __shared__ TileMoves s_mv;
  uint32_t moved = 0;
  if (threadIdx.x == 0) s_mv = TileMoves{0u, 0u, 0u};  // before the barriers below
  G2PStage<T, D, 64 * NW> stage;
  g2p_stage_load<T, D, 64 * NW>(a, origin, stage);
  int ccount, coff, maxcnt;
  __shared__ uint32_t s_pid[G2P_PID_CAP<D>], s_key[G2P_PID_CAP<D>];
  // 3D Float64 Julia-layout fields leave through LDS rows (RowStore): 573 us
  // without and 260 us with them on the Taylor rod (1.48 M particles).  In
  // Float32 the rows' instructions and registers cost more than the requests
  // they save (840 us without, 938 us with them on the 13.4 M-particle block);
  // a 2D particle's Vec and Mat are 2 and 4 scalars, which the lanes store
  // contiguously as they are.
  constexpr bool ROWS = D == 3 && AOS && sizeof(T) == 8;
  __shared__ T s_rows[ROWS ? NW : 1][ROWS ? 64 * D * D : 1];
  T* const s_row = s_rows[ROWS ? wave : 0];
  tile_class_counts<NW>(skeys, start, cnt, s_cnt, ccount, coff, maxcnt, a.perm, poff, s_pid, s_key,
                        G2P_PID_CAP<D>);  // barrier after the staging of ids and keys
  g2p_stage_store<T, D, 64 * NW>(a, origin, stage, s_n, s_nodex);
  __syncthreads();
  // Two walks of the tile's particles.  Class order (lane = class, iteration k =
  // the k-th particle of every class) reads the layered storage contiguously
  // and takes maxcnt iterations.  Sorted order (iteration k = sorted positions
  // 64k .. 64k+63) takes ceil(cnt/64); a tile whose classes are uneven or
  // sparse uses it when that saves a third of the iterations.
  const int n_sorted = (cnt + 63) / 64;
  const bool by_sorted = 3 * n_sorted < 2 * maxcnt;
  const int kend = by_sorted ? n_sorted : maxcnt;
  auto live = [&](int k) { return by_sorted ? k * 64 + lane < cnt : k < ccount; };
  auto slot = [&](int k) { return start + uint32_t(by_sorted ? k * 64 + lane : coff + k); };  // sorted position
  // a particle's id and sort key come from LDS (staged with the class
  // counts), an iteration ahead of the loads they address: those loads do not
  // wait behind the previous particle's stores, as a global load of the id
  // would (the memory counter drains in issue order)
  struct Ahead {
    uint32_t pid, key;
  };
  // staged: the tile's ids are all in LDS (cnt <= G2P_PID_CAP<D>); the walk is
  // compiled for each case so that neither waits on the other's loads
  auto ahead = [&](int k, auto staged) {
    Ahead r{0u, 0u};
    if (live(k)) {
      const uint32_t li = slot(k) - start;
      if constexpr (decltype(staged)::value) {
        r.pid = s_pid[li];
        r.key = s_key[li];
      } else {
        r.pid = a.perm[start + li] - poff;
        r.key = skeys[start + li];
      }
    }
    return r;
  };
  auto fetch = [&](int k, const Ahead& q, G2PIn<T, D, AOS>& in) {
    if (!live(k)) return;
    g2p_load<T, D, BASIS, AOS>(a, q.pid, in);
    in.dst = a.dest ? a.dest[slot(k)] : q.pid;
    in.key = q.key;
    in.cls = by_sorted ? q.key & 63u : uint32_t(lane);
  };
  // two register sets alternate between the particle being updated and the
  // one being loaded (wave w walks k = w, w+NW, ...)
  G2PIn<T, D, AOS> pa, pb;
  std::memset(static_cast<void*>(&pa), 0, sizeof(pa));
  std::memset(static_cast<void*>(&pb), 0, sizeof(pb));
  auto particle = [&](int k, const G2PIn<T, D, AOS>& cur, G2PIn<T, D, AOS>& nxt, const Ahead& q_next,
                      Ahead& q_after, auto staged) {
    const bool act = live(k);
    q_after = ahead(k + 2 * NW, staged);
    fetch(k + NW, q_next, nxt);
    if constexpr (!ROWS) {
      if (!act) return;
    }
    g2p_particle<T, D, BASIS, AOS, SEP, ROWS, NT>(a, cur, s_n, s_nodex, mo.nk ? slot(k) : 0u, tile, ltile, start, mo,
                                              &s_mv, moved, ntiles, act, s_row, [](const auto&...) {});
  };
  auto walk = [&](auto staged) {
    Ahead qa = ahead(wave + NW, staged), qb{0u, 0u};
    fetch(wave, ahead(wave, staged), pa);
    for (int k = wave; k < kend; k += 2 * NW) {
      particle(k, pa, pb, qa, qb, staged);
      if (k + NW < kend) particle(k + NW, pb, pa, qb, qa, staged);
    }
  };
  if (cnt <= G2P_PID_CAP<D>)
    walk(std::true_type{});
  else
    walk(std::false_type{});
  if (mo.nk) tile_moves_end(mo, tile, start, cnt, ntiles, &s_mv, moved);
}

template <typename T, int D, int BASIS, bool AOS, int NW, bool BATCH = false, bool SEP = false, bool NT = false>
__global__ __launch_bounds__(64 * NW, sizeof(T) == 4 ? TESS_G2P_WAVES_PER_SIMD : 2) void k_g2p_fast(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                       const MoveOut mo, uint32_t ntiles) {
  const int64_t j = item_of<BATCH>(blockIdx.x, a.n_active);
  if (j < a.n_active) k_g2p_fast_body<T, D, BASIS, AOS, NW, BATCH, SEP, NT>(a, skeys, mo, ntiles, j);
}

// Forms whose item count is read on the device at `count` (launch sizes fixed
// in advance): one workgroup per possible item, those past the count ending
// at once (_grid), or a persistent grid sized to the device walking the items
// (_persist; a multiple of 8 workgroups keeps each XCD on a contiguous run of
// them, as xcd_remap does for one workgroup per item).
template <typename T, int D, int BASIS, bool AOS, int NW, bool BATCH = false, bool SEP = false>
__global__ __launch_bounds__(64 * NW, sizeof(T) == 4 ? TESS_G2P_WAVES_PER_SIMD : 2) void k_g2p_fast_grid(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                       const MoveOut mo, uint32_t ntiles, const uint32_t* __restrict__ count) {
  const int64_t N = int64_t(*count), R = ((N + 7) >> 3) << 3;
  // xcd_remap is a bijection of [0, R) only: workgroups past R end here
  const int64_t j = item_of<BATCH>(blockIdx.x, N);
  if (int64_t(blockIdx.x) < R && j < N) k_g2p_fast_body<T, D, BASIS, AOS, NW, BATCH, SEP, false>(a, skeys, mo, ntiles, j);
}
template <typename T, int D, int BASIS, bool AOS, int NW, bool BATCH = false, bool SEP = false>
__global__ __launch_bounds__(64 * NW, sizeof(T) == 4 ? TESS_G2P_WAVES_PER_SIMD : 2) void k_g2p_fast_persist(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                       const MoveOut mo, uint32_t ntiles, const uint32_t* __restrict__ count) {
  const int64_t N = int64_t(*count), R = ((N + 7) >> 3) << 3;
  for (int64_t it = blockIdx.x; it < R; it += gridDim.x) {
    const int64_t j = item_of<BATCH>(it, N);
    if (j < N) k_g2p_fast_body<T, D, BASIS, AOS, NW, BATCH, SEP, false>(a, skeys, mo, ntiles, j);
    __syncthreads();  // the next item reuses the workgroup's LDS
  }
}


// ---- gather + grid-node half ------------------------------------------------
// ---- single-sweep @G2P2G -------------------------------------------------------
//
// One pass over a tile's particles runs both halves of a @G2P2G program
// (src/Transfer/g2p2g.jl:100-159) with one set of weights, those of the
// positions before the pass.  NP producer waves run the G2P half, one layer of
// class lanes each per round (the k-th particle of every class, as k_g2p_fast
// walks them: gather, update, writes).  They hand each particle's position
// before the update, mass, mₚv and -Vσ to NC consumer waves through LDS.  The
// consumers evaluate the jets of that position, own the stencil offsets of
// k_p2g_fast's waves and accumulate those layers one round behind the
// producers (double-buffered exchange, one barrier per round).
// They see the layers in k_p2g_fast's order and run its arithmetic, so the
// tile's partial is the one that the G2P kernel followed by the P2G kernel at
// the kept positions produces.  The particles are read once per pass instead
// of twice, and the G2P half's memory waits overlap the P2G half's arithmetic.
//
// σ is exchanged as its D(D+1)/2 distinct entries: neo_hookean forms it
// symmetric to the last bit (both triangles from the same products).

// index of σ's entry (r, b), r >= b, among the distinct entries
__host__ __device__ constexpr int sym_index(int r, int b, int D) { return b * D - b * (b - 1) / 2 + (r - b); }

// producer waves of the single-sweep kernel (0: as many as the LDS budget allows)
#ifndef TESS_G2P2G_PRODUCERS
#define TESS_G2P2G_PRODUCERS 0
#endif
template <typename T, int D, int BASIS>
struct G2P2GShape {
  static constexpr int SW = support_width(BASIS);
  static constexpr int NV = 1 + 2 * D;
  static constexpr int NS = D * (D + 1) / 2;
  static constexpr bool HAS_L = BASIS == TESS_UGIMP;
  // exchange rows per particle: x[D] (and l) before the update, mass, mₚv[D], -Vσ[NS]
  static constexpr int XL = D, XM = D + (HAS_L ? 1 : 0), XV = XM + 1, XA = XV + D, XR = XA + NS;
  // consumer waves: those of k_p2g_fast (3D: one per last-axis offset; 2D: one
  // while the stencil's accumulators fit)
  static constexpr int NC = (D == 3 || Pow<SW, D>::v * NV * int(sizeof(T)) / 4 > 96) ? SW : 1;
  static constexpr int lds(int np) {
    return int(sizeof(T)) * (2 * np * XR * 64 + 2 * D * Geo<D>::PSZ + D * Geo<D>::TS) + 4 * (2 * PID_CAP + 64);
  }
  // producer waves: eight waves per workgroup, two workgroups per CU at 128
  // VGPRs (Float32)
  static constexpr int NP_AUTO = 8 - NC;
  static constexpr int NP = TESS_G2P2G_PRODUCERS > 0 ? TESS_G2P2G_PRODUCERS : NP_AUTO;
  // waves per SIMD to compile for: as many workgroups per CU as the LDS holds
  // (at most two), at most 4 waves per SIMD; Float64 1
  static constexpr int wps(int np) {
    const int wg = lds(np) <= 80 * 1024 ? 2 : 1;
    const int w = (wg * (np + NC) + 3) / 4;
    return sizeof(T) != 4 ? 1 : w < 1 ? 1 : w > 4 ? 4 : w;
  }
};

template <typename T, int D, int BASIS, bool AOS, int NP, int NC>
__device__ __forceinline__ void k_g2p2g_fast_body(Args<T, D>& a, const uint32_t* __restrict__ skeys,
                                                  const MoveOut mo, uint32_t ntiles,
                                                  uint32_t* __restrict__ misplaced, const int64_t j) {
  using G = Geo<D>;
  using SH = G2P2GShape<T, D, BASIS>;
  constexpr int SW = SH::SW, NV = SH::NV, XR = SH::XR, XM = SH::XM, XV = SH::XV, XA = SH::XA;
  constexpr int KN = SW / NC;                   // last-axis offsets per consumer
  constexpr int NSL = Pow<SW, D - 1>::v * KN;  // offsets per consumer
  constexpr int NT = 64 * (NP + NC);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));  // uniform: scalar branches
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  uint32_t poff;
  const uint32_t ltile = bind_tile<false>(a, tile, poff);
  int tI[D], origin[D];
  unlin<D>(ltile, a.ntiles, tI);
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = tI[d] * G::BW - 1;
  __shared__ T s_n[2 * D][G::PSZ];
  __shared__ T s_nodex[D][G::TS];
  __shared__ uint32_t s_cnt[64];
  __shared__ uint32_t s_pid[PID_CAP], s_key[PID_CAP];
  __shared__ TileMoves s_mv;
  uint32_t moved = 0;
  if (threadIdx.x == 0) s_mv = TileMoves{0u, 0u, 0u};  // before the barriers below
  // [round parity][producer][row][class lane]; after the last round the
  // tile's node sums take its place: the consumers' slabs (several consumers)
  // or one array per component over the footprint (one)
  using SL = Slab<T, D, SW, KN>;
  constexpr int XWORDS = 2 * NP * XR * 64;
  constexpr int SUMW = NC > 1 ? NC * SL::SIZE : NV * G::PSZ;
  __shared__ __align__(16) T s_xraw[XWORDS > SUMW ? XWORDS : SUMW];
  T(*s_x)[NP][XR][64] = reinterpret_cast<T(*)[NP][XR][64]>(s_xraw);
  T(*s_tile)[G::PSZ] = reinterpret_cast<T(*)[G::PSZ]>(s_xraw);
  G2PStage<T, D, NT> stage;
  g2p_stage_load<T, D, NT>(a, origin, stage);
  int ccount, coff, maxcnt;
  tile_class_counts<NP + NC>(skeys, start, cnt, s_cnt, ccount, coff, maxcnt, a.perm, poff, s_pid, s_key,
                             PID_CAP);  // barrier after the staging of ids and keys
  g2p_stage_store<T, D, NT>(a, origin, stage, s_n, s_nodex);
  __syncthreads();
  const int nround = (maxcnt + NP - 1) / NP;  // the same in every wave
  auto zero_tile = [&]() {
    static_assert(NV * G::PSZ * sizeof(T) % 16 == 0, "node sums in 16-byte words");
    for (int q = int(threadIdx.x); q < int(NV * G::PSZ * sizeof(T) / 16); q += NT)
      reinterpret_cast<uint4*>(&s_tile[0][0])[q] = make_uint4(0u, 0u, 0u, 0u);
  };
  // Both roles pass the same barriers: nround + 1 in the rounds, then one after
  // the consumers fill their slabs (several consumers), or one after the node
  // sums are zeroed and one as the consumer adds its stencil (one).
  if (wave < NP) {
    // producer: layers k = wave, wave + NP, ... (round r takes k = r*NP + wave)
    auto ahead = [&](int k, auto staged) {
      uint32_t pid = 0u, key = 0u;
      if (k < ccount) {
        if constexpr (decltype(staged)::value) {
          pid = s_pid[coff + k];
          key = s_key[coff + k];
        } else {
          pid = a.perm[start + coff + k] - poff;
          key = skeys[start + coff + k];
        }
      }
      return uint2{pid, key};
    };
    auto fetch = [&](int k, const uint2& q, G2PIn<T, D, AOS>& in) {
      if (k >= ccount) return;
      g2p_load<T, D, BASIS, AOS>(a, q.x, in);
      in.dst = q.x;
      in.key = q.y;
      in.cls = uint32_t(lane);
    };
    G2PIn<T, D, AOS> pa, pb;
    std::memset(static_cast<void*>(&pa), 0, sizeof(pa));
    std::memset(static_cast<void*>(&pb), 0, sizeof(pb));
    auto produce = [&](int r, const G2PIn<T, D, AOS>& cur, G2PIn<T, D, AOS>& nxt, const uint2& q_next, uint2& q_after,
                     auto staged) {
      if (r < nround) {
        const int k = r * NP + wave;
        q_after = ahead(k + 2 * NP, staged);
        fetch(k + NP, q_next, nxt);
        T(*xr)[64] = s_x[r & 1][wave];
        if (k < ccount) {
          g2p_particle<T, D, BASIS, AOS, false, false, sizeof(T) == 4>(
              a, cur, s_n, s_nodex, start + uint32_t(coff + k), tile, ltile, start, mo, &s_mv, moved, ntiles, true,
              static_cast<T*>(nullptr),
              [&](const auto&, const auto&, const auto& vn, const auto& sg, const T Vn) {
#pragma unroll
                for (int d = 0; d < D; ++d) xr[d][lane] = cur.x[d];
                if constexpr (SH::HAS_L) xr[SH::XL][lane] = cur.l;
                const T mp = a.mp;
                xr[XM][lane] = mp;
#pragma unroll
                for (int c = 0; c < D; ++c) xr[XV + c][lane] = mp * vn[c];
                const T negV = -Vn;
#pragma unroll
                for (int b = 0; b < D; ++b)
#pragma unroll
                  for (int rr = b; rr < D; ++rr) xr[XA + sym_index(rr, b, D)][lane] = negV * sg[rr + D * b];
              });
        } else {
          // no particle: a finite position, zero mass and stress (exact zero contributions)
#pragma unroll
          for (int q = 0; q < XR; ++q) xr[q][lane] = T(0);
        }
      }
      __syncthreads();
    };
    auto walk = [&](auto staged) {
      uint2 qa = ahead(wave + NP, staged), qb{0u, 0u};
      fetch(wave, ahead(wave, staged), pa);
      for (int r = 0; r <= nround; r += 2) {
        produce(r, pa, pb, qa, qb, staged);
        if (r + 1 <= nround) produce(r + 1, pb, pa, qb, qa, staged);
      }
    };
    if (cnt <= PID_CAP)
      walk(std::true_type{});
    else
      walk(std::false_type{});
    if constexpr (NC > 1) {
      __syncthreads();
    } else {
      zero_tile();
      __syncthreads();
      __syncthreads();
    }
  } else {
    // consumer `pass`: the stencil offsets with last-axis offset pass*KN .. pass*KN+KN-1
    const int pass = wave - NP;
    int ccoord[D];
    {
      int r = lane;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        ccoord[d] = r % G::BW;
        r /= G::BW;
      }
    }
    T am[NSL], amv[D][NSL], af[D][NSL];
#pragma unroll
    for (int o = 0; o < NSL; ++o) {
      am[o] = T(0);
#pragma unroll
      for (int c = 0; c < D; ++c) {
        amv[c][o] = T(0);
        af[c][o] = T(0);
      }
    }
    const T hinv = a.mesh.h_inv;
    uint32_t bad = 0, last = 0;
    for (int r = 0; r <= nround; ++r) {
      if (r > 0) {
        for (int p = 0; p < NP; ++p) {
          const int k = (r - 1) * NP + p;
          if (k >= maxcnt) break;  // uniform
          const T(*xr)[64] = s_x[(r - 1) & 1][p];
          // the jets of the position before the update, as k_p2g_fast evaluates them
          T x[D], l = T(0);
#pragma unroll
          for (int d = 0; d < D; ++d) x[d] = xr[d][lane];
          if constexpr (SH::HAS_L) l = xr[SH::XL][lane];
          T val[D][SW], der[D][SW], vl[KN], dl[KN], mpv[D], A[D * D];
#pragma unroll
          for (int d = 0; d < D; ++d) {
            const T xi = (x[d] - a.mesh.xmin[d]) * hinv;
            int lo, hi;
            axis_window<T, BASIS>(xi, l, a.mesh.dims[d], lo, hi);
            axis_jets_mixed<T, BASIS>(x[d], a.mesh.xmin[d], ccoord[d], hi - lo, s_nodex[d], l, hinv, val[d], der[d]);
          }
#pragma unroll
          for (int q = 0; q < KN; ++q) {
            vl[q] = val[D - 1][pass * KN + q];
            dl[q] = der[D - 1][pass * KN + q];
          }
          const T mpe = xr[XM][lane];
#pragma unroll
          for (int c = 0; c < D; ++c) mpv[c] = xr[XV + c][lane];
#pragma unroll
          for (int b = 0; b < D; ++b)
#pragma unroll
            for (int rr = 0; rr < D; ++rr)
              A[rr + D * b] = xr[XA + (rr >= b ? sym_index(rr, b, D) : sym_index(b, rr, D))][lane];
          p2g_accumulate<T, D, SW, KN>(val, der, vl, dl, mpe, mpv, A, am, amv, af);
          if (misplaced && pass == 0) {
            const bool act = k < ccount;
            uint32_t pid = 0u;
            if (act) pid = cnt <= PID_CAP ? s_pid[coff + k] : a.perm[start + coff + k] - poff;
            bad += broken_pair(__ballot(act), k, pid, last);
          }
        }
      }
      __syncthreads();
    }
    if constexpr (NC > 1) {
      // each consumer zeroes and fills its own slab (the exchange is read out:
      // the rounds ended with a barrier)
      T* const slab = s_xraw + pass * SL::SIZE;
      for (int q = lane; q < int(SL::SIZE * sizeof(T) / 16); q += 64)
        reinterpret_cast<uint4*>(slab)[q] = make_uint4(0u, 0u, 0u, 0u);
      if (ccount > 0) p2g_stencil_to_slab<T, D, SW, KN>(slab, ccoord, pass, am, amv, af);
      __syncthreads();
    } else {
      zero_tile();
      __syncthreads();
      if (ccount > 0) p2g_stencil_to_lds<T, D, SW, KN>(s_tile, ccoord, pass, am, amv, af);
      __syncthreads();
    }
    if (misplaced && pass == 0) {
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) bad += __shfl_xor(bad, off, 64);
      if (lane == 0 && bad) atomicAdd(lane_of(misplaced, LANE_BROKEN), bad);
    }
  }
  if constexpr (NC > 1)
    p2g_write_partial_slabs<T, D, SW, KN, NC, NT>(a, j, s_xraw);
  else
    p2g_write_partial<T, D, SW, NT>(a, j, s_tile);
  if (mo.nk) tile_moves_end(mo, tile, start, cnt, ntiles, &s_mv, moved);
}

template <typename T, int D, int BASIS, bool AOS, int NP, int NC>
__global__ __launch_bounds__(64 * (NP + NC), (G2P2GShape<T, D, BASIS>::wps(NP))) void k_g2p2g_fast(
    Args<T, D> a, const uint32_t* __restrict__ skeys, const MoveOut mo, uint32_t ntiles,
    uint32_t* __restrict__ misplaced) {
  const int64_t j = item_of<false>(blockIdx.x, a.n_active);
  if (j < a.n_active) k_g2p2g_fast_body<T, D, BASIS, AOS, NP, NC>(a, skeys, mo, ntiles, misplaced, j);
}

template <typename T, int D, int SW, bool GAOS, bool BATCH>
__device__ __forceinline__ void k_gather_grid_body(Args<T, D>& a, uint32_t* __restrict__ lanes, const int64_t j) {
  using G = Geo<D>;
  using PT = Part<D, SW>;
  constexpr int NV = 1 + 2 * D;
  constexpr int NB = (D == 3) ? 27 : 9;
  const uint32_t B = a.nb_list[j];
  uint32_t poff;  // a batch's scene: local node block; tiles of the scene start at toff
  const uint32_t Bl = bind_tile<BATCH>(a, B, poff);
  const uint32_t toff = B - Bl;
  int Bi[D], I[D], rr[D];
  unlin<D>(Bl, a.ntiles, Bi);
  // slots of the 3^dim neighbour tiles (-1: no partial)
  __shared__ int s_slot[NB];
  if (threadIdx.x < NB) {
    int r = int(threadIdx.x), t = 0, mul = 1;
    bool ok = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int b = Bi[d] + (r % 3) - 1;
      r /= 3;
      ok = ok && b >= 0 && b < a.ntiles[d];
      t += b * mul;
      mul *= a.ntiles[d];
    }
    s_slot[threadIdx.x] = (ok && a.tile_flag[toff + t]) ? int(a.tile_slot[toff + t]) : -1;
  }
  __syncthreads();
  {
    int r = threadIdx.x;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      rr[d] = r % G::BW;
      r /= G::BW;
      I[d] = Bi[d] * G::BW + rr[d];
      if (I[d] >= a.mesh.dims[d]) return;
    }
  }
  // Tiles covering this node, per axis: B-1 when the node lies in the
  // footprint of the tile below (r < SW-2), B, and B+1 when r == BW-1; at
  // most two per axis.  All their partial values are loaded first, then
  // summed in a fixed order (last axis outermost, ascending tiles).
  int lo[3] = {0, 0, 0}, two[3] = {0, 0, 0};
#pragma unroll
  for (int d = 0; d < D; ++d) {
    lo[d] = rr[d] < SW - 2 ? -1 : 0;
    two[d] = (lo[d] < 0 || rr[d] == G::BW - 1) ? 1 : 0;
  }
  constexpr int NC = 1 << D;
  T pv[NC][NV];
  bool use[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    bool ok = true;
    int nb = 0, q = 0, mulb = 1, mulq = 1;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int k = (c >> d) & 1;
      ok = ok && k <= two[d];
      const int o = lo[d] + k;
      nb += (o + 1) * mulb;
      mulb *= 3;
      q += (rr[d] + 1 - o * G::BW) * mulq;  // node index inside that tile's partial
      mulq *= PT::E;
    }
    const int slot = ok ? s_slot[nb] : -1;
    use[c] = slot >= 0;
    // a skipped candidate reads tile slot 0's first node (a valid address) and is not added
    const T* P = a.partials + (use[c] ? int64_t(slot) * PT::SIZE + int64_t(q) * NV : 0);
#pragma unroll
    for (int v = 0; v < NV; ++v) pv[c][v] = P[v];
  }
  T acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = T(0);
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = use[c] ? acc[v] + pv[c][v] : acc[v];
  const int64_t i = grid_slot(a, I);
  // grid-node half with the guarded Float64 division (test/transfer.jl:102-104)
  const double md = double(acc[0]);
  const bool has = md > 0.0;
  {
    // nodes with m > 0 in this block
    const uint64_t m = __ballot(has);
    if (m && (threadIdx.x & 63) == __ffsll((unsigned long long)__ballot(true)) - 1)
      atomicAdd(lane_of(lanes, LANE_NODES), uint32_t(__popcll(m)));
  }
  const double minv = has ? 1.0 / md : 0.0;
  if (i < 0) return;  // SpGrid node of an inactive block: no storage (and no support, checked by P2G)
  a.gm(i) = acc[0];
  T mvo[D], fo[D], vno[D], vo[D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    const T mvc = acc[1 + c], fc = acc[1 + D + c];
    const T vn = T(double(mvc) * minv);
    const T accel = T(double(fc) * minv) + (has ? a.gravity[c] : T(0));
    T vc = vn + accel * a.dt;
    const bool wall = (((a.slip >> (2 * c)) & 1) && I[c] == 0) ||
                      (((a.slip >> (2 * c + 1)) & 1) && I[c] == a.mesh.dims[c] - 1);
    if (wall) vc = T(0);
    mvo[c] = mvc;
    fo[c] = fc;
    vno[c] = vn;
    vo[c] = vc;
  }
#pragma unroll
  for (int c = 0; c < D; ++c) {
    fldw<T, D, GAOS>(a.gmv, i, c) = mvo[c];
    fldw<T, D, GAOS>(a.gf, i, c) = fo[c];
    fldw<T, D, GAOS>(a.gvn, i, c) = vno[c];
    fldw<T, D, GAOS>(a.gv, i, c) = vo[c];
  }
}

template <typename T, int D, int SW, bool GAOS, bool BATCH = false>
__global__ __launch_bounds__(64) void k_gather_grid(Args<T, D> a, uint32_t* __restrict__ lanes) {
  // the workgroups past the node blocks zero the stale ones
  const int64_t past = int64_t(blockIdx.x) - (((a.n_nb + 7) >> 3) << 3);
  if (past >= 0) {
    if (past < a.n_stale) zero_stale_block<T, D, BATCH>(a, a.stale_list[past]);
    return;
  }
  const int64_t j = item_of<BATCH>(blockIdx.x, a.n_nb);
  if (j < a.n_nb) k_gather_grid_body<T, D, SW, GAOS, BATCH>(a, lanes, j);
}

// Forms whose item count is read on the device at `count` (launch sizes fixed
// in advance): one workgroup per possible item, those past the count ending
// at once (_grid), or a persistent grid sized to the device walking the items
// (_persist; a multiple of 8 workgroups keeps each XCD on a contiguous run of
// them, as xcd_remap does for one workgroup per item).
template <typename T, int D, int SW, bool GAOS, bool BATCH = false>
__global__ __launch_bounds__(64) void k_gather_grid_grid(Args<T, D> a, uint32_t* __restrict__ lanes, const uint32_t* __restrict__ count) {
  const int64_t N = int64_t(*count), R = ((N + 7) >> 3) << 3;
  // xcd_remap is a bijection of [0, R) only: workgroups past R end here
  const int64_t j = item_of<BATCH>(blockIdx.x, N);
  if (int64_t(blockIdx.x) < R && j < N) k_gather_grid_body<T, D, SW, GAOS, BATCH>(a, lanes, j);
}
template <typename T, int D, int SW, bool GAOS, bool BATCH = false>
__global__ __launch_bounds__(64) void k_gather_grid_persist(Args<T, D> a, uint32_t* __restrict__ lanes, const uint32_t* __restrict__ count) {
  const int64_t N = int64_t(*count), R = ((N + 7) >> 3) << 3;
  for (int64_t it = blockIdx.x; it < R; it += gridDim.x) {
    const int64_t j = item_of<BATCH>(it, N);
    if (j < N) k_gather_grid_body<T, D, SW, GAOS, BATCH>(a, lanes, j);
    __syncthreads();  // the next item reuses the workgroup's LDS
  }
}


// ---- G2P -------------------------------------------------------------------

// What the particle equations read of a particle, loaded before the sums: a load
// issued after the first stores would wait for them.
template <typename T, int D>
struct ParticleIn {
  T v[D], x[D], F[D * D];
  __device__ __forceinline__ ParticleIn(const Args<T, D>& a, int64_t p) {
    get_row(a.p_rows, a.v, p, v);
    get_row(a.p_rows, a.x, p, x);
    get_row(a.p_rows, a.F, p, F);
  }
};

// Particle equations of the README @G2P block (README.md:81-86) after the sums.
template <typename T, int D>
__device__ __forceinline__ void particle_update(const Args<T, D>& a, const ParticleIn<T, D>& in, int64_t p, int64_t dst,
                                                const T* dv, const T (&L)[D * D], const T* dx) {
  const T dt = a.dt;
  const bool rows = a.p_rows;
  T vn[D], xn[D], M[D * D], Fn[D * D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    vn[c] = in.v[c] + dv[c];
    xn[c] = in.x[c] + dx[c];
    if (a.x_keep) a.x_keep[dst * D + c] = in.x[c];
  }
  put_row(rows, a.ov, dst, vn);
  put_row(rows, a.ogradv, dst, L);
  put_row(rows, a.ox, dst, xn);
#pragma unroll
  for (int b = 0; b < D; ++b)
#pragma unroll
    for (int r = 0; r < D; ++r) M[r + D * b] = (r == b ? T(1) : T(0)) + L[r + D * b] * dt;
#pragma unroll
  for (int b = 0; b < D; ++b)
#pragma unroll
    for (int r = 0; r < D; ++r) {
      T s = M[r] * in.F[D * b];
#pragma unroll
      for (int k = 1; k < D; ++k) s = s + M[r + D * k] * in.F[k + D * b];
      Fn[r + D * b] = s;
    }
  put_row(rows, a.oF, dst, Fn);
  T sg[D * D], Vn;
  neo_hookean<T, D>(Fn, a.lambda, a.mu, a.V0, a.logE.p != nullptr, a.logE.p ? a.logE(p) : T(0), sg, Vn);
  put_row(rows, a.osigma, dst, sg);
  a.oV(dst) = Vn;
}

// Stored and general corrected weights.  The waves of a tile walk its particles
// in turns of 64, in class or sorted order as k_g2p_fast does; the footprint's
// vⁿ and v are staged in LDS once per tile.  Bound as k_p2g_tile is; on the same
// particles one wave per tile took 83 and 356 us, four take 78 and 130 us, and 52
// and 105 us with everything loaded ahead and in 16-byte words.
constexpr int G2P_TILE_WAVES = 4;  // (8: 51 us instead of 52)

template <typename T, int D, int BASIS, bool STORED, bool CORR = false>
__global__ __launch_bounds__(64 * G2P_TILE_WAVES) void k_g2p_tile(Args<T, D> a, const uint32_t* __restrict__ skeys) {
  using G = Geo<D>;
  constexpr int SW = support_width(BASIS), NW = G2P_TILE_WAVES;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int64_t j = xcd_remap(blockIdx.x, a.n_active);
  if (j >= a.n_active) return;
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  int tI[D], origin[D];
  unlin<D>(tile, a.ntiles, tI);
#pragma unroll
  for (int d = 0; d < D; ++d) origin[d] = tI[d] * G::BW - 1;
  __shared__ T s_vn[D][G::NFOOT];
  __shared__ T s_v[D][G::NFOOT];
  __shared__ T s_nodex[D][G::TS];
  __shared__ uint32_t s_cnt[64];
  for (int q = int(threadIdx.x); q < G::NFOOT; q += 64 * NW) {
    int I[D], r = q;
    bool in = true;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      I[d] = origin[d] + r % G::TS;
      r /= G::TS;
      in = in && I[d] >= 0 && I[d] < a.mesh.dims[d];
    }
    const int64_t i = in ? grid_slot(a, I) : -1;
    in = i >= 0;
#pragma unroll
    for (int c = 0; c < D; ++c) {
      s_vn[c][q] = in ? a.gvn(i, c) : T(0);
      s_v[c][q] = in ? a.gv(i, c) : T(0);
    }
  }
  stage_nodes<T, D>(a.mesh, origin, s_nodex);
  int ccount, coff, maxcnt;
  __shared__ uint32_t s_pid[PID_CAP], s_key[PID_CAP];
  // contains the barrier after staging
  tile_class_counts<NW>(skeys, start, cnt, s_cnt, ccount, coff, maxcnt, a.perm, 0, s_pid, s_key, PID_CAP);
  const int n_sorted = (cnt + 63) / 64;
  const bool by_sorted = 3 * n_sorted < 2 * maxcnt;
  const int kend = by_sorted ? n_sorted : maxcnt;
  const T hinv = a.mesh.h_inv, dt = a.dt;
  for (int k = wave; k < kend; k += NW) {
    const int at = by_sorted ? k * 64 + lane : coff + k;
    if (by_sorted ? at >= cnt : k >= ccount) continue;
    const uint32_t pid = cnt <= PID_CAP ? s_pid[at] : a.perm[start + uint32_t(at)];
    int ccoord[D];  // class coordinates
    {
      uint32_t r = by_sorted ? (cnt <= PID_CAP ? s_key[at] : skeys[start + uint32_t(at)]) & 63u : uint32_t(lane);
#pragma unroll
      for (int d = 0; d < D; ++d) {
        ccoord[d] = int(r % G::BW);
        r /= G::BW;
      }
    }
    T x[D], l;
    int lo[D], hi[D];
    particle_window<T, D, BASIS, STORED>(a, pid, x, l, lo, hi, nullptr);
    const ParticleIn<T, D> in(a, pid);
    int ext[D];
#pragma unroll
    for (int d = 0; d < D; ++d) ext[d] = hi[d] - lo[d];
    T val[D][SW], der[D][SW];
    if constexpr (!STORED) {
#pragma unroll
      for (int d = 0; d < D; ++d) axis_jets<T, D, BASIS>(x[d], ccoord[d], s_nodex[d], l, hinv, val[d], der[d]);
    }
    Corrected<T, D, SW> cs;
    if constexpr (CORR) correct_jets<T, D, BASIS>(a, x, lo, ext, ccoord, s_nodex, cs, val, der);
    T dv[D], L[D * D], dx[D];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      dv[c] = T(0);
      dx[c] = T(0);
    }
#pragma unroll
    for (int q = 0; q < D * D; ++q) L[q] = T(0);
    // column-major walk of the window (eachindex(window)); stored weights are
    // loaded a row at a time
    T sw[STORED ? SW : 1], sg[STORED ? SW : 1][D];
#pragma unroll
    for (int o = 0; o < Pow<SW, D>::v; ++o) {
      if constexpr (STORED) {
        if (o % SW == 0) stored_weights<T, D, Pow<SW, D>::v>(a, pid, o, sw, sg);
      }
      int aa[D], r = o;
      bool ok = true;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        aa[d] = r % SW;
        r /= SW;
        ok = ok && aa[d] <= ext[d];
      }
      if (!ok) continue;
      T w, g[D];
      if constexpr (STORED) {
        w = sw[o % SW];
#pragma unroll
        for (int c = 0; c < D; ++c) g[c] = sg[o % SW][c];
      } else if (CORR && cs.mode == CORR_GENERAL) {
        cs.node(val, aa, filter_pass<D>(a.filter, a.mesh.dims, lo, aa), hinv, w, g);
      } else {
        w = val[0][aa[0]];
#pragma unroll
        for (int d = 1; d < D; ++d) w = w * val[d][aa[d]];
#pragma unroll
        for (int c = 0; c < D; ++c) {
          T gg = (c == 0) ? der[0][aa[0]] : val[0][aa[0]];
#pragma unroll
          for (int d = 1; d < D; ++d) gg = gg * ((d == c) ? der[d][aa[d]] : val[d][aa[d]]);
          g[c] = gg * hinv;
        }
      }
      int q = 0, mul = 1;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        q += (ccoord[d] + aa[d]) * mul;
        mul *= G::TS;
      }
      T vi[D];
#pragma unroll
      for (int c = 0; c < D; ++c) vi[c] = s_v[c][q];
#pragma unroll
      for (int c = 0; c < D; ++c) dv[c] += w * (vi[c] - s_vn[c][q]);
#pragma unroll
      for (int b = 0; b < D; ++b)
#pragma unroll
        for (int r2 = 0; r2 < D; ++r2) L[r2 + D * b] += vi[r2] * g[b];
#pragma unroll
      for (int c = 0; c < D; ++c) dx[c] += (w * vi[c]) * dt;
    }
    particle_update<T, D>(a, in, pid, pid, dv, L, dx);
  }
}

// Particles outside the mesh have an empty window: the sums are zero and only
// the particle equations run (g2p.jl:123-153).
template <typename T, int D, bool BATCH = false>
__global__ __launch_bounds__(256) void k_g2p_outside(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                     uint32_t* __restrict__ nk) {
  const int64_t j = a.n_inside + int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (j >= a.n) return;
  uint32_t pid = a.perm[j];
  if constexpr (BATCH) pid -= uint32_t(bind_scene(a, scene_of(a.scene_poff, a.nscenes, pid)).poff);
  if (nk) nk[j] = skeys[j];  // the position does not change: the key stays
  T dv[D], L[D * D], dx[D];
#pragma unroll
  for (int c = 0; c < D; ++c) {
    dv[c] = T(0);
    dx[c] = T(0);
  }
#pragma unroll
  for (int k = 0; k < D * D; ++k) L[k] = T(0);
  particle_update<T, D>(a, ParticleIn<T, D>(a, pid), pid, a.dest ? a.dest[j] : pid, dv, L, dx);
}

// ---- host side ----------------------------------------------------------------

// True when every particle field is Julia-native AoS (components contiguous,
// element stride = component count), the layout the vectorised kernels assume.
inline bool julia_layout(const tess_particles& P, int D) {
  auto ok = [](const tess_field& f, int nc) { return !f.ptr || (f.comp_stride == 1 && f.elem_stride == nc) ||
                                                      (nc == 1 && f.elem_stride == 1); };
  return ok(P.x, D) && ok(P.v, D) && ok(P.V, 1) && ok(P.grad_v, D * D) && ok(P.F, D * D) && ok(P.sigma, D * D);
}

template <typename T, int D>
Args<T, D> make_args(const tess_mesh& mesh, const tess_grid* G, const tess_particles& P, const tess_weights* W,
                     const tess_params* prm) {
  Args<T, D> a;
  std::memset(static_cast<void*>(&a), 0, sizeof(a));
  a.mesh = dmesh<T, D>(mesh);
  a.x = dfield<T>(P.x);
  a.v = dfield<T>(P.v);
  a.V = dfield<T>(P.V);
  a.gradv = dfield<T>(P.grad_v);
  a.F = dfield<T>(P.F);
  a.sigma = dfield<T>(P.sigma);
  a.l = dfield<T>(P.l);
  a.logE = dfield<T>(P.logE);
  if (G) {
    a.gm = dfield<T>(G->m);
    a.gmv = dfield<T>(G->mv);
    a.gf = dfield<T>(G->f);
    a.gvn = dfield<T>(G->vn);
    a.gv = dfield<T>(G->v);
  }
  if (W) {
    a.window = W->window;
    a.w = dfield<T>(W->w);
    a.gw = dfield<T>(W->grad_w);
    a.w_rows = W->w.elem_stride == 1 && W->grad_w.elem_stride == D && W->grad_w.comp_stride == 1;
  }
  a.p_rows = julia_layout(P, D);
  write_in_place(a);
  a.n = P.n;
  if (prm) {
    a.mp = T(prm->mp);
    a.dt = T(prm->dt);
    a.lambda = prm->lambda;
    a.mu = prm->mu;
    a.V0 = prm->V0;
    for (int d = 0; d < D; ++d) a.gravity[d] = T(prm->gravity[d]);
    a.slip = prm->slip_walls;
  }
  for (int d = 0; d < D; ++d) a.ntiles[d] = int32_t(((mesh.dims[d] - 1) >> Geo<D>::LT) + 1);
  return a;
}

template <typename T, int D>
void set_sparse(Args<T, D>& a, const tess_mesh& mesh, const tess_sparsity* sp) {
  if (!sp) return;
  a.numbering = sp->blocknumbering;
  a.spL = mesh.block_size_log2;
  for (int d = 0; d < D; ++d) a.nblk[d] = int32_t(((mesh.dims[d] - 1) >> mesh.block_size_log2) + 1);
}

template <typename T, int D>
void fill_binning_ptrs(tess_ctx* ctx, Args<T, D>& a) {
  const Binning& b = ctx->bin;
  a.perm = static_cast<const uint32_t*>(ctx->vals.ptr);
  a.tile_start = static_cast<const uint32_t*>(ctx->tile_start.ptr);
  a.tile_end = static_cast<const uint32_t*>(ctx->tile_end.ptr);
  a.active = static_cast<const uint32_t*>(ctx->active_tiles.ptr);
  a.tile_flag = static_cast<const uint32_t*>(ctx->tile_flag.ptr);
  a.tile_slot = static_cast<const uint32_t*>(ctx->tile_slot.ptr);
  a.nb_list = static_cast<const uint32_t*>(ctx->nb_list.ptr);
  a.nb_flag = static_cast<const uint32_t*>(ctx->nb_flag.ptr);
  a.n_inside = b.n_inside;
  a.n_active = b.n_active;
  a.n_nb = b.n_nodeblocks;
}

// The corrected basis and node filter of the current call (deferred weights
// only: stored weights already hold the corrected values).
template <typename T, int D, bool STORED>
void set_correction(tess_ctx* ctx, Args<T, D>& a) {
  a.corr = STORED ? 0 : ctx->corr;
  a.filter = STORED ? nullptr : ctx->corr_filter;
}

inline bool grid_julia_layout(const tess_grid& G, int D) {
  auto ok = [D](const tess_field& f) { return f.comp_stride == 1 && f.elem_stride == D; };
  return ok(G.mv) && ok(G.f) && ok(G.vn) && ok(G.v);
}

inline unsigned blocks_for(int64_t n, int threads) { return unsigned(std::max<int64_t>(1, ceil_div(n, threads))); }

int key_bits_for(uint64_t maxkey) {
  int b = 0;
  while (b < 32 && (uint64_t(1) << b) <= maxkey) ++b;
  return b;
}

// Where a re-binning of n particles sorts every key instead of merging the changed
// ones.  The sort takes some 60 us and 0.12 ns per key.  The merge takes little per
// particle, but one workgroup works on a tile's arrivals at some 25 ns each, and on
// a tile's run (and its leavers) at some 20 ns per particle: the lines lie near
// where such a workgroup alone takes as long as the sort.  P2G on 3D Float32
// particles, always merged and now: 2 M put outside the mesh 53 and 0.32 ms, a tenth
// of them 5.4 and 0.53 ms; 1 M spread from one 2D tile 25 and 0.25 ms; 200 k in eight
// tiles 5.1 and 2.1 ms.
inline uint32_t merge_crowd(int64_t n) { return uint32_t(2048 + n / 256); }     // arrivals of a tile
inline uint32_t merge_tile_max(int64_t n) { return uint32_t(4096 + n / 128); }  // particles of a tile
// arrivals in all: 8 M particles, all in other tiles, 2.55 ms merged and 2.11 ms
// sorted, 2 M 0.59 and 0.55, 0.2 M 0.146 and 0.161
inline uint32_t merge_many(int64_t n) { return uint32_t((512 << 10) + n / 2); }

// The re-binning's buffers for n particles and the context's current tables.
inline MoveOut move_out(tess_ctx* ctx, int64_t n, int64_t ntiles) {
  const size_t m = size_t(std::max<int64_t>(n, 1));
  MoveOut mo;
  mo.nk = ctx->inc_nk.as<uint32_t>(m);
  mo.stay = ctx->tile_stay.as<uint32_t>(size_t(ntiles) + 1);
  mo.tin = ctx->tile_tin.as<uint32_t>(size_t(ntiles) + 1);
  mo.out = ctx->inc_out.as<uint2>(m);
  mo.lanes = lane_counters(ctx);
  return mo;
}
inline MoveOut no_moves() { return MoveOut{nullptr, nullptr, nullptr, nullptr, nullptr}; }

// The node-block list of the last P2G, where it is in the alternate set (the
// stale zeroing may still need it), into a buffer of its own.
inline void save_prev_list(tess_ctx* ctx) {
  if (ctx->prev_list != tess_ctx::PrevList::Alternate || ctx->prev_nodeblocks == 0) return;
  uint32_t* keep = ctx->nb_list_prev.as<uint32_t>(size_t(ctx->prev_nodeblocks));
  TESS_HIP(hipMemcpyAsync(keep, ctx->alt_nb_list.ptr, size_t(ctx->prev_nodeblocks) * sizeof(uint32_t),
                          hipMemcpyDeviceToDevice, ctx->stream));
  ctx->prev_list = tess_ctx::PrevList::Copied;
}

// Arguments that build the tables of ntiles tiles into the alternate set, whose
// buffers grow here where the mesh has more tiles than they hold (and lose what
// they held).
inline TabArgs table_args(tess_ctx* ctx, int64_t ntiles) {
  save_prev_list(ctx);
  TabArgs t;
  std::memset(static_cast<void*>(&t), 0, sizeof(t));
  const size_t nt = size_t(ntiles) + 1;
  t.stay = ctx->tile_stay.as<uint32_t>(nt);
  t.tin = ctx->tile_tin.as<uint32_t>(nt);
  t.ntiles = ntiles;
  t.sums = ctx->tab_sums.as<uint32_t>(size_t(tab_blocks(ntiles)) * 4);
  t.start = ctx->alt_start.as<uint32_t>(nt);
  t.end = ctx->alt_end.as<uint32_t>(nt);
  t.flag = ctx->alt_flag.as<uint32_t>(nt);
  t.slot = ctx->alt_slot.as<uint32_t>(nt);
  t.active = ctx->alt_active.as<uint32_t>(nt);
  t.nb_flag = ctx->alt_nb_flag.as<uint32_t>(nt);
  t.nb_list = ctx->alt_nb_list.as<uint32_t>(nt);
  t.seg = ctx->tile_seg.as<uint32_t>(nt);
  t.lanes = lane_counters(ctx);
  t.counters = ctx->counters.as<uint32_t>(64);
  t.host = reinterpret_cast<uint32_t*>(ctx->counters_host);
  t.crowd = t.many = t.tile_max = UINT32_MAX;
  return t;
}

// Builds the tables of table_args into the alternate set.  Returns the number of
// the report it enqueued.
inline uint32_t build_tables(tess_ctx* ctx, TabArgs& t) {
  if (++ctx->report_seq == 0) ctx->report_seq = 1;
  t.seq = ctx->report_seq;
  launch_tables(ctx->stream, t);
  return t.seq;
}

// The alternate tables become the current ones.
inline void swap_tables(tess_ctx* ctx) {
  if (ctx->prev_list == tess_ctx::PrevList::Current) ctx->prev_list = tess_ctx::PrevList::Alternate;
  std::swap(ctx->tile_start, ctx->alt_start);
  std::swap(ctx->tile_end, ctx->alt_end);
  std::swap(ctx->tile_flag, ctx->alt_flag);
  std::swap(ctx->tile_slot, ctx->alt_slot);
  std::swap(ctx->active_tiles, ctx->alt_active);
  std::swap(ctx->nb_flag, ctx->alt_nb_flag);
  std::swap(ctx->nb_list, ctx->alt_nb_list);
}

// What a report of the lanes says about the last P2G, once.
inline void take_report(tess_ctx* ctx) {
  const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx->counters_host);
  if (ctx->broken_pending) ctx->broken_count = int64_t(hc[CNT_MISPLACED]);
  if (ctx->nodes_pending) ctx->last_active_nodes = int64_t(hc[CNT_NODES]);
  ctx->broken_pending = false;
  ctx->nodes_pending = false;
}

// Waits for report number seq: its words arrive in pinned memory while the
// kernel that writes them still runs, which the end of the stream's work would
// tell 5-10 us later.  The stream is asked now and then, so that a failed launch
// or a report that never comes ends the wait.
inline void wait_report(tess_ctx* ctx, uint32_t seq) {
  const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx->counters_host);
  auto there = [&]() {
    bool all = true;
    for (int r = 0; r < REPORTERS; ++r) all = all && __atomic_load_n(hc + CNT_SEQ + r, __ATOMIC_ACQUIRE) == seq;
    return all;
  };
  for (uint32_t spin = 1; !there(); ++spin) {
    if (spin % 4096 != 0) {
      __builtin_ia32_pause();
      continue;
    }
    const hipError_t e = hipStreamQuery(ctx->stream);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    TESS_HIP(e);
    if (!there()) raise(TESS_ERR_STATE, "the binning's report did not arrive");
  }
}

// The merge of the particles whose key changed, from the current tables to the
// alternate ones (which build_tables has enqueued).
inline MergeArgs merge_args(tess_ctx* ctx, int64_t n, int64_t ntiles, int64_t old_active) {
  const size_t m = size_t(std::max<int64_t>(n, 1));
  MergeArgs g;
  std::memset(static_cast<void*>(&g), 0, sizeof(g));
  g.n = n;
  g.ntiles = ntiles;
  g.old_active = static_cast<const uint32_t*>(ctx->active_tiles.ptr);
  g.old_start = static_cast<const uint32_t*>(ctx->tile_start.ptr);
  g.old_end = static_cast<const uint32_t*>(ctx->tile_end.ptr);
  g.new_active = static_cast<const uint32_t*>(ctx->alt_active.ptr);
  g.new_start = static_cast<const uint32_t*>(ctx->alt_start.ptr);
  g.new_end = static_cast<const uint32_t*>(ctx->alt_end.ptr);
  g.old_active_n = old_active;
  g.stay = static_cast<const uint32_t*>(ctx->tile_stay.ptr);
  g.nk = static_cast<const uint32_t*>(ctx->inc_nk.ptr);
  g.perm_old = static_cast<const uint32_t*>(ctx->vals.ptr);
  g.seg_off = static_cast<const uint32_t*>(ctx->tile_seg.ptr);
  g.out = static_cast<const uint2*>(ctx->inc_out.ptr);
  g.seg = ctx->inc_seg.as<uint2>(m);
  g.seg_alt = ctx->inc_seg2.as<uint2>(m);
  g.keys_new = ctx->skeys2.as<uint32_t>(m);
  g.perm_new = ctx->perm2.as<uint32_t>(m);
  g.crowd = merge_crowd(n);
  g.pos_bits = key_bits_for(uint64_t(m));
  return g;
}

// Launches the merge behind the tables, before the host has their report: its
// launches and the wait overlap.  The counts are the device's, and the launch
// guesses an eighth more active tiles than before; merge_finish adds the rest.
inline MergeArgs merge_ahead(tess_ctx* ctx, int64_t n, int64_t ntiles, int64_t old_active) {
  MergeArgs g = merge_args(ctx, n, ntiles, old_active);
  const uint32_t* counters = static_cast<const uint32_t*>(ctx->counters.ptr);
  g.gate = counters;
  g.new_count = counters + CNT_ACTIVE;
  g.new_active_n = std::min(ntiles, old_active + old_active / 8 + 64);
  launch_merge(ctx->stream, g, 0);
  return g;
}

// After the report of a merge launched ahead: the particles outside the mesh, and
// (keys_sorted, vals) become the new ones.
inline void merge_finish(tess_ctx* ctx, MergeArgs& g, int64_t old_inside) {
  const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx->counters_host);
  g.out_in = hc[CNT_OUTIN];
  g.first_tile = g.new_active_n;
  launch_merge_tiles(ctx->stream, g, int64_t(hc[CNT_ACTIVE]) - g.first_tile);
  if (g.n > int64_t(hc[CNT_INSIDE]))
    launch_merge_outside(ctx->stream, g, unsigned(std::min<int64_t>(blocks_for(g.n - old_inside, 256), 2048)));
  std::swap(ctx->keys_sorted, ctx->skeys2);
  std::swap(ctx->vals, ctx->perm2);
}

// Every next key sorted in the previous order, which is what the merge gives too.
inline void resort_keys(tess_ctx* ctx, int64_t n, int key_bits) {
  radix_sort_pairs(ctx, static_cast<const uint32_t*>(ctx->inc_nk.ptr), static_cast<const uint32_t*>(ctx->vals.ptr),
                   ctx->skeys2.as<uint32_t>(size_t(n)), ctx->perm2.as<uint32_t>(size_t(n)), n, key_bits);
  std::swap(ctx->keys_sorted, ctx->skeys2);
  std::swap(ctx->vals, ctx->perm2);
}

// Debug builds (-DTESS_DEBUG=1, `make debug`): after every binning the host
// reads the binning back and checks its invariants (the permutation, sorted
// keys, each tile's run of keys, the active-tile list), raising
// TESS_ERR_STATE on a violation instead of letting a later kernel index
// through it.
#ifndef TESS_DEBUG
#define TESS_DEBUG 0
#endif
inline void debug_check_binning(hipStream_t st, const uint32_t* skeys, const uint32_t* perm, const uint32_t* tstart,
                                const uint32_t* tend, const uint32_t* active, int64_t n, int64_t ntiles,
                                int64_t n_active, int64_t n_inside, const char* where) {
  if (!TESS_DEBUG) return;
  auto fail = [&](const std::string& what) { raise(TESS_ERR_STATE, std::string("debug check (") + where + "): " + what); };
  TESS_HIP(hipStreamSynchronize(st));
  const size_t nn = size_t(std::max<int64_t>(n, 0)), nt = size_t(std::max<int64_t>(ntiles, 0));
  std::vector<uint32_t> sk(nn), pm(nn), ts(nt), te(nt), act(size_t(std::max<int64_t>(n_active, 0)));
  auto get = [&](std::vector<uint32_t>& v, const uint32_t* src) {
    if (!v.empty()) TESS_HIP(hipMemcpy(v.data(), src, v.size() * sizeof(uint32_t), hipMemcpyDeviceToHost));
  };
  get(sk, skeys);
  get(pm, perm);
  get(ts, tstart);
  get(te, tend);
  get(act, active);
  const uint64_t outside = uint64_t(ntiles) * 64u;
  std::vector<uint8_t> seen(sk.size(), 0);
  int64_t inside = 0;
  for (int64_t j = 0; j < n; ++j) {
    if (pm[size_t(j)] >= uint64_t(n) || seen[pm[size_t(j)]]) fail("the permutation repeats or leaves [0, n)");
    seen[pm[size_t(j)]] = 1;
    if (sk[size_t(j)] > outside) fail("a sort key past the tiles");
    if (j > 0 && sk[size_t(j)] < sk[size_t(j - 1)]) fail("sort keys out of order at " + std::to_string(j));
    inside += sk[size_t(j)] < outside ? 1 : 0;
  }
  if (n_inside >= 0 && inside != n_inside) fail("inside count " + std::to_string(n_inside) + " != " + std::to_string(inside));
  int64_t nact = 0, j = 0;
  for (int64_t t = 0; t < ntiles; ++t) {
    const int64_t a = j;
    while (j < inside && int64_t(sk[size_t(j)] >> 6) == t) ++j;
    if (j > a) {
      if (ts[size_t(t)] != uint64_t(a) || te[size_t(t)] != uint64_t(j)) fail("tile run of " + std::to_string(t));
      if (nact >= n_active || act[size_t(nact)] != uint64_t(t)) fail("active-tile list at " + std::to_string(nact));
      ++nact;
    } else if (te[size_t(t)] > ts[size_t(t)]) {
      fail("a particle run for the empty tile " + std::to_string(t));
    }
  }
  if (nact != n_active) fail("active tiles " + std::to_string(n_active) + " != " + std::to_string(nact));
}

template <typename T, int D, int BASIS, bool STORED>
void bin_particles_run(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P, const tess_weights* W,
                       bool keys_from_g2p);

template <typename T, int D, int BASIS, bool STORED>
void bin_particles(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P, const tess_weights* W,
                   bool keys_from_g2p = false) {
  bin_particles_run<T, D, BASIS, STORED>(ctx, mesh, P, W, keys_from_g2p);
  if (TESS_DEBUG && P.n > 0) {
    const Binning& b = ctx->bin;
    debug_check_binning(ctx->stream, static_cast<const uint32_t*>(ctx->keys_sorted.ptr),
                        static_cast<const uint32_t*>(ctx->vals.ptr), static_cast<const uint32_t*>(ctx->tile_start.ptr),
                        static_cast<const uint32_t*>(ctx->tile_end.ptr),
                        static_cast<const uint32_t*>(ctx->active_tiles.ptr), P.n, b.ntiles, b.n_active, b.n_inside,
                        "bin_particles");
  }
}

template <typename T, int D, int BASIS, bool STORED>
void bin_particles_run(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P, const tess_weights* W,
                       bool keys_from_g2p) {
  Args<T, D> a = make_args<T, D>(mesh, nullptr, P, W, nullptr);
  const int64_t n = P.n;
  uint64_t ntiles = 1;
  for (int d = 0; d < D; ++d) ntiles *= uint64_t(a.ntiles[d]);
  if (ntiles * 64 >= uint64_t(UINT32_MAX) || n >= int64_t(UINT32_MAX))
    raise(TESS_ERR_ARGUMENT, "mesh or particle count exceeds the 32-bit binning range");
  Binning& b = ctx->bin;
  b.valid = false;
  const size_t m = size_t(std::max<int64_t>(n, 1));
  uint32_t* counters = ctx->counters.as<uint32_t>(64);
  const int tok = prof_begin(ctx, "binning", 0.0);
  const int kbits = key_bits_for(ntiles * 64);
  const bool incremental = b.state_valid && b.state_n == n && b.state_ntiles == int64_t(ntiles) &&
                           b.state_dim == D && n > 0;
  const bool precomputed = keys_from_g2p && b.keys_ready && b.x_ptr == P.x.ptr && b.tile_log2 == Geo<D>::LT &&
                           b.basis == BASIS && b.dtype == mesh.dtype;
  b.keys_ready = false;
  TabArgs tab = table_args(ctx, int64_t(ntiles));
  for (int d = 0; d < 3; ++d) tab.nt[d] = d < D ? a.ntiles[d] : 1;
  tab.tile_max = merge_tile_max(n);
  const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx->counters_host);
  uint32_t err = 0;
  if (incremental) {
    // keys in the previous sorted order, from the previous G2P of the same step
    // loop or from the positions; the tables they give; one readback
    const MoveOut mo = move_out(ctx, n, int64_t(ntiles));
    const bool flat = !precomputed && b.crowded;
    if (!precomputed) {
      fill_binning_ptrs<T, D>(ctx, a);
      const uint32_t* skeys = static_cast<const uint32_t*>(ctx->keys_sorted.ptr);
      if (flat) {
        hipLaunchKernelGGL((k_rekey_flat<T, D, BASIS, STORED>), dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, a,
                           skeys, uint32_t(ntiles), mo, counters);
        TESS_HIP(hipGetLastError());
      }
      if (!flat && b.n_active > 0) {
        hipLaunchKernelGGL((k_rekey<T, D, BASIS, STORED>), dim3(xcd_grid(b.n_active)), dim3(256), 0, ctx->stream, a,
                           skeys, uint32_t(ntiles), mo, counters);
        TESS_HIP(hipGetLastError());
      }
      if (!flat && n > b.n_inside) {
        hipLaunchKernelGGL((k_rekey_outside<T, D, BASIS, STORED>), dim3(blocks_for(n - b.n_inside, 256)), dim3(256),
                           0, ctx->stream, a, uint32_t(ntiles), mo, counters);
        TESS_HIP(hipGetLastError());
      }
    }
    // (meshes of as many tiles with other axes give equal keys, not equal node blocks)
    bool same_kind = b.tile_log2 == Geo<D>::LT && b.basis == BASIS && b.dtype == mesh.dtype;
    for (int d = 0; d < D; ++d) same_kind = same_kind && b.ntiles_axis[d] == a.ntiles[d];
    tab.may_keep = same_kind ? 1 : 0;
    tab.crowd = merge_crowd(n);
    tab.many = merge_many(n);
    const uint32_t seq = build_tables(ctx, tab);
    // (over many tiles, whose workgroups cost 0.2 ns each to find nothing to do,
    // not ahead while the last binning found no changed key)
    const bool ahead = !b.crowded && (ctx->last_movers != 0 || b.n_active <= 8192);
    MergeArgs merge;
    if (ahead) merge = merge_ahead(ctx, n, int64_t(ntiles), b.n_active);
    wait_report(ctx, seq);
    take_report(ctx);
    ctx->last_movers = int64_t(hc[CNT_MOVED]);
    err = hc[CNT_ERR];
    const bool recount = flat || (hc[CNT_RESORT] & RESORT_RECOUNT);
    const bool resort = ctx->last_movers > 0 && (recount || b.crowded || hc[CNT_RESORT] || hc[CNT_ARRIVE] > tab.many);
    if (!ahead && ctx->last_movers > 0 && !resort) merge = merge_ahead(ctx, n, int64_t(ntiles), b.n_active);
    if (ctx->last_movers == 0 && same_kind && !(err & ERR_GIMP_LENGTH)) {
      // no particle changed its key: the previous order and tile lists stand
      ctx->last_misplaced = (ctx->misplaced_x_ptr == P.x.ptr && ctx->misplaced_n == n) ? ctx->broken_count : -1;
      ctx->kept_binnings += 1;
      b.x_ptr = P.x.ptr;
      b.valid = true;
      prof_end(ctx, tok);
      return;
    }
    if (resort) {
      resort_keys(ctx, n, kbits);
    } else if (ctx->last_movers > 0) {
      merge_finish(ctx, merge, b.n_inside);
    }
    if (recount) {
      // (the tables above had no counts of these keys; the ones of this report stand)
      tab.may_keep = 0;
      launch_tile_counts(ctx->stream, static_cast<const uint32_t*>(ctx->keys_sorted.ptr), n, int64_t(ntiles), tab.stay,
                         tab.tin);
      wait_report(ctx, build_tables(ctx, tab));
    }
  } else {
    uint32_t* skeys = ctx->keys_sorted.as<uint32_t>(m);
    uint32_t* perm = ctx->vals.as<uint32_t>(m);
    if (n > 0) {
      uint32_t* keys = ctx->keys.as<uint32_t>(m);
      hipLaunchKernelGGL((k_bin_keys<T, D, BASIS, STORED>), dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, a,
                         keys, uint32_t(ntiles), counters);
      TESS_HIP(hipGetLastError());
      radix_sort_pairs(ctx, keys, nullptr, skeys, perm, n, kbits);
    }
    ctx->last_movers = -1;
    launch_tile_counts(ctx->stream, skeys, n, int64_t(ntiles), tab.stay, tab.tin);
    wait_report(ctx, build_tables(ctx, tab));
    take_report(ctx);
    err = hc[CNT_ERR];
  }
  prof_end(ctx, tok);
  if (err & ERR_GIMP_LENGTH) raise(TESS_ERR_ARGUMENT, "uGIMP requires 0 ≤ pt.l ≤ spacing(mesh)");
  if (err & ERR_WINDOW)
    raise(TESS_ERR_DIMENSION, "stored support window is larger than the basis support width");
  swap_tables(ctx);
  b.n_inside = int64_t(hc[CNT_INSIDE]);
  // layout score of the previous P2G on this particle set (consumed by the step driver)
  ctx->last_misplaced = (ctx->misplaced_x_ptr == P.x.ptr && ctx->misplaced_n == n) ? ctx->broken_count : -1;
  b.n_active = int64_t(hc[CNT_ACTIVE]);
  b.n_nodeblocks = int64_t(hc[CNT_NB]);
  b.crowded = (hc[CNT_RESORT] & RESORT_TILE) != 0;
  b.x_ptr = P.x.ptr;
  b.n = n;
  b.dim = D;
  b.dtype = mesh.dtype;
  b.basis = BASIS;
  b.tile_log2 = Geo<D>::LT;
  b.ntiles = int64_t(ntiles);
  for (int d = 0; d < 3; ++d) b.ntiles_axis[d] = d < D ? a.ntiles[d] : 1;
  b.valid = true;
  b.state_valid = n > 0;
  b.state_n = n;
  b.state_ntiles = int64_t(ntiles);
  b.state_dim = D;
}

// P2G after binning: zeroing of what this call does not overwrite, the tile
// kernel and the gather.  count_misplaced asks the tile kernel to count
// particles not stored in the layered order (for the step driver's reorder).
// With `sweep`, the tile partials come from sweep(a, sorted keys, misplaced)
// in place of the P2G kernel (the single-sweep @G2P2G kernel, which reads the
// grid's v and vⁿ: the grid is zeroed after it).
template <typename T, int D>
using SweepFn = std::function<void(Args<T, D>&, const uint32_t*, uint32_t*)>;

template <typename T, int D, int BASIS, bool STORED>
void p2g_launch(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                const tess_weights* W, const tess_params& prm, bool count_misplaced, const tess_sparsity* sp,
                const SweepFn<T, D>* sweep = nullptr, bool fresh_numbering = false) {
  using Gm = Geo<D>;
  constexpr int NV = 1 + 2 * D;
  constexpr int SW = support_width(BASIS);
  // all sw^dim offsets in one pass while the accumulators fit ~200 VGPRs,
  // else one pass per offset along the last axis
  constexpr int NPASS = (Pow<SW, D>::v * NV * int(sizeof(T)) / 4 <= 100) ? 1 : SW;
  Args<T, D> a = make_args<T, D>(mesh, &G, P, W, &prm);
  fill_binning_ptrs<T, D>(ctx, a);
  set_sparse<T, D>(a, mesh, sp);
  set_correction<T, D, STORED>(ctx, a);
  uint32_t* counters = static_cast<uint32_t*>(ctx->counters.ptr);
  int64_t nnodes = 1;
  for (int d = 0; d < D; ++d) nnodes *= mesh.dims[d];
  // zero what this call will not overwrite: everything on first use of a
  // grid, else the node blocks that were written last time and are not now.
  // An SpGrid's storage is zeroed whole (its numbering may have changed).
  bool fresh = ctx->last_grid_m != G.m.ptr || ctx->prev_tile_log2 != Gm::LT;
  for (int d = 0; d < D; ++d) fresh = fresh || ctx->prev_dims[d] != mesh.dims[d];
  // The numbering was built from these particles (fresh_numbering): with blocks
  // of at least two nodes every class window lies within the activated blocks,
  // and there is nothing to check.
  const bool check = sp && !(fresh_numbering && mesh.block_size_log2 >= 1 && !TESS_DEBUG);
  if (check) {
    a.p2g_err = counters + CNT_P2GERR;
    TESS_HIP(hipMemsetAsync(a.p2g_err, 0, sizeof(uint32_t), ctx->stream));
  }
  auto zero_grid = [&]() {
    if (sp) {
      if (sp->storage_len > 0) {
        hipLaunchKernelGGL((k_zero_grid<T, D>), dim3(blocks_for(sp->storage_len, 256)), dim3(256), 0, ctx->stream,
                           a, sp->storage_len);
        TESS_HIP(hipGetLastError());
      }
    } else if (fresh) {
      hipLaunchKernelGGL((k_zero_grid<T, D>), dim3(blocks_for(nnodes, 256)), dim3(256), 0, ctx->stream, a, nnodes);
      TESS_HIP(hipGetLastError());
    }
  };
  // stale node blocks are zeroed by the gather's launch; there are none while
  // the tables are still those of the last P2G (no binning since has swapped them)
  const bool stale = !sp && !fresh && ctx->prev_nodeblocks > 0 && ctx->prev_list != tess_ctx::PrevList::Current;
  if (stale) {
    a.stale_list = static_cast<const uint32_t*>(ctx->prev_list == tess_ctx::PrevList::Alternate ? ctx->alt_nb_list.ptr
                                                                                                : ctx->nb_list_prev.ptr);
    a.n_stale = ctx->prev_nodeblocks;
  }
  if (!sweep) zero_grid();
  const Binning& b = ctx->bin;
  // broken pairs and nodes with mass are counted into the lanes, which the next
  // binning's report sums and resets; a count nothing has reported yet (another
  // P2G, on the same binning) starts over
  uint32_t* lanes = lane_counters(ctx);
  uint32_t* misplaced = nullptr;
  if (ctx->broken_pending || ctx->nodes_pending) {
    TESS_HIP(hipMemsetAsync(lanes + LANE_BROKEN * LANES * LANE_STRIDE, 0, size_t(2) * LANES * LANE_STRIDE * 4, ctx->stream));
    ctx->broken_pending = ctx->nodes_pending = false;
  }
  ctx->nodes_pending = true;
  if (count_misplaced) {
    misplaced = lanes;
    ctx->broken_pending = true;
    ctx->misplaced_x_ptr = P.x.ptr;
    ctx->misplaced_n = P.n;
    ctx->misplaced_pairs = b.n_inside - b.n_active;
  } else {
    ctx->misplaced_x_ptr = nullptr;
  }
  if (b.n_active > 0 && sweep) {
    a.partials = ctx->partials.as<T>(size_t(b.n_active) * Part<D, SW>::SIZE);
    (*sweep)(a, static_cast<const uint32_t*>(ctx->keys_sorted.ptr), misplaced);
  } else if (b.n_active > 0) {
    a.partials = ctx->partials.as<T>(size_t(b.n_active) * Part<D, SW>::SIZE);
    // algorithmic bytes: x, v, V, σ per particle
    const int tok = prof_begin(ctx, "k_p2g_tile", double(b.n_inside) * sizeof(T) * (2 * D + 1 + D * D));
    const uint32_t* sk = static_cast<const uint32_t*>(ctx->keys_sorted.ptr);
    const dim3 tile_block(64 * NPASS * P2G_TILE_SPLIT<D, NPASS>);
    if constexpr (STORED) {
      hipLaunchKernelGGL((k_p2g_tile<T, D, BASIS, STORED, NPASS>), dim3(xcd_grid(b.n_active)), tile_block, 0,
                         ctx->stream, a, sk, misplaced);
    } else if (a.corr && !separable_correction(a.corr, BASIS, a.filter != nullptr)) {
      bool solo = false;
      if constexpr (P2G_TILE_SOLO<T, D, NPASS>) {
        if (b.n_active >= P2G_SOLO_TILES) {
          constexpr int WP = D == 2 ? NPASS : 1;
          hipLaunchKernelGGL((k_p2g_tile<T, D, BASIS, false, NPASS, true, WP, 1>), dim3(xcd_grid(b.n_active)),
                             dim3(64 * WP), 0, ctx->stream, a, sk, misplaced);
          solo = true;
        }
      }
      if (!solo)
        hipLaunchKernelGGL((k_p2g_tile<T, D, BASIS, false, NPASS, true>), dim3(xcd_grid(b.n_active)), tile_block, 0,
                           ctx->stream, a, sk, misplaced);
    } else {
      // 3D: one wave per offset along z; 2D: one wave while the stencil fits
      constexpr int NPF = (D == 3 || Pow<SW, D>::v * NV * int(sizeof(T)) / 4 > 96) ? SW : 1;
      const bool aos = julia_layout(P, D);
      bool done = false;
      if constexpr (BASIS == TESS_BSPLINE_QUADRATIC || BASIS == TESS_BSPLINE_CUBIC) {
        if (a.corr) {  // separable corrected basis: the same kernel with corrected axis jets
          if (aos)
            hipLaunchKernelGGL((k_p2g_fast<T, D, BASIS, NPF, true, false, true>), dim3(xcd_grid(b.n_active)),
                               dim3(64 * NPF), 0, ctx->stream, a, sk, misplaced);
          else
            hipLaunchKernelGGL((k_p2g_fast<T, D, BASIS, NPF, false, false, true>), dim3(xcd_grid(b.n_active)),
                               dim3(64 * NPF), 0, ctx->stream, a, sk, misplaced);
          done = true;
        }
      }
      if (!done) {
        if (aos)
          hipLaunchKernelGGL((k_p2g_fast<T, D, BASIS, NPF, true>), dim3(xcd_grid(b.n_active)), dim3(64 * NPF), 0,
                             ctx->stream, a, sk, misplaced);
        else
          hipLaunchKernelGGL((k_p2g_fast<T, D, BASIS, NPF, false>), dim3(xcd_grid(b.n_active)), dim3(64 * NPF), 0,
                             ctx->stream, a, sk, misplaced);
      }
    }
    TESS_HIP(hipGetLastError());
    prof_end(ctx, tok);
  }
  if (sweep) zero_grid();
  if (b.n_nodeblocks > 0 || a.n_stale > 0) {
    // algorithmic bytes per active node: m, mv, f written, read back by the
    // grid-node half, vⁿ and v written (the node count of the previous call)
    const double nodes = double(std::max<int64_t>(ctx->last_active_nodes, 0));
    const int tok = prof_begin(ctx, "k_gather_grid", nodes * sizeof(T) * (2 * (2 * D + 1) + 2 * D));
    const dim3 grid(xcd_grid(b.n_nodeblocks) + unsigned(a.n_stale));
    if (grid_julia_layout(G, D))
      hipLaunchKernelGGL((k_gather_grid<T, D, SW, true>), grid, dim3(64), 0, ctx->stream, a, lanes);
    else
      hipLaunchKernelGGL((k_gather_grid<T, D, SW, false>), grid, dim3(64), 0, ctx->stream, a, lanes);
    TESS_HIP(hipGetLastError());
    prof_end(ctx, tok);
  }
  // this call's node blocks are what the next call's stale zeroing looks at
  ctx->prev_nodeblocks = b.n_nodeblocks;
  ctx->prev_list = tess_ctx::PrevList::Current;
  ctx->last_grid_m = sp ? nullptr : G.m.ptr;  // a dense grid after an SpGrid call starts from a full zero
  ctx->prev_tile_log2 = Gm::LT;
  for (int d = 0; d < D; ++d) ctx->prev_dims[d] = mesh.dims[d];
  if (check) {
    uint32_t* hc = reinterpret_cast<uint32_t*>(ctx->counters_host);
    TESS_HIP(hipMemcpyAsync(hc + CNT_P2GERR, counters + CNT_P2GERR, sizeof(uint32_t), hipMemcpyDeviceToHost,
                            ctx->stream));
    TESS_HIP(hipStreamSynchronize(ctx->stream));
    if (hc[CNT_P2GERR] & ERR_INACTIVE)
      raise(TESS_ERR_STATE, "@P2G: inactive SpGrid support node. Call update_sparsity! before @P2G.");
  }
}

// fraction of layered neighbour pairs (particles inside the mesh minus active
// tiles) that are consecutive in storage; 1 with no pairs
inline double layered_contiguity(int64_t broken, int64_t pairs) {
  return pairs > 0 ? 1.0 - double(broken) / double(pairs) : 1.0;
}

template <typename T, int D, int BASIS, bool STORED>
void g2p_launch(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                const tess_weights* W, const tess_params& prm, const tess_sparsity* sp, bool write_keys = false,
                T* x_keep = nullptr, const tess_particles* out = nullptr, const uint32_t* dest = nullptr) {
  const Binning& b = ctx->bin;
  Args<T, D> a = make_args<T, D>(mesh, &G, P, W, &prm);
  a.x_keep = x_keep;
  if (out) {
    a.ox = dfield<T>(out->x);
    a.ov = dfield<T>(out->v);
    a.oV = dfield<T>(out->V);
    a.ogradv = dfield<T>(out->grad_v);
    a.oF = dfield<T>(out->F);
    a.osigma = dfield<T>(out->sigma);
    a.dest = dest;
    a.p_rows = a.p_rows && julia_layout(*out, D);
  }
  fill_binning_ptrs<T, D>(ctx, a);
  set_sparse<T, D>(a, mesh, sp);
  set_correction<T, D, STORED>(ctx, a);
  // next-step keys at the sorted positions (deferred weights in the fast kernel)
  const bool generic = a.corr && !separable_correction(a.corr, BASIS, a.filter != nullptr);
  const MoveOut mo = write_keys && !STORED && !generic && P.n > 0 ? move_out(ctx, P.n, b.ntiles) : no_moves();
  const uint32_t* skeys_now = static_cast<const uint32_t*>(ctx->keys_sorted.ptr);
  // (rows are addressed by 32-bit scalar offsets; past them the kernel for any strides)
  const bool aos = julia_layout(P, D) && (D == 2 || sizeof(T) == 4 || P.n < int64_t(UINT32_MAX) / (D * D));
  // the particles are written in the layered order: this step puts them there,
  // or the last P2G that counted found nearly every neighbour pair in place
  const bool layered = dest || (ctx->last_misplaced >= 0 && ctx->misplaced_x_ptr == P.x.ptr &&
                                layered_contiguity(ctx->last_misplaced, ctx->misplaced_pairs) >= 0.98);
  if (b.n_active > 0) {
    // algorithmic bytes: x, v, F read and v, ∇v, x, F, σ, V written per
    // particle; vⁿ, v read per active node
    const double nodes = double(std::max<int64_t>(ctx->last_active_nodes, 0));
    const int per_p = 2 * D + D * D + 2 * D + 3 * D * D + 1;
    const int tok = prof_begin(ctx, "k_g2p_tile",
                               double(b.n_inside) * sizeof(T) * per_p + nodes * sizeof(T) * 2 * D);
    const uint32_t* sk = static_cast<const uint32_t*>(ctx->keys_sorted.ptr);
    if constexpr (STORED) {
      hipLaunchKernelGGL((k_g2p_tile<T, D, BASIS, STORED>), dim3(xcd_grid(b.n_active)), dim3(64 * G2P_TILE_WAVES), 0,
                         ctx->stream, a, sk);
    } else if (generic) {
      hipLaunchKernelGGL((k_g2p_tile<T, D, BASIS, false, true>), dim3(xcd_grid(b.n_active)), dim3(64 * G2P_TILE_WAVES),
                         0, ctx->stream, a, sk);
    } else {
      constexpr int NW = TESS_G2P_WAVES_PER_TILE;
      const dim3 grid(xcd_grid(b.n_active)), block(64 * NW);
      const uint32_t nt = uint32_t(b.ntiles);
      auto launch = [&](auto sep, auto stream) {
        constexpr bool SEP = decltype(sep)::value, NT = decltype(stream)::value;
        if (aos)
          hipLaunchKernelGGL((k_g2p_fast<T, D, BASIS, true, NW, false, SEP, NT>), grid, block, 0, ctx->stream, a, sk,
                             mo, nt);
        else
          hipLaunchKernelGGL((k_g2p_fast<T, D, BASIS, false, NW, false, SEP>), grid, block, 0, ctx->stream, a, sk, mo,
                             nt);
      };
      auto pick = [&](auto sep) {
        if constexpr (sizeof(T) == 4) {  // (Float64 rows fill lines by themselves: 260 us NT, 252 us plain on the rod)
          if (layered) return launch(sep, std::true_type{});
        }
        launch(sep, std::false_type{});
      };
      bool done = false;
      if constexpr (BASIS == TESS_BSPLINE_QUADRATIC || BASIS == TESS_BSPLINE_CUBIC) {
        if (a.corr) {  // separable corrected basis
          pick(std::true_type{});
          done = true;
        }
      }
      if (!done) pick(std::false_type{});
    }
    TESS_HIP(hipGetLastError());
    prof_end(ctx, tok);
  }
  if (P.n > b.n_inside) {
    hipLaunchKernelGGL((k_g2p_outside<T, D>), dim3(blocks_for(P.n - b.n_inside, 256)), dim3(256), 0, ctx->stream,
                       a, skeys_now, mo.nk);
    TESS_HIP(hipGetLastError());
  }
  ctx->bin.valid = false;  // positions moved
  ctx->bin.keys_ready = mo.nk != nullptr;
}

// Layered storage order of the binned particles: inside each tile the k-th
// particle of every class, classes ascending, then the next k.  Writes the
// gather order (new storage slot -> old particle) and the sorted-slot -> new
// storage index map.
template <typename T, int D>
__global__ __launch_bounds__(64) void k_layered_order(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                       uint32_t* __restrict__ order, uint32_t* __restrict__ perm_new,
                                                       uint32_t* __restrict__ broken = nullptr) {
  const int lane = threadIdx.x;
  const int64_t j = blockIdx.x;
  if (j >= a.n_active) return;
  const uint32_t tile = a.active[j];
  const uint32_t start = a.tile_start[tile];
  const int cnt = int(a.tile_end[tile] - start);
  __shared__ uint32_t s_cnt[64];
  int ccount, coff, maxcnt;
  tile_class_counts(skeys, start, cnt, s_cnt, ccount, coff, maxcnt);
  uint32_t layer_off = 0, bad = 0, last = 0;
  for (int k = 0; k < maxcnt; ++k) {
    const uint64_t has = __ballot(k < ccount);
    const uint32_t pid = k < ccount ? a.perm[start + coff + k] : 0u;
    if (k < ccount) {
      const uint32_t dest = start + layer_off + uint32_t(__popcll(has & lanemask_lt64()));
      order[dest] = pid;
      perm_new[start + coff + k] = dest;
    }
    if (broken) bad += broken_pair(has, k, pid, last);
    layer_off += uint32_t(__popcll(has));
  }
  if (broken) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) bad += __shfl_xor(bad, off, 64);
    if (lane == 0) broken[j] = bad;
  }
}

__global__ void k_tail_identity(const uint32_t* __restrict__ perm, int64_t from, int64_t n,
                                uint32_t* __restrict__ order, uint32_t* __restrict__ perm_new) {
  const int64_t j = from + int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (j >= n) return;
  order[j] = perm[j];
  perm_new[j] = uint32_t(j);
}

// The layered order of the current binning: order[new index] = particle (in
// ctx->keys) and the new index of the particle at each sorted position (in
// ctx->keys_alt, returned).
template <typename T, int D>
uint32_t* layered_maps(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P) {
  const Binning& b = ctx->bin;
  const int64_t n = P.n;
  Args<T, D> a = make_args<T, D>(mesh, nullptr, P, nullptr, nullptr);
  fill_binning_ptrs<T, D>(ctx, a);
  uint32_t* order = ctx->keys.as<uint32_t>(size_t(n));        // raw keys are dead after the sort
  uint32_t* perm_new = ctx->keys_alt.as<uint32_t>(size_t(n));
  if (b.n_active > 0) {
    hipLaunchKernelGGL((k_layered_order<T, D>), dim3(unsigned(b.n_active)), dim3(64), 0, ctx->stream, a,
                       static_cast<const uint32_t*>(ctx->keys_sorted.ptr), order, perm_new);
    TESS_HIP(hipGetLastError());
  }
  if (n > b.n_inside) {
    hipLaunchKernelGGL(k_tail_identity, dim3(blocks_for(n - b.n_inside, 256)), dim3(256), 0, ctx->stream,
                       static_cast<const uint32_t*>(ctx->vals.ptr), b.n_inside, n, order, perm_new);
    TESS_HIP(hipGetLastError());
  }
  return perm_new;
}

// Moves the particles into the layered order where they are stored.
template <typename T, int D>
void layered_reorder(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P) {
  if (P.n == 0) return;
  layered_maps<T, D>(ctx, mesh, P);
  permute_particles(ctx, mesh, P, static_cast<const uint32_t*>(ctx->keys.ptr));
  std::swap(ctx->vals, ctx->keys_alt);
}

// ---- reorders that ride on G2P -------------------------------------------------
//
// G2P rewrites every particle field but l and log E, so a step that reorders
// lets it write the particles at their layered places into a second set of
// arrays instead of moving them before the step: nothing is read or written
// twice.  P2G and the gather half of that step read the particles where they
// were, in the same order, so every sum is the same.  The loop then goes on
// with the second set; a call's last step writes the caller's arrays again (in
// place of the second set, at no cost), and only a reorder in that last step,
// or an error, leaves a copy to make.
//
// Moving the 34 scalars of a particle before the step took a gather and a
// write-back pass: 3.3 ms for 13.4 M particles (Float32), beside 1.5 ms for the
// step.  What is left is the pair of maps (0.1 ms) and the copy of at most one
// reorder per call (0.6 ms).  The second set (34 scalars per particle in 3D, and an
// eighth) stays with the context; where the device has no memory for it the loop
// moves the particles before the step, through one field's scratch.
class MovingParticles {
 public:
  // allowed: the step's G2P is the one that can write elsewhere
  MovingParticles(tess_ctx* ctx, const tess_particles& P, int D, size_t scalar, bool allowed)
      : ctx_(ctx), home_(P), cur_(P), D_(D), scalar_(scalar), can_(allowed && P.n > 0) {
    for (int f = 0; f < 6; ++f) {
      const tess_field& a = field(home_, f);
      const int nc = comps(f);
      const bool aos = a.elem_stride == nc && (nc == 1 || a.comp_stride == 1);
      const bool soa = a.elem_stride == 1 && a.comp_stride == P.n;
      can_ = can_ && a.ptr && (aos || soa);
    }
  }
  // asked before a reordering step's work is enqueued: whether there is, or can
  // be, a second set (without it the particles are moved where they are stored)
  bool can_move() {
    if (can_ && home()) can_ = ctx_->moved.fits(bytes());
    return can_;
  }
  const tess_particles& now() const { return cur_; }
  bool home() const { return cur_.x.ptr == home_.x.ptr; }
  // the set the particles are not in (same layout)
  tess_particles other() {
    if (!home()) return home_;
    tess_particles q = home_;
    char* p = static_cast<char*>(ctx_->moved.get(bytes()));
    for (int f = 0; f < 6; ++f) {
      const_cast<tess_field&>(field(q, f)).ptr = p;
      p += span(f);
    }
    return q;
  }
  // the particles have been written to `to`
  void moved_to(const tess_particles& to) {
    if (to.x.ptr == cur_.x.ptr) return;
    rename(cur_.x.ptr, to.x.ptr);
    cur_ = to;
  }
  // back into the caller's arrays
  void settle() {
    if (home()) return;
    const void* src[6];
    void* dst[6];
    int64_t bytes[6];
    for (int f = 0; f < 6; ++f) {
      src[f] = field(cur_, f).ptr;
      dst[f] = field(home_, f).ptr;
      bytes[f] = home_.n * comps(f) * int64_t(scalar_);
    }
    rename(cur_.x.ptr, home_.x.ptr);
    cur_ = home_;
    copy_arrays(ctx_->stream, src, dst, bytes, 6);
  }

 private:
  static const tess_field& field(const tess_particles& P, int f) {
    const tess_field* t[6] = {&P.x, &P.v, &P.V, &P.grad_v, &P.F, &P.sigma};
    return *t[f];
  }
  int comps(int f) const { return f < 2 ? D_ : f == 2 ? 1 : D_ * D_; }
  size_t span(int f) const { return (size_t(home_.n) * size_t(comps(f)) * scalar_ + 255) & ~size_t(255); }
  size_t bytes() const {
    size_t b = 0;
    for (int f = 0; f < 6; ++f) b += span(f);
    return b;
  }
  void rename(const void* from, const void* to) {
    if (ctx_->bin.x_ptr == from) ctx_->bin.x_ptr = to;
    if (ctx_->misplaced_x_ptr == from) ctx_->misplaced_x_ptr = to;
  }
  tess_ctx* ctx_;
  tess_particles home_, cur_;
  int D_;
  size_t scalar_;
  bool can_;
};

// After a G2P that wrote the particles at their layered places: the binning's
// permutation, and the fields G2P does not write.
template <typename T, int D>
void take_layered(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P) {
  permute_constants(ctx, mesh, P, static_cast<const uint32_t*>(ctx->keys.ptr));
  std::swap(ctx->vals, ctx->keys_alt);
}

// The G2P of a deferred-weight loop is k_g2p_fast (not the general corrected
// form, whose kernel updates in place).
template <int BASIS>
bool fast_g2p(const tess_ctx* ctx) {
  return !ctx->corr || separable_correction(ctx->corr, BASIS, ctx->corr_filter != nullptr);
}

// Whether the loop's test asks for a reorder of the binned particles.
inline bool reorder_wanted(tess_ctx* ctx, double threshold) {
  if (!(threshold > 0.0) || ctx->bin.n_inside == 0) return false;
  if (threshold >= 1.0) return true;
  return ctx->last_misplaced >= 0 && layered_contiguity(ctx->last_misplaced, ctx->misplaced_pairs) < threshold;
}

template <typename T, int D, int BASIS, bool STORED>
void p2g_impl(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
              const tess_weights* W, const tess_params& prm, const tess_sparsity* sp) {
  bin_particles<T, D, BASIS, STORED>(ctx, mesh, P, W);
  p2g_launch<T, D, BASIS, STORED>(ctx, mesh, G, P, W, prm, false, sp);
}

template <typename T, int D, int BASIS, bool STORED>
void g2p_impl(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
              const tess_weights* W, const tess_params& prm, const tess_sparsity* sp) {
  // a standalone G2P bins again: device addresses alone cannot prove that the
  // particle set is unchanged since the last P2G
  bin_particles<T, D, BASIS, STORED>(ctx, mesh, P, W);
  g2p_launch<T, D, BASIS, STORED>(ctx, mesh, G, P, W, prm, sp);
}

// A @G2P2G pass as one particle sweep (k_g2p2g_fast) where it is asked for
// (TESS_G2P2G_SWEEP=1 in the environment) and applies (deferred weights
// without kernel correction).  The particles were binned at their current
// positions.  The sweep runs both halves and writes the tile partials;
// p2g_launch then zeroes the grid and runs the grid-node half.  With
// write_keys the sweep also writes the next binning's keys.  Returns false
// (nothing enqueued) where the caller composes the G2P and P2G kernels, the
// default: on the 13.4 M-particle block drop the sweep takes 1.23 ms against
// 0.72 + 0.43 ms for the two kernels (its producer waves, 10 per CU against
// the G2P kernel's 12, wait on memory, and the per-round barrier couples them
// to the consumers).
inline bool g2p2g_sweep_enabled() {
  const char* e = std::getenv("TESS_G2P2G_SWEEP");
  return e && e[0] == '1' && e[1] == '\0';
}

template <typename T, int D, int BASIS>
bool g2p2g_sweep(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                 const tess_params& prm, bool write_keys, bool count_misplaced) {
  if (ctx->corr != 0 || !g2p2g_sweep_enabled()) return false;
  using SH = G2P2GShape<T, D, BASIS>;
  const Binning& b = ctx->bin;
  const MoveOut mo = write_keys && P.n > 0 ? move_out(ctx, P.n, b.ntiles) : no_moves();
  const bool aos = julia_layout(P, D);
  const uint32_t nt = uint32_t(b.ntiles);
  const SweepFn<T, D> sweep = [&](Args<T, D>& a, const uint32_t* sk, uint32_t* misplaced) {
    // algorithmic bytes: those of the G2P kernel (x, v, F read; v, ∇v, x, F,
    // σ, V written; vⁿ, v read per active node); the P2G half reads nothing
    const double nodes = double(std::max<int64_t>(ctx->last_active_nodes, 0));
    const int per_p = 2 * D + D * D + 2 * D + 3 * D * D + 1;
    const int tok = prof_begin(ctx, "k_g2p2g_tile", double(b.n_inside) * sizeof(T) * per_p + nodes * sizeof(T) * 2 * D);
    const dim3 grid(xcd_grid(b.n_active)), block(64 * (SH::NP + SH::NC));
    if (aos)
      hipLaunchKernelGGL((k_g2p2g_fast<T, D, BASIS, true, SH::NP, SH::NC>), grid, block, 0, ctx->stream, a, sk, mo,
                         nt, misplaced);
    else
      hipLaunchKernelGGL((k_g2p2g_fast<T, D, BASIS, false, SH::NP, SH::NC>), grid, block, 0, ctx->stream, a, sk, mo,
                         nt, misplaced);
    TESS_HIP(hipGetLastError());
    prof_end(ctx, tok);
  };
  p2g_launch<T, D, BASIS, false>(ctx, mesh, G, P, nullptr, prm, count_misplaced, nullptr, &sweep);
  if (P.n > b.n_inside) {  // particles outside the mesh: the G2P half's update with zero sums
    Args<T, D> a = make_args<T, D>(mesh, &G, P, nullptr, &prm);
    fill_binning_ptrs<T, D>(ctx, a);
    hipLaunchKernelGGL((k_g2p_outside<T, D>), dim3(blocks_for(P.n - b.n_inside, 256)), dim3(256), 0, ctx->stream,
                       a, static_cast<const uint32_t*>(ctx->keys_sorted.ptr), mo.nk);
    TESS_HIP(hipGetLastError());
  }
  ctx->bin.valid = false;  // positions moved
  ctx->bin.keys_ready = mo.nk != nullptr;
  return true;
}

// @G2P2G of the README program (src/Transfer/g2p2g.jl:100-159): one set of
// weights, at the positions before the pass, serves the G2P half and the P2G
// half.  One binning at those positions orders both halves: the G2P kernel
// updates the particles, then the P2G kernels scatter the updated v, V, σ with
// the weights of the old positions (stored windows, or the positions the G2P
// kernel writes aside as it moves the particles), and the grid-node half follows.
template <typename T, int D, int BASIS, bool STORED>
void g2p2g_impl(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                const tess_weights* W, const tess_params& prm) {
  bin_particles<T, D, BASIS, STORED>(ctx, mesh, P, W);
  if constexpr (!STORED) {
    if (g2p2g_sweep<T, D, BASIS>(ctx, mesh, G, P, prm, false, false)) return;
  }
  // the G2P half keeps each particle's position before its update aside
  // (deferred weights), for the P2G half's weights
  tess_particles Pold = P;
  T* xo = nullptr;
  if (!STORED && P.n > 0) {
    xo = ctx->g2p2g_x.as<T>(size_t(P.n) * D);
    Pold.x = tess_field{xo, D, 1};
  }
  g2p_launch<T, D, BASIS, STORED>(ctx, mesh, G, P, W, prm, nullptr, false, xo);
  ctx->bin.valid = true;  // the binning describes the old positions the P2G half reads
  p2g_launch<T, D, BASIS, STORED>(ctx, mesh, G, Pold, W, prm, false, nullptr);
  ctx->bin.valid = false;  // the particles have moved
}

// nsteps @G2P2G passes of the README program (deferred weights), the time loop
// of a program written as one @G2P2G block: each pass bins at the positions
// before it (from the second pass on with the keys the previous pass's G2P
// wrote), keeps those positions for its P2G half, and reorders the particles
// into the layered order at the threshold, as step_impl does.
template <typename T, int D, int BASIS>
void g2p2g_steps_impl(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                      const tess_params& prm, int nsteps, double reorder_threshold) {
  const bool sweeps = ctx->corr == 0 && g2p2g_sweep_enabled();
  MovingParticles mp(ctx, P, D, sizeof(T), !sweeps && fast_g2p<BASIS>(ctx));
  try {
    for (int s = 0; s < nsteps; ++s) {
      const bool last = s + 1 == nsteps;
      bin_particles<T, D, BASIS, false>(ctx, mesh, mp.now(), nullptr, s > 0);
      const uint32_t* dest = nullptr;
      if (reorder_wanted(ctx, reorder_threshold)) {
        if (mp.can_move()) dest = layered_maps<T, D>(ctx, mesh, mp.now());
        else layered_reorder<T, D>(ctx, mesh, mp.now());
        ctx->reorders += 1;
      }
      if (!g2p2g_sweep<T, D, BASIS>(ctx, mesh, G, mp.now(), prm, !last, reorder_threshold > 0.0)) {
        const tess_particles to = dest ? mp.other() : last ? P : mp.now();
        T* xo = P.n > 0 ? ctx->g2p2g_x.as<T>(size_t(P.n) * D) : nullptr;
        // the G2P half writes the positions before its update to xo
        g2p_launch<T, D, BASIS, false>(ctx, mesh, G, mp.now(), nullptr, prm, nullptr, !last, xo, &to, dest);
        if (dest) take_layered<T, D>(ctx, mesh, mp.now());
        mp.moved_to(to);
        tess_particles Pold = mp.now();
        if (xo) Pold.x = tess_field{xo, D, 1};
        ctx->bin.valid = true;  // the binning describes the old positions the P2G half reads
        p2g_launch<T, D, BASIS, false>(ctx, mesh, G, Pold, nullptr, prm, reorder_threshold > 0.0, nullptr);
        ctx->bin.valid = false;
      }
      // the storage order the P2G half measured is that of the particles themselves
      if (reorder_threshold > 0.0) ctx->misplaced_x_ptr = mp.now().x.ptr;
    }
  } catch (...) {
    mp.settle();
    throw;
  }
  mp.settle();
}

// nsteps of the README loop body (deferred weights).  With reorder_threshold
// in (0, 1], particles are moved into the layered order when the contiguity
// score measured by the previous step's P2G (the fraction of neighbours in the
// layered order whose storage indices are consecutive, the estimator of
// block_ordered_particle_contiguity) is below the threshold (1 reorders every
// step), the role of reorder_particles!(particles, partition; threshold) in
// the reference loop.
//
// *done (may be NULL) counts the steps whose transfers were enqueued; an SpGrid
// step that finds its storage too small raises before any of its own work, so
// after the error *done steps have run and the caller resizes and runs the
// remaining nsteps - *done.
//
// hook (may be NULL) is called as (*hook)(0, s) before step s touches the
// particles and (*hook)(1, s) once its binning and P2G grid are in place,
// before its G2P (the adjoint's replays copy states and snapshots there).
template <typename T, int D, int BASIS, bool STORED>
void step_impl(tess_ctx* ctx, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
               const tess_params& prm, int nsteps, double reorder_threshold, tess_sparsity* sp,
               int* done = nullptr, const std::function<void(int, int)>* hook = nullptr) {
  MovingParticles mp(ctx, P, D, sizeof(T), !STORED && fast_g2p<BASIS>(ctx));
  try {
    for (int s = 0; s < nsteps; ++s) {
      const bool last = s + 1 == nsteps;
      if (done) *done = s;
      if (hook) (*hook)(0, s);
      // from the second step on, the previous G2P wrote the keys (same call, so
      // nothing else moved the particles in between)
      auto bin = [&]() { bin_particles<T, D, BASIS, false>(ctx, mesh, mp.now(), nullptr, s > 0); };
      if (!sp) {
        bin();
      } else {
        // update_sparsity!(grid, xₚ) at the top of the SpGrid loop (src/Grids/grid.jl:97-101);
        // the binning's readback brings its totals too.  A binning that fails leaves
        // the new numbering, whose storage length later calls check against: sp
        // takes it before the error goes on
        run_sparsity_update(ctx, mesh, mp.now().x, P.n, *sp, nullptr, true);
        try {
          bin();
        } catch (...) {
          if (hipStreamSynchronize(ctx->stream) == hipSuccess) take_sparsity(ctx, mesh, *sp, nullptr);
          throw;
        }
        take_sparsity(ctx, mesh, *sp, nullptr);
        if (sp->storage_len > sp->capacity)
          raise(TESS_ERR_STATE, "SpGrid storage holds " + std::to_string(sp->capacity) + " nodes but the active blocks need " +
                                    std::to_string(sp->storage_len) + "; resize the grid arrays and call again");
      }
      const uint32_t* dest = nullptr;
      if (reorder_wanted(ctx, reorder_threshold)) {
        if (mp.can_move()) dest = layered_maps<T, D>(ctx, mesh, mp.now());
        else layered_reorder<T, D>(ctx, mesh, mp.now());
        ctx->reorders += 1;
      }
      // (P2G reads the particles where they are; in the layered order that its
      // G2P gives them no neighbour pair is broken)
      p2g_launch<T, D, BASIS, false>(ctx, mesh, G, mp.now(), nullptr, prm, reorder_threshold > 0.0 && !dest, sp, nullptr,
                                        sp != nullptr);
      if (dest) {
        ctx->misplaced_x_ptr = mp.now().x.ptr;
        ctx->misplaced_n = P.n;
        ctx->misplaced_pairs = ctx->bin.n_inside - ctx->bin.n_active;
        ctx->broken_count = 0;
      }
      if (hook) (*hook)(1, s);
      const tess_particles to = dest ? mp.other() : last ? P : mp.now();
      g2p_launch<T, D, BASIS, false>(ctx, mesh, G, mp.now(), nullptr, prm, sp, !last, nullptr, &to, dest);
      if (dest) take_layered<T, D>(ctx, mesh, mp.now());
      mp.moved_to(to);
    }
  } catch (...) {
    mp.settle();
    throw;
  }
  mp.settle();
  if (done) *done = nsteps;
}

template <template <typename, int, int, bool> class Op, typename... Args_>
void dispatch(int basis, const tess_mesh& mesh, bool stored, Args_&&... args) {
#define TESS_CASE(T_, D_, B_)                                     \
  if (mesh.dim == D_ && basis == B_) {                            \
    if (stored)                                                   \
      Op<T_, D_, B_, true>::run(std::forward<Args_>(args)...);    \
    else                                                          \
      Op<T_, D_, B_, false>::run(std::forward<Args_>(args)...);   \
    return;                                                       \
  }
#define TESS_CASES(T_, D_)                        \
  TESS_CASE(T_, D_, TESS_BSPLINE_LINEAR)          \
  TESS_CASE(T_, D_, TESS_BSPLINE_QUADRATIC)       \
  TESS_CASE(T_, D_, TESS_BSPLINE_CUBIC)           \
  TESS_CASE(T_, D_, TESS_UGIMP)
#ifdef TESS_PART
  TESS_CASES(TESS_PART_T, TESS_PART_D)
#endif
#undef TESS_CASES
#undef TESS_CASE
  raise(TESS_ERR_UNSUPPORTED, "unsupported (dim, dtype, basis) combination");
}

template <typename T, int D, int B, bool S>
struct P2GOp {
  static void run(tess_ctx* ctx, const tess_mesh& m, const tess_grid& G, const tess_particles& P,
                  const tess_weights* W, const tess_params& prm, const tess_sparsity* sp) {
    p2g_impl<T, D, B, S>(ctx, m, G, P, W, prm, sp);
  }
};
template <typename T, int D, int B, bool S>
struct G2POp {
  static void run(tess_ctx* ctx, const tess_mesh& m, const tess_grid& G, const tess_particles& P,
                  const tess_weights* W, const tess_params& prm, const tess_sparsity* sp) {
    g2p_impl<T, D, B, S>(ctx, m, G, P, W, prm, sp);
  }
};
template <typename T, int D, int B, bool S>
struct G2P2GOp {
  static void run(tess_ctx* ctx, const tess_mesh& m, const tess_grid& G, const tess_particles& P,
                  const tess_weights* W, const tess_params& prm) {
    g2p2g_impl<T, D, B, S>(ctx, m, G, P, W, prm);
  }
};
template <typename T, int D, int B, bool S>
struct G2P2GStepsOp {
  static void run(tess_ctx* ctx, const tess_mesh& m, const tess_grid& G, const tess_particles& P,
                  const tess_params& prm, int nsteps, double thr) {
    if constexpr (!S) g2p2g_steps_impl<T, D, B>(ctx, m, G, P, prm, nsteps, thr);
  }
};
template <typename T, int D, int B, bool S>
struct StepOp {
  static void run(tess_ctx* ctx, const tess_mesh& m, const tess_grid& G, const tess_particles& P,
                  const tess_params& prm, int nsteps, double thr, tess_sparsity* sp, int* done) {
    if constexpr (!S) step_impl<T, D, B, false>(ctx, m, G, P, prm, nsteps, thr, sp, done);
  }
};

}  // namespace
}  // namespace tess
