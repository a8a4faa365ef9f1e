// Batches of independent scenes (the engine's batching extension; no
// counterpart in the reference).  Scenes of one dimension, dtype and basis but
// their own mesh, particle count, constants and Δt are stepped together: the
// tiles and particles of all scenes share one index space (scene s owns tiles
// [toff_s, toff_s+1) and particles [poff_s, poff_s+1)), so each kernel of a
// step — keys, sort, tile runs, P2G, gather, G2P — is one launch for the whole
// batch.  Tile kernels look their scene up from the tile index
// (scene_of/bind_scene in transfer_impl.hpp).  An autotuner times the launch
// variants (waves per tile in P2G and G2P) on the batch itself.
#ifdef TESS_PART

#include "transfer_impl.hpp"

#include <algorithm>
#include <vector>

namespace tess {
namespace {

template <typename T, int D>
SceneRec<T, D> scene_record(const tess_scene& sc, int64_t toff, int64_t poff) {
  SceneRec<T, D> r;
  std::memset(static_cast<void*>(&r), 0, sizeof(r));
  const Args<T, D> a = make_args<T, D>(sc.mesh, &sc.grid, sc.particles, nullptr, &sc.params);
  r.mesh = a.mesh;
  r.x = a.x;
  r.v = a.v;
  r.V = a.V;
  r.gradv = a.gradv;
  r.F = a.F;
  r.sigma = a.sigma;
  r.l = a.l;
  r.logE = a.logE;
  r.gm = a.gm;
  r.gmv = a.gmv;
  r.gf = a.gf;
  r.gvn = a.gvn;
  r.gv = a.gv;
  r.mp = a.mp;
  r.dt = a.dt;
  r.lambda = a.lambda;
  r.mu = a.mu;
  r.V0 = a.V0;
  for (int d = 0; d < D; ++d) {
    r.gravity[d] = a.gravity[d];
    r.ntiles[d] = a.ntiles[d];
  }
  r.slip = a.slip;
  r.toff = toff;
  r.poff = poff;
  r.n = sc.particles.n;
  r.nnodes = 1;
  for (int d = 0; d < D; ++d) r.nnodes *= sc.mesh.dims[d];
  return r;
}

// scene of each global tile: the tile kernels start from it (a search of the
// scenes' first tiles was eight dependent loads at the start of each workgroup)
__global__ __launch_bounds__(256) void k_tile_scene(const int64_t* __restrict__ toff, int32_t nscenes, int64_t ntiles,
                                                    uint32_t* __restrict__ tile_scene) {
  const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (t < ntiles) tile_scene[t] = uint32_t(scene_of(toff, nscenes, t));
}

template <typename T, int D>
void batch_create_impl(tess_ctx* ctx, tess_batch& b) {
  std::vector<SceneRec<T, D>> recs;
  for (int s = 0; s < b.nscenes; ++s) recs.push_back(scene_record<T, D>(b.scenes[size_t(s)], b.toff[size_t(s)], b.poff[size_t(s)]));
  void* p = b.recs.get(recs.size() * sizeof(SceneRec<T, D>));
  TESS_HIP(hipMemcpyAsync(p, recs.data(), recs.size() * sizeof(SceneRec<T, D>), hipMemcpyHostToDevice, ctx->stream));
  TESS_HIP(hipMemcpyAsync(b.d_toff.get(b.toff.size() * 8), b.toff.data(), b.toff.size() * 8, hipMemcpyHostToDevice,
                          ctx->stream));
  TESS_HIP(hipMemcpyAsync(b.d_poff.get(b.poff.size() * 8), b.poff.data(), b.poff.size() * 8, hipMemcpyHostToDevice,
                          ctx->stream));
  std::vector<int32_t> nt;  // tiles per axis of each scene
  for (const auto& r : recs)
    for (int d = 0; d < 3; ++d) nt.push_back(d < D ? r.ntiles[d < D ? d : 0] : 1);
  TESS_HIP(hipMemcpyAsync(b.d_nt.get(nt.size() * 4), nt.data(), nt.size() * 4, hipMemcpyHostToDevice, ctx->stream));
  hipLaunchKernelGGL(k_tile_scene, dim3(blocks_for(b.tiles_total, 256)), dim3(256), 0, ctx->stream,
                     static_cast<const int64_t*>(b.d_toff.ptr), b.nscenes, b.tiles_total,
                     b.d_tscene.as<uint32_t>(size_t(std::max<int64_t>(b.tiles_total, 1))));
  TESS_HIP(hipGetLastError());
  TESS_HIP(hipStreamSynchronize(ctx->stream));
}

template <typename T, int D>
Args<T, D> batch_args(tess_ctx* ctx, tess_batch& b) {
  Args<T, D> a;
  std::memset(static_cast<void*>(&a), 0, sizeof(a));
  a.scenes = static_cast<const SceneRec<T, D>*>(b.recs.ptr);
  a.scene_toff = static_cast<const int64_t*>(b.d_toff.ptr);
  a.scene_poff = static_cast<const int64_t*>(b.d_poff.ptr);
  a.tile_scene = static_cast<const uint32_t*>(b.d_tscene.ptr);
  a.nscenes = b.nscenes;
  a.n = b.ntot;
  fill_binning_ptrs<T, D>(ctx, a);
  return a;
}

// Arguments that build the batch's tables into the alternate set.
inline TabArgs batch_tables(tess_ctx* ctx, tess_batch& B) {
  TabArgs t = table_args(ctx, B.tiles_total);
  t.scene_toff = static_cast<const int64_t*>(B.d_toff.ptr);
  t.scene_nt = static_cast<const int32_t*>(B.d_nt.ptr);
  t.tile_scene = static_cast<const uint32_t*>(B.d_tscene.ptr);
  return t;
}

// Full sort of the batch's keys on a call's first step (the batch-wide tile
// space), the merge of the changed keys from then on, and the tile tables, as
// bin_particles does.
template <typename T, int D, int BASIS>
void batch_bin_run(tess_ctx* ctx, tess_batch& B, bool keys_from_g2p);

template <typename T, int D, int BASIS>
void batch_bin(tess_ctx* ctx, tess_batch& B, bool keys_from_g2p) {
  batch_bin_run<T, D, BASIS>(ctx, B, keys_from_g2p);
  if (TESS_DEBUG && B.ntot > 0) {
    const Binning& b = ctx->bin;
    debug_check_binning(ctx->stream, static_cast<const uint32_t*>(ctx->keys_sorted.ptr),
                        static_cast<const uint32_t*>(ctx->vals.ptr), static_cast<const uint32_t*>(ctx->tile_start.ptr),
                        static_cast<const uint32_t*>(ctx->tile_end.ptr),
                        static_cast<const uint32_t*>(ctx->active_tiles.ptr), B.ntot, B.tiles_total, b.n_active,
                        b.n_inside, "batch_bin");
  }
}

template <typename T, int D, int BASIS>
void batch_bin_run(tess_ctx* ctx, tess_batch& B, bool keys_from_g2p) {
  const int64_t n = B.ntot;
  const uint64_t ntiles = uint64_t(B.tiles_total);
  Binning& b = ctx->bin;
  const bool incremental = keys_from_g2p && B.keys_ready && B.binned && b.n == n && b.ntiles == int64_t(ntiles) &&
                           n > 0;
  B.keys_ready = false;
  b.valid = false;
  b.state_valid = false;  // the single-scene incremental state does not describe a batch
  b.keys_ready = false;
  uint32_t* counters = ctx->counters.as<uint32_t>(64);
  const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx->counters_host);
  const size_t m = size_t(std::max<int64_t>(n, 1));
  TabArgs tab = batch_tables(ctx, B);
  tab.tile_max = merge_tile_max(n);
  const int tok = prof_begin(ctx, "binning", 0.0);
  if (incremental) {
    // the last G2P wrote the keys and counted the particles whose key changed;
    // with none the previous order and tile lists stand
    tab.crowd = merge_crowd(n);
    tab.many = merge_many(n);
    const uint32_t seq = build_tables(ctx, tab);
    MergeArgs merge;
    if (!b.crowded) merge = merge_ahead(ctx, n, int64_t(ntiles), b.n_active);
    wait_report(ctx, seq);
    take_report(ctx);
    ctx->last_active_nodes = int64_t(hc[CNT_NODES]);
    if (hc[CNT_MOVED] == 0) {
      B.kept_binnings += 1;
      b.valid = true;
      prof_end(ctx, tok);
      return;
    }
    if (b.crowded || hc[CNT_RESORT] || hc[CNT_ARRIVE] > tab.many) resort_keys(ctx, n, key_bits_for(ntiles * 64));
    else merge_finish(ctx, merge, b.n_inside);
  } else {
    Args<T, D> a = batch_args<T, D>(ctx, B);
    uint32_t* skeys = ctx->keys_sorted.as<uint32_t>(m);
    uint32_t* perm = ctx->vals.as<uint32_t>(m);
    if (n > 0) {
      uint32_t* keys = ctx->keys.as<uint32_t>(m);
      hipLaunchKernelGGL((k_bin_keys<T, D, BASIS, false, true>), dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, a,
                         keys, uint32_t(ntiles), counters);
      TESS_HIP(hipGetLastError());
      radix_sort_pairs(ctx, keys, nullptr, skeys, perm, n, key_bits_for(ntiles * 64));
    }
    launch_tile_counts(ctx->stream, skeys, n, int64_t(ntiles), tab.stay, tab.tin);
    wait_report(ctx, build_tables(ctx, tab));
    take_report(ctx);
    ctx->last_active_nodes = int64_t(hc[CNT_NODES]);  // written by the previous step's gather
  }
  prof_end(ctx, tok);
  if (hc[CNT_ERR] & ERR_GIMP_LENGTH) raise(TESS_ERR_ARGUMENT, "uGIMP requires 0 ≤ pt.l ≤ spacing(mesh)");
  swap_tables(ctx);
  b.n_inside = int64_t(hc[CNT_INSIDE]);
  b.n_active = int64_t(hc[CNT_ACTIVE]);
  b.n_nodeblocks = int64_t(hc[CNT_NB]);
  b.crowded = (hc[CNT_RESORT] & RESORT_TILE) != 0;
  b.ntiles = int64_t(ntiles);
  b.n = n;
  b.valid = true;
  B.binned = true;
}

// ---- layered reorder of a batch ------------------------------------------------
//
// Each scene's particles into the layered order of its tiles (the order the
// tile kernels read contiguously), its particles outside the mesh after them
// in their previous order.  Every particle stays in its scene's arrays: the
// layered slot L of a scene-s particle becomes global index L + (particles
// outside the mesh in scenes before s), since the scene's inside particles
// start at sorted position poff_s minus those.

__global__ void k_mark_outside(const uint32_t* __restrict__ perm, int64_t from, int64_t n, uint32_t* __restrict__ flag) {
  const int64_t j = from + int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (j < n) flag[perm[j]] = 1u;
}

// new global index of the particle at each sorted position (pout) and the
// gather order (new index -> old index)
template <typename T, int D>
__global__ __launch_bounds__(256) void k_batch_new_index(Args<T, D> a, const uint32_t* __restrict__ layered,
                                                         const uint32_t* __restrict__ R, uint32_t* __restrict__ order,
                                                         uint32_t* __restrict__ pout) {
  const int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (j < a.n) {
    const uint32_t g = a.perm[j];
    const int s = scene_near(a.scene_poff, a.nscenes, int64_t(g));
    const int64_t p0 = a.scene_poff[s], p1 = a.scene_poff[s + 1];
    const uint32_t dst = j < a.n_inside ? uint32_t(int64_t(layered[j]) + int64_t(R[p0]))
                                        : uint32_t(p1 - int64_t(R[p1] - R[p0]) + int64_t(R[g] - R[p0]));
    order[dst] = g;
    pout[j] = dst;
  }
}

// scalars of a particle's fields x, v, V, ∇v, F, σ, l, log E
template <int D>
constexpr int kStateWidth = 2 * D + 2 + 3 * D * D + 1;

// With `order`: every field of particle order[i] into row i of the packed
// scratch (field-major: field f's rows start at its component offset times n).
// Without: row i back into particle i.  A particle's fields are all loaded before
// the first is stored, contiguous ones in words of up to 16 bytes: scalar by
// scalar, a field's loads behind the previous one's stores, the two launches took
// 547 us each on 9.7 M 2D Float32 particles.
template <typename T, int D>
__global__ __launch_bounds__(256) void k_batch_state(Args<T, D> a, T* __restrict__ scratch,
                                                     const uint32_t* __restrict__ order) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= a.n) return;
  const int s = scene_near(a.scene_poff, a.nscenes, i);
  const SceneRec<T, D>& r = a.scenes[s];
  const int64_t li = (order ? int64_t(order[i]) : i) - r.poff;  // the permutation stays within the scene
  T x[D], v[D], V[1], gradv[D * D], F[D * D], sigma[D * D], l[1], logE[1];
  auto each = [&](auto&& f) {
    int64_t off = 0;
    auto field = [&](const DField<T>& d, auto& val) {
      constexpr int NC = int(sizeof(val) / sizeof(T));
      if (d.p) f(d, val, off * a.n + i * NC);
      off += NC;
    };
    field(r.x, x);
    field(r.v, v);
    field(r.V, V);
    field(r.gradv, gradv);
    field(r.F, F);
    field(r.sigma, sigma);
    field(r.l, l);
    field(r.logE, logE);
  };
  auto rows = [](const DField<T>& d, int nc) { return d.es == nc && (nc == 1 || d.cs == 1); };
  each([&](const DField<T>& d, auto& val, int64_t at) {
    if (order) get_row(rows(d, int(sizeof(val) / sizeof(T))), d, li, val);
    else __builtin_memcpy(val, scratch + at, sizeof(val));
  });
  each([&](const DField<T>& d, auto& val, int64_t at) {
    if (order) __builtin_memcpy(scratch + at, val, sizeof(val));
    else put_row(rows(d, int(sizeof(val) / sizeof(T))), d, li, val);
  });
}

// Reorders the scenes' particles when the batch's contiguity score is below
// `threshold`, or at every call when threshold >= 1 (reorder_particles!,
// src/Parallel/cpu_block_strategy.jl:222-278).  The score is the fraction of
// neighbours in the layered order whose storage indices are consecutive,
// counted by the previous step's P2G, or on a call's first step by
// k_layered_order; the binning's permutation follows the particles.
template <typename T, int D>
void batch_reorder(tess_ctx* ctx, tess_batch& B, double threshold) {
  const Binning& b = ctx->bin;
  const int64_t n = B.ntot;
  if (n == 0 || b.n_active == 0) return;
  Args<T, D> a = batch_args<T, D>(ctx, B);
  uint32_t* layered = ctx->keys_alt.as<uint32_t>(size_t(n));
  uint32_t* order = ctx->keys.as<uint32_t>(size_t(n));  // the raw keys are dead after the sort
  uint32_t* pout = ctx->inc_pout.as<uint32_t>(size_t(n));
  uint32_t* R = ctx->inc_rank.as<uint32_t>(size_t(n) + 1);
  uint32_t* broken = ctx->reorder_cnt.as<uint32_t>(size_t(b.n_active));
  uint32_t* counters = ctx->counters.as<uint32_t>(CNT_SLOTS);
  const uint32_t* sk = static_cast<const uint32_t*>(ctx->keys_sorted.ptr);
  uint32_t* hc = reinterpret_cast<uint32_t*>(ctx->counters_host);
  const bool by_p2g_count = threshold < 1.0 && B.counted;
  if (by_p2g_count) {
    // the previous step's P2G counted the broken pairs; the binning's readback
    // brought the count to the host
    if (!(layered_contiguity(int64_t(hc[CNT_MISPLACED]), B.counted_pairs) < threshold)) return;
  }
  const bool count_here = threshold < 1.0 && !B.counted;
  hipLaunchKernelGGL((k_layered_order<T, D>), dim3(unsigned(b.n_active)), dim3(64), 0, ctx->stream, a, sk, pout,
                     layered, count_here ? broken : nullptr);
  TESS_HIP(hipGetLastError());
  if (count_here) {
    sum_u32(ctx, broken, b.n_active, counters + CNT_MISPLACED);
    TESS_HIP(hipMemcpyAsync(hc + CNT_MISPLACED, counters + CNT_MISPLACED, sizeof(uint32_t), hipMemcpyDeviceToHost,
                            ctx->stream));
    TESS_HIP(hipStreamSynchronize(ctx->stream));
    if (!(layered_contiguity(int64_t(hc[CNT_MISPLACED]), b.n_inside - b.n_active) < threshold)) return;
  }
  TESS_HIP(hipMemsetAsync(R, 0, (size_t(n) + 1) * sizeof(uint32_t), ctx->stream));
  if (n > b.n_inside) {
    hipLaunchKernelGGL(k_mark_outside, dim3(blocks_for(n - b.n_inside, 256)), dim3(256), 0, ctx->stream, a.perm,
                       b.n_inside, n, R);
    TESS_HIP(hipGetLastError());
  }
  exclusive_scan_u32(ctx, R, n + 1, nullptr);
  hipLaunchKernelGGL((k_batch_new_index<T, D>), dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, a, layered, R,
                     order, pout);
  TESS_HIP(hipGetLastError());
  T* scratch = ctx->reorder_tmp.as<T>(size_t(n) * kStateWidth<D>);
  hipLaunchKernelGGL((k_batch_state<T, D>), dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, a, scratch,
                     static_cast<const uint32_t*>(order));
  TESS_HIP(hipGetLastError());
  hipLaunchKernelGGL((k_batch_state<T, D>), dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, a, scratch,
                     static_cast<const uint32_t*>(nullptr));
  TESS_HIP(hipGetLastError());
  TESS_HIP(hipMemcpyAsync(ctx->vals.ptr, pout, size_t(n) * sizeof(uint32_t), hipMemcpyDeviceToDevice, ctx->stream));
  B.reorders += 1;
  if (by_p2g_count) B.reorders_by_count += 1;
}

template <typename T, int D, int BASIS, int NP>
void launch_p2g(tess_ctx* ctx, const Args<T, D>& a, int64_t n_active, const uint32_t* sk, uint32_t* broken) {
  hipLaunchKernelGGL((k_p2g_fast<T, D, BASIS, NP, true, true>), dim3(xcd_grid(n_active)), dim3(64 * NP), 0,
                     ctx->stream, a, sk, broken);
  TESS_HIP(hipGetLastError());
}

template <typename T, int D, int BASIS, int NW>
void launch_g2p(tess_ctx* ctx, const Args<T, D>& a, int64_t n_active, const uint32_t* sk, const MoveOut& mo) {
  const uint32_t nt = uint32_t(ctx->bin.ntiles);
  hipLaunchKernelGGL((k_g2p_fast<T, D, BASIS, true, NW, true>), dim3(xcd_grid(n_active)), dim3(64 * NW), 0,
                     ctx->stream, a, sk, mo, nt);
  TESS_HIP(hipGetLastError());
}

template <typename T, int D, int BASIS>
void batch_step_impl(tess_ctx* ctx, tess_batch& B, int nsteps) {
  constexpr int SW = support_width(BASIS);
  B.counted = false;  // the context's counters may have served other calls since
  if (B.last_graph) {
    // graph-mode steps wrote node blocks the eager stale list does not name
    B.zeroed = false;
    B.last_graph = false;
  }
  for (int s = 0; s < nsteps; ++s) {
    // from the second step of the call on, the previous G2P wrote the keys
    batch_bin<T, D, BASIS>(ctx, B, s > 0);
    if (B.reorder_threshold > 0.0) {
      const int tok = prof_begin(ctx, "reorder", 0.0);
      batch_reorder<T, D>(ctx, B, B.reorder_threshold);
      prof_end(ctx, tok);
    }
    const Binning& b = ctx->bin;
    Args<T, D> a = batch_args<T, D>(ctx, B);
    // zero what this step does not overwrite: every grid the first time, then
    // the node blocks written last step and not now
    if (!B.zeroed) {
      hipLaunchKernelGGL((k_zero_grid_batch<T, D>), dim3(blocks_for(B.max_nodes, 256), unsigned(B.nscenes)), dim3(256),
                         0, ctx->stream, a);
      TESS_HIP(hipGetLastError());
      B.zeroed = true;
    } else if (B.prev_nb > 0) {
      hipLaunchKernelGGL((k_zero_stale<T, D, true>), dim3(unsigned(B.prev_nb)), dim3(64), 0, ctx->stream, a,
                         static_cast<const uint32_t*>(B.prev_list.ptr), B.prev_nb);
      TESS_HIP(hipGetLastError());
    }
    const uint32_t* sk = static_cast<const uint32_t*>(ctx->keys_sorted.ptr);
    if (b.n_active > 0) {
      a.partials = ctx->partials.as<T>(size_t(b.n_active) * Part<D, SW>::SIZE);
      const int tok = prof_begin(ctx, "k_p2g_tile", double(b.n_inside) * sizeof(T) * (2 * D + 1 + D * D));
      // with a threshold in (0, 1) P2G counts the broken layered pairs for the
      // next step's reorder test
      const bool count = B.reorder_threshold > 0.0 && B.reorder_threshold < 1.0;
      uint32_t* broken = count ? lane_counters(ctx) : nullptr;
      if (D == 3 || (B.variant & 1)) launch_p2g<T, D, BASIS, SW>(ctx, a, b.n_active, sk, broken);
      else launch_p2g<T, D, BASIS, 1>(ctx, a, b.n_active, sk, broken);
      prof_end(ctx, tok);
      if (count) B.counted_pairs = b.n_inside - b.n_active;
      B.counted = count;
    } else {
      B.counted = false;
    }
    if (b.n_nodeblocks > 0) {
      const int tok = prof_begin(ctx, "k_gather_grid", 0.0);
      hipLaunchKernelGGL((k_gather_grid<T, D, SW, true, true>), dim3(xcd_grid(b.n_nodeblocks)), dim3(64), 0, ctx->stream,
                         a, lane_counters(ctx));
      TESS_HIP(hipGetLastError());
      prof_end(ctx, tok);
      uint32_t* prev = B.prev_list.as<uint32_t>(size_t(b.n_nodeblocks));
      TESS_HIP(hipMemcpyAsync(prev, ctx->nb_list.ptr, size_t(b.n_nodeblocks) * sizeof(uint32_t),
                              hipMemcpyDeviceToDevice, ctx->stream));
    }
    B.prev_nb = b.n_nodeblocks;
    // next-step keys at the sorted positions while the call goes on
    const MoveOut mo = s + 1 < nsteps && B.ntot > 0 ? move_out(ctx, B.ntot, B.tiles_total) : no_moves();
    if (b.n_active > 0) {
      const int tok = prof_begin(ctx, "k_g2p_tile",
                                 double(b.n_inside) * sizeof(T) * (2 * D + D * D + 2 * D + 3 * D * D + 1));
      if (B.variant & 4) launch_g2p<T, D, BASIS, 1>(ctx, a, b.n_active, sk, mo);
      else if (B.variant & 2) launch_g2p<T, D, BASIS, 2>(ctx, a, b.n_active, sk, mo);
      else launch_g2p<T, D, BASIS, 4>(ctx, a, b.n_active, sk, mo);
      prof_end(ctx, tok);
    }
    if (B.ntot > b.n_inside) {
      hipLaunchKernelGGL((k_g2p_outside<T, D, true>), dim3(blocks_for(B.ntot - b.n_inside, 256)), dim3(256), 0,
                         ctx->stream, a, sk, mo.nk);
      TESS_HIP(hipGetLastError());
    }
    B.keys_ready = mo.nk != nullptr;
  }
  // the single-scene zeroing bookkeeping no longer describes any grid
  ctx->last_grid_m = nullptr;
  ctx->bin.valid = false;
}

// ---- graph mode ----------------------------------------------------------------
//
// With bit 3 of the variant a batch steps on a private context (its own stream
// and scratch, so no other call can move the buffers a captured step points
// at).  Its step reads nothing back to the host: the binning merges the
// particles whose key changed (every launch size fixed by the batch), the counts of inside
// particles, active tiles and touched node blocks stay on the device, and the
// tile and node-block kernels are persistent launches (a grid sized to the
// device by its occupancy) that walk those lists up to the device-side counts.
// Zeroing is done by kernels.  The step is captured once into a hipGraph and
// replayed; the reorder test, which needs the host, runs between chunks of
// graph_chunk replays.

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* __restrict__ p, int64_t n, uint32_t v) {
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) p[i] = v;
}

void fill_u32(hipStream_t st, uint32_t* p, int64_t n, uint32_t v) {
  if (n <= 0) return;
  const unsigned g = unsigned(std::min<int64_t>(blocks_for(n, 256), 4096));
  hipLaunchKernelGGL(k_fill_u32, dim3(g), dim3(256), 0, st, p, n, v);
  TESS_HIP(hipGetLastError());
}

// The nodes of the node blocks listed by the previous step and not flagged by
// this one, back to zero (the count read on the device).
template <typename T, int D>
__global__ __launch_bounds__(64) void k_zero_stale_persist(Args<T, D> a, const uint32_t* __restrict__ prev_list,
                                                           const uint32_t* __restrict__ prev_count) {
  const int64_t np = int64_t(*prev_count);
  for (int64_t j = blockIdx.x; j < np; j += gridDim.x) {
    const uint32_t B = prev_list[j];
    zero_stale_block<T, D, true>(a, B);
  }
}

// This step's node-block list and count become the next step's stale list.
__global__ __launch_bounds__(256) void k_save_list(const uint32_t* __restrict__ list, const uint32_t* __restrict__ count,
                                                   uint32_t* __restrict__ prev_list, uint32_t* __restrict__ prev_count) {
  const int64_t n = int64_t(*count);
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256)
    prev_list[i] = list[i];
  if (blockIdx.x == 0 && threadIdx.x == 0) *prev_count = uint32_t(n);
}

// Particles outside their mesh (sorted positions from the device count of
// inside particles to n): the update with zero grid increments.
template <typename T, int D>
__global__ __launch_bounds__(256) void k_g2p_outside_persist(Args<T, D> a, const uint32_t* __restrict__ skeys,
                                                             uint32_t* __restrict__ nk,
                                                             const uint32_t* __restrict__ n_inside) {
  const int64_t from = int64_t(*n_inside);
  for (int64_t j = from + int64_t(blockIdx.x) * 256 + threadIdx.x; j < a.n; j += int64_t(gridDim.x) * 256) {
    nk[j] = skeys[j];  // the position does not change: the key stays
    uint32_t pid = a.perm[j];
    pid -= uint32_t(bind_scene(a, scene_of(a.scene_poff, a.nscenes, pid)).poff);
    T dv[D], L[D * D], dx[D];
#pragma unroll
    for (int c = 0; c < D; ++c) {
      dv[c] = T(0);
      dx[c] = T(0);
    }
#pragma unroll
    for (int k = 0; k < D * D; ++k) L[k] = T(0);
    particle_update<T, D>(a, ParticleIn<T, D>(a, pid), pid, pid, dv, L, dx);
  }
}

int device_cus(int dev) {
  int c = 0;
  TESS_HIP(hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev));
  return std::max(c, 1);
}

// Workgroups of a persistent launch: twice what the occupancy query reports
// the CUs hold at once, at most one per work item, a multiple of 8.
unsigned persist_grid(const void* kern, int threads, int64_t max_items, int cus) {
  int per = 0;
  TESS_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, threads, 0));
  int64_t g = 2 * int64_t(std::max(per, 1)) * cus;
  g = std::min<int64_t>(g, int64_t(xcd_grid(std::max<int64_t>(max_items, 1))));
  return unsigned(((g + 7) / 8) * 8);
}

template <typename T, int D, int BASIS, int NP>
const void* p2g_persist_fn() {
  return reinterpret_cast<const void*>(&k_p2g_fast_persist<T, D, BASIS, NP, true, true>);
}
template <typename T, int D, int BASIS, int NW>
const void* g2p_persist_fn() {
  return reinterpret_cast<const void*>(&k_g2p_fast_persist<T, D, BASIS, true, NW, true>);
}

template <typename T, int D, int BASIS>
void batch_graph_grids(tess_ctx* g, tess_batch& B) {
  constexpr int SW = support_width(BASIS);
  const int cus = device_cus(g->device);
  const int64_t nt = B.tiles_total;
  const bool split = D == 3 || (B.variant & 1);
  B.grid_p2g = split ? persist_grid(p2g_persist_fn<T, D, BASIS, SW>(), 64 * SW, nt, cus)
                     : persist_grid(p2g_persist_fn<T, D, BASIS, 1>(), 64, nt, cus);
  if (B.variant & 4) B.grid_g2p = persist_grid(g2p_persist_fn<T, D, BASIS, 1>(), 64, nt, cus);
  else if (B.variant & 2) B.grid_g2p = persist_grid(g2p_persist_fn<T, D, BASIS, 2>(), 128, nt, cus);
  else B.grid_g2p = persist_grid(g2p_persist_fn<T, D, BASIS, 4>(), 256, nt, cus);
  B.grid_gather = persist_grid(reinterpret_cast<const void*>(&k_gather_grid_persist<T, D, SW, true, true>), 64, nt,
                               cus);
  B.grid_zero = persist_grid(reinterpret_cast<const void*>(&k_zero_stale_persist<T, D>), 64, nt, cus);
  B.grid_out = persist_grid(reinterpret_cast<const void*>(&k_g2p_outside_persist<T, D>), 256,
                            ceil_div(std::max<int64_t>(B.ntot, 1), int64_t(256)), cus);
}

// Graph mode's binning double buffer: sorted keys, permutation and tile tables
// in set 0 (keys_sorted, vals, tile_start, ...) or set 1 (skeys2, perm2,
// alt_start, ...).
struct BinSet {
  uint32_t *keys, *perm, *start, *end, *flag, *slot, *active, *nb_flag, *nb_list;
};
inline BinSet bin_set(tess_ctx* g, int64_t n, int64_t ntiles, int which) {
  const size_t m = size_t(std::max<int64_t>(n, 1)), nt = size_t(ntiles) + 1;
  auto get = [&](Buffer& a, Buffer& b, size_t k) { return (which ? b : a).as<uint32_t>(k); };
  return BinSet{get(g->keys_sorted, g->skeys2, m),       get(g->vals, g->perm2, m),
                get(g->tile_start, g->alt_start, nt),    get(g->tile_end, g->alt_end, nt),
                get(g->tile_flag, g->alt_flag, nt),      get(g->tile_slot, g->alt_slot, nt),
                get(g->active_tiles, g->alt_active, nt), get(g->nb_flag, g->alt_nb_flag, nt),
                get(g->nb_list, g->alt_nb_list, nt)};
}

// One step of the batch on context g, every launch size fixed and every count
// on the device.  full: the binning sorts every particle's key into set 0
// (the step that starts each call); else it merges the particles whose key
// the previous step's G2P changed (MoveOut, over the sorted positions and tiles
// of set `in`) into set 1-in, the form that is captured, whatever their number:
// no host is there to sort them instead.  Either way the G2P writes the next keys
// and each tile's counts and leavers.
template <typename T, int D, int BASIS>
void batch_graph_step(tess_ctx* g, tess_batch& B, bool full, int in) {
  constexpr int SW = support_width(BASIS);
  const int64_t n = B.ntot;
  const uint64_t ntiles = uint64_t(B.tiles_total);
  const size_t m = size_t(std::max<int64_t>(n, 1));
  hipStream_t st = g->stream;
  uint32_t* counters = g->counters.as<uint32_t>(64);
  uint32_t* keys = g->keys.as<uint32_t>(m);
  const int64_t nt64 = int64_t(ntiles);
  const int out = full ? 0 : 1 - in;
  const BinSet cur = bin_set(g, n, nt64, out), old = bin_set(g, n, nt64, 1 - out);
  const MoveOut mo = move_out(g, n, nt64);
  uint2* seg = g->inc_seg.as<uint2>(m);
  uint2* seg_alt = g->inc_seg2.as<uint2>(m);
  uint32_t* lanes = lane_counters(g);
  uint32_t* prev_list = B.g_prev_list.as<uint32_t>(ntiles);
  uint32_t* prev_count = B.g_prev_count.as<uint32_t>(64);
  T* partials = g->partials.as<T>(size_t(ntiles) * Part<D, SW>::SIZE);
  // the scans' work area at its largest use (the reorder's ranks), so no later
  // call moves it
  g->scan_tmp.get(scan_work_bytes(n + 1));
  uint32_t* skeys = cur.keys;
  const uint32_t* nblist = cur.nb_list;
  Args<T, D> a = batch_args<T, D>(g, B);
  a.perm = cur.perm;
  a.tile_start = cur.start;
  a.tile_end = cur.end;
  a.active = cur.active;
  a.tile_flag = cur.flag;
  a.tile_slot = cur.slot;
  a.nb_list = cur.nb_list;
  a.nb_flag = cur.nb_flag;
  a.partials = partials;
  TabArgs tab = batch_tables(g, B);
  tab.start = cur.start;
  tab.end = cur.end;
  tab.flag = cur.flag;
  tab.slot = cur.slot;
  tab.active = cur.active;
  tab.nb_flag = cur.nb_flag;
  tab.nb_list = cur.nb_list;
  tab.keep_err = 1;  // the call's one readback of the error flags comes at its end
  if (full) {
    fill_u32(st, counters + CNT_ERR, 1, 0u);
    if (n > 0) {
      hipLaunchKernelGGL((k_bin_keys<T, D, BASIS, false, true>), dim3(blocks_for(n, 256)), dim3(256), 0, st, a, keys,
                         uint32_t(ntiles), counters);
      TESS_HIP(hipGetLastError());
      radix_sort_pairs(g, keys, nullptr, skeys, cur.perm, n, key_bits_for(ntiles * 64));
    }
    launch_tile_counts(st, skeys, n, nt64, tab.stay, tab.tin);
    launch_tables(st, tab);
  } else {
    // the particles whose key changed merged into the previous order, every
    // count on the device
    launch_tables(st, tab);
    MergeArgs g2;
    std::memset(static_cast<void*>(&g2), 0, sizeof(g2));
    g2.n = n;
    g2.ntiles = nt64;
    g2.old_active = old.active;
    g2.old_start = old.start;
    g2.old_end = old.end;
    g2.new_active = cur.active;
    g2.new_start = cur.start;
    g2.new_end = cur.end;
    g2.old_count = counters + CNT_PREV_ACTIVE;
    g2.new_count = counters + CNT_ACTIVE;
    g2.old_active_n = g2.new_active_n = nt64;
    g2.stay = mo.stay;
    g2.nk = mo.nk;
    g2.perm_old = old.perm;
    g2.seg_off = tab.seg;
    g2.out = mo.out;
    g2.seg = seg;
    g2.seg_alt = seg_alt;
    g2.keys_new = cur.keys;
    g2.perm_new = cur.perm;
    g2.counters = counters;
    g2.crowd = merge_crowd(n);
    g2.pos_bits = key_bits_for(uint64_t(m));
    launch_merge(st, g2, n > 0 ? unsigned(std::min<int64_t>(blocks_for(n, 256), 512)) : 0u);
  }
  // grids: the previous step's stale node blocks, P2G, the grid-node half
  hipLaunchKernelGGL((k_zero_stale_persist<T, D>), dim3(B.grid_zero), dim3(64), 0, st, a,
                     static_cast<const uint32_t*>(prev_list), static_cast<const uint32_t*>(prev_count));
  TESS_HIP(hipGetLastError());
  const uint32_t* sk = skeys;
  const uint32_t* n_active = counters + CNT_ACTIVE;
  const uint32_t* n_nb = counters + CNT_NB;
  // bit 4: persistent grids; else one workgroup per possible tile or node block
  const bool persist = (B.variant & 16) != 0;
  const dim3 all_tiles(xcd_grid(int64_t(ntiles)));
  uint32_t* none = nullptr;
  if (D == 3 || (B.variant & 1)) {
    if (persist)
      hipLaunchKernelGGL((k_p2g_fast_persist<T, D, BASIS, SW, true, true>), dim3(B.grid_p2g), dim3(64 * SW), 0, st, a,
                         sk, none, n_active);
    else
      hipLaunchKernelGGL((k_p2g_fast_grid<T, D, BASIS, SW, true, true>), all_tiles, dim3(64 * SW), 0, st, a, sk, none,
                         n_active);
  } else {
    if (persist)
      hipLaunchKernelGGL((k_p2g_fast_persist<T, D, BASIS, 1, true, true>), dim3(B.grid_p2g), dim3(64), 0, st, a, sk,
                         none, n_active);
    else
      hipLaunchKernelGGL((k_p2g_fast_grid<T, D, BASIS, 1, true, true>), all_tiles, dim3(64), 0, st, a, sk, none,
                         n_active);
  }
  TESS_HIP(hipGetLastError());
  if (persist)
    hipLaunchKernelGGL((k_gather_grid_persist<T, D, SW, true, true>), dim3(B.grid_gather), dim3(64), 0, st, a, lanes,
                       n_nb);
  else
    hipLaunchKernelGGL((k_gather_grid_grid<T, D, SW, true, true>), all_tiles, dim3(64), 0, st, a, lanes, n_nb);
  TESS_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_save_list, dim3(unsigned(std::min<int64_t>(blocks_for(int64_t(ntiles), 256), 1024))), dim3(256),
                     0, st, nblist, n_nb, prev_list, prev_count);
  TESS_HIP(hipGetLastError());
  // G2P over the active tiles (with the next keys and each tile's counts and
  // leavers), then the particles outside every mesh
  const uint32_t nt32 = uint32_t(ntiles);
  const int nw = (B.variant & 4) ? 1 : (B.variant & 2) ? 2 : 4;
  auto g2p = [&](auto nwc) {
    constexpr int NW = decltype(nwc)::value;
    if (persist)
      hipLaunchKernelGGL((k_g2p_fast_persist<T, D, BASIS, true, NW, true>), dim3(B.grid_g2p), dim3(64 * NW), 0, st, a,
                         sk, mo, nt32, n_active);
    else
      hipLaunchKernelGGL((k_g2p_fast_grid<T, D, BASIS, true, NW, true>), all_tiles, dim3(64 * NW), 0, st, a, sk, mo,
                         nt32, n_active);
  };
  if (nw == 1) g2p(std::integral_constant<int, 1>{});
  else if (nw == 2) g2p(std::integral_constant<int, 2>{});
  else g2p(std::integral_constant<int, 4>{});
  TESS_HIP(hipGetLastError());
  if (n > 0) {
    hipLaunchKernelGGL((k_g2p_outside_persist<T, D>), dim3(B.grid_out), dim3(256), 0, st, a, sk, mo.nk,
                       static_cast<const uint32_t*>(counters + CNT_INSIDE));
    TESS_HIP(hipGetLastError());
  }
}

void graph_release(tess_batch& B) {
  for (int p = 0; p < 2; ++p) {
    if (B.graph_exec[p]) (void)hipGraphExecDestroy(B.graph_exec[p]);
    if (B.graph[p]) (void)hipGraphDestroy(B.graph[p]);
    B.graph_exec[p] = nullptr;
    B.graph[p] = nullptr;
  }
  B.captured_variant = -1;
  B.graph_deps.clear();
}

// Every buffer a captured step points at, with its address at the capture.
std::vector<std::pair<const Buffer*, void*>> graph_buffers(tess_ctx* g, tess_batch& B) {
  const Buffer* bufs[] = {&g->counters,   &g->lanes,      &g->keys,        &g->keys_sorted, &g->vals,
                          &g->skeys2,     &g->perm2,      &g->keys_alt,    &g->vals_alt,    &g->hist,
                          &g->scan_tmp,   &g->inc_nk,     &g->tile_stay,   &g->tile_tin,    &g->inc_out,
                          &g->inc_seg,    &g->inc_seg2,   &g->tab_sums,    &g->tile_seg,    &g->tile_start,
                          &g->tile_end,   &g->tile_flag,  &g->tile_slot,   &g->active_tiles, &g->nb_flag,
                          &g->nb_list,    &g->alt_start,  &g->alt_end,     &g->alt_flag,    &g->alt_slot,
                          &g->alt_active, &g->alt_nb_flag, &g->alt_nb_list, &g->partials,   &B.g_prev_list,
                          &B.g_prev_count, &B.recs,       &B.d_toff,       &B.d_poff,       &B.d_nt,
                          &B.d_tscene};
  std::vector<std::pair<const Buffer*, void*>> v;
  for (const Buffer* b : bufs) v.emplace_back(b, b->ptr);
  return v;
}

bool graph_deps_hold(const tess_batch& B) {
  for (const auto& d : B.graph_deps)
    if (d.first->ptr != d.second) return false;
  return !B.graph_deps.empty();
}

// The reorder test between replays, on the binning the last step left in set
// `cur` (its counts read back), exactly as an eager step would run it.
template <typename T, int D>
void graph_reorder_check(tess_ctx* g, tess_batch& B, int cur) {
  uint32_t* hc = reinterpret_cast<uint32_t*>(g->counters_host);
  TESS_HIP(hipMemcpyAsync(hc, g->counters.as<uint32_t>(CNT_SLOTS), CNT_SLOTS * sizeof(uint32_t),
                          hipMemcpyDeviceToHost, g->stream));
  TESS_HIP(hipStreamSynchronize(g->stream));
  Binning& b = g->bin;
  b.n = B.ntot;
  b.ntiles = B.tiles_total;
  b.n_inside = B.ntot > 0 ? int64_t(hc[CNT_INSIDE]) : 0;
  b.n_active = int64_t(hc[CNT_ACTIVE]);
  b.n_nodeblocks = int64_t(hc[CNT_NB]);
  b.valid = true;
  if (cur == 1) {
    std::swap(g->keys_sorted, g->skeys2);
    std::swap(g->vals, g->perm2);
    swap_tables(g);
  }
  B.counted = false;
  try {
    batch_reorder<T, D>(g, B, B.reorder_threshold);
  } catch (...) {
    if (cur == 1) {
      std::swap(g->keys_sorted, g->skeys2);
      std::swap(g->vals, g->perm2);
      swap_tables(g);
    }
    throw;
  }
  if (cur == 1) {
    std::swap(g->keys_sorted, g->skeys2);
    std::swap(g->vals, g->perm2);
    swap_tables(g);
  }
  b.valid = false;
}

template <typename T, int D, int BASIS>
void batch_graph_run(tess_ctx* ctx, tess_batch& B, int nsteps) {
  if (nsteps <= 0) return;
  for (auto& e : B.graph_ev)
    if (!e) {
      hipEvent_t ev = nullptr;
      const hipError_t err = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      if (err == hipSuccess) e = ev;  // kept before any error is raised
      TESS_HIP(err);
    }
  if (!B.gctx) {
    hipStream_t gs = nullptr;
    const hipError_t err = hipStreamCreateWithFlags(&gs, hipStreamNonBlocking);
    try {
      TESS_HIP(err);
      B.gctx = ctx_new(ctx->device, gs);
    } catch (...) {
      if (gs) (void)hipStreamDestroy(gs);
      throw;
    }
  }
  tess_ctx* g = B.gctx;
  hipStream_t gs = g->stream;
  // the caller's work on its stream comes first
  TESS_HIP(hipEventRecord(B.graph_ev[0], ctx->stream));
  TESS_HIP(hipStreamWaitEvent(gs, B.graph_ev[0], 0));
  uint32_t* prev_count = B.g_prev_count.as<uint32_t>(64);
  B.g_prev_list.as<uint32_t>(size_t(std::max<int64_t>(B.tiles_total, 1)));
  if (!B.last_graph) {
    // eager steps wrote node blocks this mode's stale list does not name
    Args<T, D> a = batch_args<T, D>(g, B);
    hipLaunchKernelGGL((k_zero_grid_batch<T, D>), dim3(blocks_for(B.max_nodes, 256), unsigned(B.nscenes)), dim3(256),
                       0, gs, a);
    TESS_HIP(hipGetLastError());
    fill_u32(gs, prev_count, 1, 0u);
    B.last_graph = true;
  }
  if (B.captured_variant != B.variant) graph_release(B);
  batch_graph_grids<T, D, BASIS>(g, B);
  // each call starts with an ordinary step whose binning sorts every particle
  // (the positions may have changed since the last call); it leaves set 0
  batch_graph_step<T, D, BASIS>(g, B, true, 0);
  int done = 1, cur = 0, since_test = 0;
  while (done < nsteps) {
    if (!graph_deps_hold(B)) {
      // first use, another variant, or a buffer moved: capture both parities
      // (capturing launches nothing)
      graph_release(B);
      TESS_HIP(hipStreamSynchronize(gs));
      for (int p = 0; p < 2; ++p) {
        TESS_HIP_EXACT(hipStreamBeginCapture(gs, hipStreamCaptureModeRelaxed));
        try {
          batch_graph_step<T, D, BASIS>(g, B, false, p);
        } catch (...) {
          hipGraph_t dead = nullptr;
          (void)hipStreamEndCapture(gs, &dead);
          if (dead) (void)hipGraphDestroy(dead);
          graph_release(B);
          throw;
        }
        TESS_HIP_EXACT(hipStreamEndCapture(gs, &B.graph[p]));
        TESS_HIP(hipGraphInstantiate(&B.graph_exec[p], B.graph[p], nullptr, nullptr, 0));
      }
      B.graph_deps = graph_buffers(g, B);
      B.captured_variant = B.variant;
      B.captures += 1;
    }
    if (B.reorder_threshold > 0.0 && B.ntot > 0 && since_test == 0) {
      graph_reorder_check<T, D>(g, B, cur);
      if (!graph_deps_hold(B)) {
        // the test moved a buffer the graphs use: start over from the positions
        batch_graph_step<T, D, BASIS>(g, B, true, 0);
        ++done;
        cur = 0;
        continue;
      }
    }
    TESS_HIP(hipGraphLaunch(B.graph_exec[cur], gs));
    cur = 1 - cur;
    ++done;
    B.graph_replays += 1;
    since_test = (since_test + 1) % std::max(B.graph_chunk, 1);
  }
  TESS_HIP(hipEventRecord(B.graph_ev[1], gs));
  TESS_HIP(hipStreamWaitEvent(ctx->stream, B.graph_ev[1], 0));
  // the error flags of the call's binnings (one readback per call)
  uint32_t* hc = reinterpret_cast<uint32_t*>(g->counters_host);
  TESS_HIP(hipMemcpyAsync(hc, g->counters.as<uint32_t>(CNT_SLOTS), CNT_SLOTS * sizeof(uint32_t),
                          hipMemcpyDeviceToHost, gs));
  TESS_HIP(hipStreamSynchronize(gs));
  if (hc[CNT_ERR] & ERR_GIMP_LENGTH) raise(TESS_ERR_ARGUMENT, "uGIMP requires 0 ≤ pt.l ≤ spacing(mesh)");
  if (TESS_DEBUG && B.ntot > 0) {
    // the last step's binning, in set `cur` (the graphs' merges checked through it)
    const BinSet last = bin_set(g, B.ntot, B.tiles_total, cur);
    debug_check_binning(gs, last.keys, last.perm, last.start, last.end, last.active, B.ntot, B.tiles_total,
                        int64_t(hc[CNT_ACTIVE]), int64_t(hc[CNT_INSIDE]), "batch graph step");
  }
  // the eager path's binning and zeroing bookkeeping no longer hold
  B.keys_ready = false;
  B.binned = false;
  B.counted = false;
  g->bin.valid = false;
  ctx->bin.valid = false;
}

template <typename T, int D, int B_, bool S>
struct BatchStepOp {
  static void run(tess_ctx* ctx, const tess_mesh&, tess_batch& b, int nsteps) {
    if constexpr (S) raise(TESS_ERR_UNSUPPORTED, "batches evaluate the basis inside the transfers");
    else if (b.variant & 8) {
      try {
        batch_graph_run<T, D, B_>(ctx, b, nsteps);
      } catch (...) {
        // a failed call leaves nothing of its own running on the batch's
        // stream: the caller may reuse the scene arrays at once
        if (b.gctx) (void)hipStreamSynchronize(b.gctx->stream);
        throw;
      }
    }
    else batch_step_impl<T, D, B_>(ctx, b, nsteps);
  }
};
template <typename T, int D, int B_, bool S>
struct BatchCreateOp {
  static void run(tess_ctx* ctx, const tess_mesh&, tess_batch& b) {
    if constexpr (!S) batch_create_impl<T, D>(ctx, b);
  }
};

}  // namespace

namespace TESS_PART {

void batch_create(tess_ctx* ctx, int basis, const tess_mesh& mesh, tess_batch& b) {
  dispatch<BatchCreateOp>(basis, mesh, false, ctx, mesh, b);
}

void batch_step(tess_ctx* ctx, int basis, const tess_mesh& mesh, tess_batch& b, int nsteps) {
  dispatch<BatchStepOp>(basis, mesh, false, ctx, mesh, b, nsteps);
}

}  // namespace TESS_PART
}  // namespace tess

#else

#include <algorithm>

#include "tess_internal.hpp"

namespace tess {
namespace {

// frees the graphs (and with them every pointer they recorded)
void graph_release(tess_batch& B) {
  for (int p = 0; p < 2; ++p) {
    if (B.graph_exec[p]) (void)hipGraphExecDestroy(B.graph_exec[p]);
    if (B.graph[p]) (void)hipGraphDestroy(B.graph[p]);
    B.graph_exec[p] = nullptr;
    B.graph[p] = nullptr;
  }
  B.captured_variant = -1;
  B.graph_deps.clear();
}

void forward_create(tess_ctx* ctx, int basis, const tess_mesh& mesh, tess_batch& b) {
  TESS_FORWARD(mesh, batch_create(ctx, basis, mesh, b));
}
void forward_step(tess_ctx* ctx, int basis, const tess_mesh& mesh, tess_batch& b, int nsteps) {
  TESS_FORWARD(mesh, batch_step(ctx, basis, mesh, b, nsteps));
}

bool julia_fields(const tess_scene& sc, int D) {
  auto pok = [](const tess_field& f, int nc) { return !f.ptr || (f.comp_stride == 1 && f.elem_stride == nc); };
  const tess_particles& P = sc.particles;
  const tess_grid& G = sc.grid;
  return pok(P.x, D) && pok(P.v, D) && pok(P.V, 1) && pok(P.grad_v, D * D) && pok(P.F, D * D) &&
         pok(P.sigma, D * D) && pok(P.l, 1) && pok(P.logE, 1) && pok(G.m, 1) && pok(G.mv, D) && pok(G.f, D) &&
         pok(G.vn, D) && pok(G.v, D);
}

}  // namespace

void run_batch_create(tess_ctx* ctx, int basis, int nscenes, const tess_scene* scenes, tess_batch** out) {
  auto* b = new tess_batch();
  b->seen_epoch = error_epoch();
  try {
    b->basis = basis;
    b->nscenes = nscenes;
    b->dim = scenes[0].mesh.dim;
    b->dtype = scenes[0].mesh.dtype;
    b->scenes.assign(scenes, scenes + nscenes);
    b->toff.assign(size_t(nscenes) + 1, 0);
    b->poff.assign(size_t(nscenes) + 1, 0);
    const int LT = b->dim == 3 ? 2 : 3;  // log2 cells per tile axis (Geo)
    for (int s = 0; s < nscenes; ++s) {
      const tess_scene& sc = scenes[s];
      if (sc.mesh.dim != b->dim || sc.mesh.dtype != b->dtype)
        raise(TESS_ERR_ARGUMENT, "all scenes of a batch share the mesh dimension and dtype");
      if (!julia_fields(sc, b->dim))
        raise(TESS_ERR_UNSUPPORTED, "batched scenes use the Julia-native field layout");
      int64_t nt = 1, nn = 1;
      for (int d = 0; d < b->dim; ++d) {
        nt *= ((sc.mesh.dims[d] - 1) >> LT) + 1;
        nn *= sc.mesh.dims[d];
      }
      b->toff[size_t(s) + 1] = b->toff[size_t(s)] + nt;
      b->poff[size_t(s) + 1] = b->poff[size_t(s)] + sc.particles.n;
      b->max_nodes = std::max(b->max_nodes, nn);
    }
    b->ntot = b->poff.back();
    b->tiles_total = b->toff.back();
    if (uint64_t(b->tiles_total) * 64 >= uint64_t(UINT32_MAX) || b->ntot >= int64_t(UINT32_MAX))
      raise(TESS_ERR_ARGUMENT, "the batch exceeds the 32-bit binning range");
    forward_create(ctx, basis, scenes[0].mesh, *b);
  } catch (...) {
    b->recs.release();
    b->d_toff.release();
    b->d_poff.release();
    b->d_nt.release();
    b->d_tscene.release();
    delete b;
    throw;
  }
  *out = b;
}

void run_batch_step(tess_ctx* ctx, tess_batch* b, int nsteps) {
  const uint64_t ep = error_epoch();
  if (b->seen_epoch != ep) {
    // a call failed since this batch's last step: its binning, zeroing lists
    // and graph-mode device state may describe work cut short, so the next
    // step zeroes every grid and bins from scratch in either mode
    if (b->gctx) {
      (void)hipStreamSynchronize(b->gctx->stream);
      b->gctx->bin.valid = false;
      b->gctx->bin.state_valid = false;
    }
    b->zeroed = false;
    b->binned = false;
    b->keys_ready = false;
    b->counted = false;
    b->last_graph = false;
    b->seen_epoch = ep;
  }
  forward_step(ctx, b->basis, b->scenes[0].mesh, *b, nsteps);
}

void run_batch_set_variant(tess_batch* b, int variant) { b->variant = variant; }

void run_batch_set_reorder(tess_batch* b, double threshold) { b->reorder_threshold = threshold; }
int run_batch_variant(const tess_batch* b) { return b->variant; }

void run_batch_stats(const tess_batch* b, int64_t* out, int n) {
  const int64_t vals[6] = {b->reorders, b->reorders_by_count, b->kept_binnings, b->variant, b->graph_replays,
                           b->captures};
  for (int k = 0; k < n && k < 6; ++k) out[k] = vals[k];
}

void run_batch_destroy(tess_batch* b) {
  if (b->gctx) {
    hipStream_t gs = b->gctx->stream;
    graph_release(*b);
    ctx_free(b->gctx);  // synchronises its stream
    if (gs) (void)hipStreamDestroy(gs);
    b->gctx = nullptr;
  }
  for (hipEvent_t e : b->graph_ev)
    if (e) (void)hipEventDestroy(e);
  b->g_prev_list.release();
  b->g_prev_count.release();
  b->recs.release();
  b->d_toff.release();
  b->d_poff.release();
  b->d_nt.release();
  b->d_tscene.release();
  b->prev_list.release();
  delete b;
}

}  // namespace tess

#endif
