// Host-side internals of libtesserae_hip: the context (stream + scratch owned by
// the library), error reporting across the C ABI, and the launchers each
// kernel file provides.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <utility>
#include <vector>

#include "../../include/tesserae_hip.h"

namespace tess {

// Error raised inside the library; converted to a tess_status + message at the
// C boundary (nothing propagates across it).
struct Error {
  tess_status code;
  std::string msg;
};

[[noreturn]] void raise(tess_status code, const std::string& msg);
void check_hip(hipError_t e, const char* what);
#define TESS_HIP(call) ::tess::check_hip((call), #call)
// the same check, never subject to failure injection (stream-capture control)
void check_hip_exact(hipError_t e, const char* what);
#define TESS_HIP_EXACT(call) ::tess::check_hip_exact((call), #call)
// incremented by every C-ABI call that fails (see check_ctx)
uint64_t error_epoch();

// A device buffer owned by the context; grows on demand, never shrinks.
struct Buffer {
  void* ptr = nullptr;
  size_t bytes = 0;
  void* get(size_t need);  // (re)allocates when need > bytes; contents undefined
  bool fits(size_t need);  // get, but false where the device has no memory for it
  void release();
  template <typename U>
  U* as(size_t count) { return static_cast<U*>(get(count * sizeof(U))); }
};

// Binning of one particle set into the P2G/G2P tiles, valid until the
// particles move.  All arrays live in ctx scratch.
struct Binning {
  bool valid = false;
  const void* x_ptr = nullptr;  // identity of the particle set it was built for
  int64_t n = 0;
  int32_t dim = 0, dtype = 0, basis = 0;
  int32_t tile_log2 = 0;
  int64_t ntiles_axis[3] = {1, 1, 1};
  int64_t ntiles = 0;
  int64_t n_inside = 0;     // particles with a non-empty window (host copy)
  int64_t n_active = 0;     // tiles holding >= 1 particle (host copy)
  int64_t n_nodeblocks = 0; // node blocks touched by some tile footprint (host copy)
  bool crowded = false;     // some tile holds more than merge_tile_max particles
  // the sorted (key, perm) arrays are a valid previous order for incremental re-binning
  bool state_valid = false;
  int64_t state_n = -1, state_ntiles = -1;
  int32_t state_dim = 0;
  // the last G2P wrote the next keys at the sorted positions and the counts
  // and leavers of every tile
  bool keys_ready = false;
};

// Per-kernel timing with HIP events on the context's stream.  Disabled by
// default; begin/end cost two event records per profiled launch when enabled.
struct ProfEntry {
  std::string name;
  double total_ms = 0.0;
  int64_t calls = 0;
  double bytes = 0.0;  // algorithmic bytes summed over the calls
};
struct Profiler {
  bool on = false;
  std::vector<ProfEntry> entries;
  std::vector<hipEvent_t> pool;
  struct Pending {
    int entry;
    hipEvent_t a, b;
  };
  std::vector<Pending> pending;
  size_t next_event = 0;
};

// The last tess_rollout of a context: checkpoints of (x, v, F, V, σ) every
// `every` steps, replayed segment by segment by the adjoint.
struct Rollout {
  bool valid = false;
  int nsteps = 0, every = 1;
  int64_t n = 0;
  int32_t dim = 0, dtype = 0, basis = 0;
  int64_t dims[3] = {0, 0, 0};
  tess_field logE{nullptr, 0, 0};
  // the last segment's states, binnings and grids as the rollout ran it, in
  // the pullback's slots (so the pullback need not replay that segment), and
  // the buffers they were written to
  bool last_kept = false;
  std::vector<Binning> last_bins;
  const void* last_seg = nullptr;
  const void* last_snaps = nullptr;
};

}  // namespace tess

namespace tess {

// device counters (words of tess_ctx::counters, reported to the same words of
// counters_host): totals of a binning, error flags, and sums over the lanes
enum {
  CNT_INSIDE = 0, CNT_ACTIVE = 1, CNT_NB = 2, CNT_ERR = 3,
  CNT_MISPLACED = 8, CNT_NODES = 9, CNT_ARRIVE = 10, CNT_P2GERR = 11, CNT_MOVED = 12, CNT_OUTIN = 13, CNT_RESORT = 14,
  CNT_PREV_ACTIVE = 15, CNT_SLOTS = 16,
  CNT_RESORTED = 16,   // device: CNT_RESORT of the last report
  CNT_MANY = 22,       // device: the last report's arrivals are too many to merge
  CNT_SCATTERED = 23,  // device: waves of k_rekey nearly all of whose particles left their tiles
  CNT_KEEP = 21,       // device: the tables being scanned are not wanted
  CNT_SEQ = 17         // host: the report's number, once by each of its REPORTERS
};
constexpr int REPORTERS = 4;
// Kernels count into lanes, one per 128-byte line, chosen by workgroup (no
// single contended address): particles whose key changed, layered neighbour
// pairs not consecutive in storage, nodes with m > 0.
enum { LANE_MOVED = 0, LANE_BROKEN = 1, LANE_NODES = 2, LANE_GROUPS = 3 };
constexpr int LANES = 32, LANE_STRIDE = 32;
constexpr size_t LANE_BYTES = size_t(LANE_GROUPS) * LANES * LANE_STRIDE * sizeof(uint32_t);

// What a kernel that computes next keys writes (see binning.hip): the keys at
// the sorted positions (nullptr: nothing is written), per tile the particles
// that stay and the arrivals, and the leavers of each tile from its run's start.
struct MoveOut {
  uint32_t* nk;
  uint32_t* stay;
  uint32_t* tin;
  uint2* out;
  uint32_t* lanes;
};

// Why a re-binning sorts every key instead of merging the changed ones (bits of
// CNT_RESORT): the per-tile counts are not complete (particles came back into the
// mesh, or nearly all were put elsewhere) and the tables wait for a count of the
// sorted keys; one tile has more arrivals, or holds more particles, than its
// workgroup should take alone.
enum { RESORT_RECOUNT = 1, RESORT_CROWD = 2, RESORT_TILE = 4 };

// The tile tables of a binning, from the per-tile counts (binning.hip).
struct TabArgs {
  uint32_t* stay;  // ntiles + 1: particles that stay, the last entry those outside the mesh
  uint32_t* tin;   // ntiles + 1: arrivals (reset)
  int64_t ntiles;
  int32_t nt[3];
  const int64_t* scene_toff;  // a batch: first tile and tiles per axis of each scene, scene of each tile
  const int32_t* scene_nt;
  const uint32_t* tile_scene;
  uint32_t* sums;  // 4 words per workgroup
  uint32_t *start, *end, *flag, *slot, *active, *nb_flag, *nb_list, *seg;
  uint32_t* lanes;
  uint32_t* counters;
  uint32_t* host;
  uint32_t seq;  // the report's number (0: nobody waits for it by number)
  int32_t keep_err;
  int32_t may_keep;  // with no changed key the old tables stand: build none (CNT_KEEP)
  uint32_t crowd;    // more arrivals in one tile than this ask for a sort (RESORT_CROWD),
  uint32_t many;     // and more in all (CNT_MANY)
  uint32_t tile_max; // and more particles in one tile (RESORT_TILE)
};

// The merge of the particles whose key changed into the previous order.
struct MergeArgs {
  int64_t n, ntiles;
  const uint32_t *old_active, *old_start, *old_end, *new_active, *new_start, *new_end;
  const uint32_t* old_count;  // device counts for launches sized by an upper bound, or nullptr
  const uint32_t* new_count;
  int64_t old_active_n, new_active_n;
  int64_t first_tile;  // of new_active, for the launch's first workgroup
  const uint32_t* stay;
  const uint32_t* nk;
  const uint32_t* perm_old;
  const uint32_t* seg_off;
  const uint2* out;
  uint2 *seg, *seg_alt;
  uint32_t *keys_new, *perm_new;
  const uint32_t* counters;  // device count of arrivals outside the mesh, or nullptr: out_in
  const uint32_t* gate;      // device counters: do nothing where they call for no merge, or nullptr
  uint32_t out_in;
  uint32_t crowd;  // more arrivals outside the mesh than this are placed by several workgroups
  int32_t pos_bits;
};

}  // namespace tess

struct tess_ctx {
  tess::Profiler prof;
  int device = 0;
  hipStream_t stream = nullptr;
  // sort + binning: keys (unsorted), keys_sorted + vals (= perm) sorted output,
  // *_alt ping-pong buffers of the radix sort
  tess::Buffer keys, keys_sorted, vals, keys_alt, vals_alt, hist, scan_tmp;
  tess::Buffer tile_start, tile_end, tile_flag, tile_slot, active_tiles;
  tess::Buffer nb_flag, nb_list, nb_list_prev;
  // the tables being built while the ones above are in use
  tess::Buffer alt_start, alt_end, alt_flag, alt_slot, alt_active, alt_nb_flag, alt_nb_list;
  tess::Buffer tab_sums, tile_seg;
  tess::Buffer partials;
  tess::Buffer per_tile;  // per-workgroup counts of the partition's contiguity score
  // re-binning scratch: the other half of (keys_sorted, vals), next keys,
  // per-tile counts, leavers, arrival segments
  tess::Buffer skeys2, perm2, inc_nk, tile_stay, tile_tin, inc_out, inc_seg, inc_seg2;
  tess::Buffer inc_pout, inc_rank;  // a batch reorder's new indices and ranks
  int64_t last_movers = -1;
  int64_t kept_binnings = 0;  // binnings that kept the previous layout (no particle changed its key)
  tess::Buffer counters;   // small device scalars
  tess::Buffer moved;      // the second set of particle arrays of a loop whose reorders ride on G2P
  tess::Buffer g2p2g_x;    // positions before a G2P2G pass (its P2G half's weights)
  tess::Buffer export_buf; // Float32 staging of tess_export_field
  // corrected basis of the current call (TESS_WLS / TESS_KERNEL_CORRECTION /
  // TESS_POLY_MULTILINEAR bits, 0 for a plain kernel) and its node filter
  int32_t corr = 0;
  const uint8_t* corr_filter = nullptr;
  tess::Buffer lanes;      // counts spread over cache lines (LANE_GROUPS groups of LANES)
  tess::Buffer host_pinned_dummy;
  uint32_t report_seq = 0;           // number of the last report asked for by number
  int64_t* counters_host = nullptr;  // pinned readback slots
  tess::Binning bin;
  // zeroing bookkeeping for the grid of the previous P2G
  const void* last_grid_m = nullptr;
  int64_t prev_nodeblocks = 0;
  // where the node-block list of the last P2G is: in the current tables, in the
  // alternate set they were swapped with, or copied out before that set was
  // built again
  enum class PrevList { Current, Alternate, Copied } prev_list = PrevList::Copied;
  int32_t prev_tile_log2 = -1;
  int64_t prev_dims[3] = {-1, -1, -1};
  // reorder scratch and the layout score of the last step's P2G
  tess::Buffer reorder_tmp, reorder_cnt;
  const void* misplaced_x_ptr = nullptr;
  int64_t misplaced_n = 0;
  int64_t misplaced_pairs = 0;  // layered neighbour pairs of that P2G's binning
  int64_t last_misplaced = -1;  // of them, pairs not consecutive in storage
  int64_t reorders = 0;
  // a P2G has counted broken pairs (nodes) since the last report of the lanes
  bool broken_pending = false, nodes_pending = false;
  int64_t broken_count = 0;
  // nodes with m > 0 written by the last gather (read back with the next binning)
  int64_t last_active_nodes = -1;
  // SpGrid block activation scratch: occupied flags (all clear between updates
  // of sp_clean blocks), active flags, per-workgroup counts
  tess::Buffer sp_occ, sp_act, sp_sums;
  int64_t sp_clean = -1;
  // adjoint: per-tile Float64 partials, node adjoints, rollout checkpoints and replay
  tess::Buffer adj_partials, adj_nodes, ro_checkpoints, ro_segment, ro_gradv, ro_snapshots;
  tess::Rollout rollout;
  // the pullback replays segments on a second context (own stream and
  // scratch, private grid ro_grid) while this context reverses the previous one
  tess_ctx* replay = nullptr;
  tess::Buffer ro_grid;
  // the failure epoch this context's caches belong to
  uint64_t seen_epoch = 0;
};

namespace tess {
// A context's state without the C-ABI checks (tess_ctx_create/destroy use them).
tess_ctx* ctx_new(int device, hipStream_t stream);
void ctx_free(tess_ctx* ctx);
}  // namespace tess

// A batch of scenes (batch.hip): the scenes as given, where each scene's tiles
// and particles start in the batch-wide index spaces, and the device copies.
struct tess_batch {
  int32_t basis = 0, dim = 0, dtype = 0, nscenes = 0;
  int64_t ntot = 0, tiles_total = 0, max_nodes = 0;
  std::vector<tess_scene> scenes;
  std::vector<int64_t> toff, poff;
  tess::Buffer recs, d_toff, d_poff, d_nt, d_tscene, prev_list;
  int64_t prev_nb = 0;
  bool zeroed = false;
  // the binning in the context is this batch's, and the last G2P wrote every
  // particle's next key (stepping within one call)
  bool binned = false, keys_ready = false;
  int64_t kept_binnings = 0;
  // bit 0: P2G one wave per last-axis offset (2D); G2P waves per tile: 4, 2 with bit 1, 1 with bit 2
  int variant = 0;
  // layered reorder of the scenes' particles when the contiguity score falls
  // below the threshold (0: never, 1: every step); reorders done so far
  double reorder_threshold = 0.0;
  int64_t reorders = 0;
  // of those, reorders decided from the broken-pair count of the previous step's P2G
  int64_t reorders_by_count = 0;
  // the last P2G of this call counted the broken layered pairs (the sum sits in
  // the counters), over this many pairs
  bool counted = false;
  int64_t counted_pairs = 0;
  // graph mode (variant bit 3): a private context on its own stream steps the
  // batch as replays of captured hipGraphs, one per parity of the binning's
  // double buffer (graph[p] reads binning set p and writes set 1-p); the
  // previous step's node-block list and count live on the device, and the
  // buffers the graphs point at are recorded to detect a reallocation
  tess_ctx* gctx = nullptr;
  hipGraph_t graph[2] = {nullptr, nullptr};
  hipGraphExec_t graph_exec[2] = {nullptr, nullptr};
  hipEvent_t graph_ev[2] = {nullptr, nullptr};
  int captured_variant = -1;
  std::vector<std::pair<const tess::Buffer*, void*>> graph_deps;
  tess::Buffer g_prev_list, g_prev_count;
  unsigned grid_p2g = 0, grid_g2p = 0, grid_gather = 0, grid_zero = 0, grid_out = 0;
  // the grids were last written by graph-mode steps (the eager bookkeeping does not know them)
  bool last_graph = false;
  // replays between two reorder tests (each test bins on the host side)
  int graph_chunk = 16;
  int64_t graph_replays = 0, captures = 0;
  // the failure epoch the batch's caches belong to
  uint64_t seen_epoch = 0;
};

namespace tess {

// ---- scans and sorts (sort.hip) ----
// Plain copy of bytes (a multiple of 16) on the context's stream.
void run_device_copy(tess_ctx* ctx, const void* src, void* dst, int64_t bytes);
// Exclusive prefix sum of n uint32 values in place; returns nothing, total is
// written to *total_dev (device) when non-null.
void exclusive_scan_u32(tess_ctx* ctx, uint32_t* data, int64_t n, uint32_t* total_dev);
// *out (device) = sum of v[0..n), one workgroup (for per-workgroup counts).
void sum_u32(tess_ctx* ctx, const uint32_t* v, int64_t n, uint32_t* out);
// Stable LSD radix sort of (key, value) pairs on the low key_bits of key.
// vals_in == nullptr means values 0..n-1.  Result lands in (keys_out, vals_out).
void radix_sort_pairs(tess_ctx* ctx, const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                      uint32_t* vals_out, int64_t n, int key_bits);
// The same sort over caller-provided work buffers on a stream (no allocation):
// hist holds sort_hist_words(n) words, keys_alt/vals_alt n words each.
struct SortWork {
  hipStream_t stream = nullptr;
  uint32_t* hist = nullptr;
  uint32_t* keys_alt = nullptr;
  uint32_t* vals_alt = nullptr;
};
size_t sort_hist_words(int64_t n);
size_t scan_work_bytes(int64_t n);
void radix_sort_pairs_ws(const SortWork& w, const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                         uint32_t* vals_out, int64_t n, int key_bits);

// ---- tile tables and the merge between two steps (binning.hip) ----
int64_t tab_blocks(int64_t ntiles);
void launch_tables(hipStream_t st, const TabArgs& a);
void launch_tile_counts(hipStream_t st, const uint32_t* skeys, int64_t n, int64_t ntiles, uint32_t* stay, uint32_t* tin);
void launch_merge(hipStream_t st, const MergeArgs& a, unsigned outside_blocks);
void launch_merge_tiles(hipStream_t st, const MergeArgs& a, int64_t tiles);
void launch_merge_outside(hipStream_t st, const MergeArgs& a, unsigned blocks);

// ---- reference-layout weights and partition (partition.hip) ----
void launch_update_weights(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_particles& P,
                           const tess_weights& W);
void run_partition_update(tess_ctx* ctx, const tess_mesh& mesh, tess_field x, int64_t n, int32_t* pidx,
                          int32_t* starts, int32_t* stops, int64_t* nassigned);
// The partition over the library's fixed device work area (no allocation);
// *nassigned is device memory.  Raises TESS_ERR_ARGUMENT beyond
// partition_noalloc_max_particles().
void run_partition_update_noalloc(const tess_mesh& mesh, tess_field x, int64_t n, int32_t* pidx, int32_t* starts,
                                  int32_t* stops, int64_t* nassigned, hipStream_t stream);
int64_t partition_noalloc_max_particles();
// Resolves the work area's address on the current device (once per device).
void noalloc_scratch_resolve();
void run_reorder(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P, int32_t* pidx,
                 int64_t nassigned, double threshold, int32_t* reordered);

// ---- SpGrid block numbering (sparse.hip) ----
// update_sparsity!(spinds, xₚ, mesh): writes sp.blocknumbering and
// sp.storage_len, *changed (host, optional) = active set changed.  Synchronises;
// with defer it only enqueues, and the caller takes the totals (take_sparsity)
// after a synchronisation of its own.
void run_sparsity_update(tess_ctx* ctx, const tess_mesh& mesh, tess_field x, int64_t n, tess_sparsity& sp,
                         int32_t* changed, bool defer = false);
void take_sparsity(tess_ctx* ctx, const tess_mesh& mesh, tess_sparsity& sp, int32_t* changed);

// ---- transfers (transfer.hip) ----
void run_p2g(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
             const tess_weights* W, const tess_params& prm);
void run_g2p(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
             const tess_weights* W, const tess_params& prm);
void run_g2p2g(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
               const tess_weights* W, const tess_params& prm);
void run_g2p2g_steps(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                     const tess_params& prm, int nsteps, double reorder_threshold);
void run_step(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
              const tess_params& prm, int nsteps, double reorder_threshold);
// The same on an SpGrid: grid fields are SpArray data vectors addressed through sp.
void run_p2g_sparse(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_sparsity& sp,
                    const tess_particles& P, const tess_weights* W, const tess_params& prm);
void run_g2p_sparse(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_sparsity& sp,
                    const tess_particles& P, const tess_weights* W, const tess_params& prm);
// *done: steps run before a TESS_ERR_STATE (storage too small), nsteps on success.
void run_step_sparse(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, tess_sparsity& sp,
                     const tess_particles& P, const tess_params& prm, int nsteps, double reorder_threshold,
                     int* done);
// ---- adjoint (adjoint.hip) ----
void run_step_adjoint(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                      const tess_params& prm, const tess_adjoint& adj);
void run_rollout(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,
                 const tess_params& prm, int nsteps, int every);
void run_rollout_adjoint(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G,
                         const tess_params& prm, const tess_adjoint& adj);
// ---- batches (batch.hip) ----
void run_export_field(tess_ctx* ctx, int32_t dtype, int32_t dim, tess_field field, int64_t n, int32_t kind,
                      float* dst);
void run_vtk_write_points(const char* path, int64_t n, const float* xyz, int32_t narrays,
                          const tess_vtk_array* arrays, int32_t compress);
void run_vtk_write_mesh(const char* path, const tess_mesh& mesh, int32_t narrays, const tess_vtk_array* arrays,
                        int32_t compress);
void run_vtm_write(const char* path, int32_t nblocks, const char* const* files);
void run_pvd_write(const char* path, int32_t n, const double* times, const char* const* files);
void run_ply_write(const char* name, int64_t n, const float* xyz);
void run_batch_create(tess_ctx* ctx, int basis, int nscenes, const tess_scene* scenes, tess_batch** out);
void run_batch_step(tess_ctx* ctx, tess_batch* b, int nsteps);
void run_batch_set_variant(tess_batch* b, int variant);
void run_batch_set_reorder(tess_batch* b, double threshold);
int run_batch_variant(const tess_batch* b);
// out[0..n): reorders, reorders decided from the previous P2G's count, kept binnings, variant
void run_batch_stats(const tess_batch* b, int64_t* out, int n);
void run_batch_destroy(tess_batch* b);
// Moves every particle field so that slot k receives particle order[k].
void permute_particles(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P, const uint32_t* order);
// The same for l and log E, which G2P does not write.
void permute_constants(tess_ctx* ctx, const tess_mesh& mesh, const tess_particles& P, const uint32_t* order);
// Copies of n <= 6 arrays in one launch (sizes in bytes, multiples of 4).
void copy_arrays(hipStream_t st, const void* const* src, void* const* dst, const int64_t* bytes, int n);

// ---- scalar type and dimension parts ------------------------------------------
// The templated files (transfer, batch, adjoint) are compiled once per (scalar
// type, dimension), in parallel: each part's functions live in the namespace
// named TESS_PART, and the same file compiled without it forwards to them.
#define TESS_PART_DECLARE(NS)                                                                                        \
  namespace NS {                                                                                                     \
  void p2g(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,             \
           const tess_weights* W, const tess_params& prm, const tess_sparsity* sp);                                  \
  void g2p(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,             \
           const tess_weights* W, const tess_params& prm, const tess_sparsity* sp);                                  \
  void g2p2g(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,           \
             const tess_weights* W, const tess_params& prm);                                                         \
  void g2p2g_steps(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,     \
                   const tess_params& prm, int nsteps, double reorder_threshold);                                    \
  void step(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,            \
            const tess_params& prm, int nsteps, double reorder_threshold, tess_sparsity* sp, int* done);             \
  void step_adjoint(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,    \
                    const tess_params& prm, const tess_adjoint& adj);                                                \
  void rollout(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_particles& P,         \
               const tess_params& prm, int nsteps, int every);                                                       \
  void rollout_adjoint(tess_ctx* ctx, int basis, const tess_mesh& mesh, const tess_grid& G, const tess_params& prm,  \
                       const tess_adjoint& adj);                                                                     \
  void batch_create(tess_ctx* ctx, int basis, const tess_mesh& mesh, tess_batch& b);                                 \
  void batch_step(tess_ctx* ctx, int basis, const tess_mesh& mesh, tess_batch& b, int nsteps);                       \
  }
TESS_PART_DECLARE(part_f32_2d)
TESS_PART_DECLARE(part_f32_3d)
TESS_PART_DECLARE(part_f64_2d)
TESS_PART_DECLARE(part_f64_3d)
#undef TESS_PART_DECLARE
#define TESS_FORWARD(mesh, ...)                                  \
  do {                                                           \
    if ((mesh).dtype == TESS_FLOAT32) {                          \
      if ((mesh).dim == 2) return part_f32_2d::__VA_ARGS__;      \
      if ((mesh).dim == 3) return part_f32_3d::__VA_ARGS__;      \
    } else {                                                     \
      if ((mesh).dim == 2) return part_f64_2d::__VA_ARGS__;      \
      if ((mesh).dim == 3) return part_f64_3d::__VA_ARGS__;      \
    }                                                            \
    raise(TESS_ERR_UNSUPPORTED, "unsupported (dim, dtype, basis) combination"); \
  } while (0)

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Profiling hooks (abi.hip): prof_begin returns a token (-1 when disabled).
int prof_begin(tess_ctx* ctx, const char* name, double bytes);
void prof_end(tess_ctx* ctx, int token);
void prof_flush(tess_ctx* ctx);

}  // namespace tess
