// Tile tables and the merge that re-bins particles between two steps.
//
// A binning keeps the particles in the stable order of their sort keys
// (tile * 64 + class) and, per tile, its run in that order.  Between two steps
// only some keys change.  The kernel that computes the new keys (G2P, or
// k_rekey from the positions) works on one tile at a time and leaves, per tile,
// the particles that stay in it (stay), an arrival count of every other tile
// (tin) and a list of those that leave (out: previous sorted position and rank
// among the arrivals of the tile they enter).  From these:
//   k_tab_reduce / k_tab_scan  new runs, active tiles, touched node blocks and
//                              arrival segments in two launches, and the
//                              totals straight into pinned host memory
//   k_scatter_out              the leavers into their tiles' arrival segments
//   k_merge_tiles              per tile: arrivals sorted by previous position,
//                              then one stable counting pass by class over
//                              (arrivals from lower positions, those that
//                              stay, arrivals from higher positions)
// The result is the stable sort of the previous order by the new keys, the
// order a full radix sort of (new key, previous order) gives.  The sort takes the
// merge's place where one tile, or all together, have too many changed keys
// (CNT_RESORT, CNT_MANY): the device says so before the merge runs.
//
// What bounds it: each kernel moves 8-20 bytes per particle or per tile and is
// short, so launches and the one readback bound it below about a million
// particles and HBM above.  The scan, compaction, radix sort and placement of
// the movers that this replaces took about 40 launches and three readbacks per
// step.  A step of two disks (10,048 particles, Float64): 209 us before, 67 us
// with this; of a falling block (1.7 M, Float32): 676 -> 476 us; one rollout
// and pullback of 132,651 particles over 40 steps: 16.7 -> 10.6 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tess_internal.hpp"

namespace tess {
namespace {

constexpr int TAB_THREADS = 1024, TAB_WAVES = TAB_THREADS / 64;

__device__ __forceinline__ uint32_t wave_scan_incl(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  return v;
}

// sum of v over the workgroup's threads, in every thread
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* s) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  uint32_t t = 0;
#pragma unroll
  for (int w = 0; w < TAB_WAVES; ++w) t += s[w];
  return t;
}

// exclusive prefix of v over the workgroup's threads
__device__ __forceinline__ uint32_t block_scan_excl(uint32_t v, uint32_t* s) {
  const uint32_t inc = wave_scan_incl(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 63) s[threadIdx.x >> 6] = inc;
  __syncthreads();
  uint32_t base = 0;
#pragma unroll
  for (int w = 0; w < TAB_WAVES; ++w) base += w < int(threadIdx.x >> 6) ? s[w] : 0u;
  return base + inc - v;
}

// Node block B holds nodes BW*B .. BW*B+BW-1 per axis; tile t's footprint
// [BW*t-1, BW*t+BW+1] touches node blocks t-1, t, t+1: block t is touched when
// a tile within one of it holds a particle (in a batch, of its own scene).
// The neighbours' counts are loaded together (clamped at the mesh's faces).
__device__ __forceinline__ bool touched(const TabArgs& a, int64_t t) {
  int nx = a.nt[0], ny = a.nt[1], nz = a.nt[2];
  int64_t t0 = 0;
  if (a.scene_toff) {
    const uint32_t s = a.tile_scene[t];
    t0 = a.scene_toff[s];
    nx = a.scene_nt[3 * s];
    ny = a.scene_nt[3 * s + 1];
    nz = a.scene_nt[3 * s + 2];
  }
  const uint32_t l = uint32_t(t - t0);
  const int x = int(l % uint32_t(nx)), y = int((l / uint32_t(nx)) % uint32_t(ny)), z = int(l / (uint32_t(nx) * uint32_t(ny)));
  const int xs[3] = {max(x - 1, 0), x, min(x + 1, nx - 1)};
  const int ys[3] = {max(y - 1, 0), y, min(y + 1, ny - 1)};
  uint32_t any = 0;
  for (int dz = nz > 1 ? -1 : 0; dz <= (nz > 1 ? 1 : 0); ++dz) {
    const int64_t zb = t0 + int64_t(min(max(z + dz, 0), nz - 1)) * ny * nx;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int64_t q = zb + int64_t(ys[j]) * nx + xs[i];
        any |= a.stay[q] | a.tin[q];
      }
  }
  return any != 0;
}

// Why a merge should not take a tile (with the last one also the outside).
__device__ __forceinline__ uint32_t crowded(const TabArgs& a, int64_t t, uint32_t arrivals, uint32_t count) {
  const bool in = arrivals > a.crowd || (t == a.ntiles - 1 && a.tin[a.ntiles] > a.crowd);
  return (in ? uint32_t(RESORT_CROWD) : 0u) | (count > a.tile_max ? uint32_t(RESORT_TILE) : 0u);
}

// Per workgroup of TAB_THREADS tiles: particles, arrivals, active tiles and
// touched node blocks; writes the touched flags.  One tile per thread: four per
// thread left a mesh of 36 k tiles on 36 workgroups of 256 threads, each thread
// walking the 27 neighbours of four tiles in turn (22 us).
__global__ __launch_bounds__(TAB_THREADS) void k_tab_reduce(TabArgs a) {
  __shared__ uint32_t s[TAB_WAVES];
  if (a.may_keep) {
    // a step in which no key changed needs the report alone: without this, the
    // two launches took 20 us over the 275 k tiles of a 256^3 mesh
    const int i = int(threadIdx.x & 63);
    const bool keep = __ballot(i < LANES && a.lanes[(LANE_MOVED * LANES + (i & (LANES - 1))) * LANE_STRIDE] != 0u) == 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.counters[CNT_KEEP] = keep ? 1u : 0u;
    if (keep) return;  // uniform
  }
  const int64_t t = int64_t(blockIdx.x) * TAB_THREADS + threadIdx.x;
  uint32_t c = 0, in = 0, pk = 0;
  if (t < a.ntiles) {
    in = a.tin[t];
    c = a.stay[t] + in;
    const uint32_t why = crowded(a, t, in, c);
    if (why) atomicOr(a.counters + CNT_RESORT, why);
    const bool f = c != 0 || touched(a, t);
    a.nb_flag[t] = f ? 1u : 0u;
    pk = (c ? 1u : 0u) | (f ? 0x10000u : 0u);
  }
  c = block_sum(c, s);
  in = block_sum(in, s);
  pk = block_sum(pk, s);
  if (threadIdx.x == 0) {
    a.sums[4 * blockIdx.x] = c;
    a.sums[4 * blockIdx.x + 1] = in;
    a.sums[4 * blockIdx.x + 2] = pk & 0xffffu;
    a.sums[4 * blockIdx.x + 3] = pk >> 16;
  }
}

// Exclusive prefix of the workgroups' sums in place, by one workgroup.  Up to
// SUMS_DIRECT workgroups the scan kernel adds the sums before its own by itself
// (at 1024 that reads 8 MB from the L2 altogether); past them that reading
// would grow with the square of the mesh.
constexpr int64_t SUMS_DIRECT = 1024;
__global__ __launch_bounds__(TAB_THREADS) void k_tab_prefix(uint32_t* __restrict__ sums, int64_t nb) {
  __shared__ uint32_t s[TAB_WAVES], s_last[4];
  uint32_t carry[4] = {0, 0, 0, 0};
  for (int64_t b0 = 0; b0 < nb; b0 += TAB_THREADS) {
    const int64_t b = b0 + threadIdx.x;
    uint32_t v[4], e[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = b < nb ? sums[4 * b + q] : 0u;
      e[q] = carry[q] + block_scan_excl(v[q], s);
      if (b < nb) sums[4 * b + q] = e[q];
      if (threadIdx.x == TAB_THREADS - 1) s_last[q] = e[q] + v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) carry[q] = s_last[q];
    __syncthreads();
  }
}

// A thread's part of the report is in host memory: its number, for wait_report.
__device__ __forceinline__ void reported(const TabArgs& a, int reporter) {
  __threadfence_system();
  if (a.seq) __hip_atomic_store(&a.host[CNT_SEQ + reporter], a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The tables of a workgroup's tiles from the sums of the workgroups before it.
// Workgroup 0 also sums the lane counters (particles whose key changed, broken
// layered pairs, nodes with mass), the last one holds the totals; both report
// to pinned host memory and reset what the next step counts into.  A mesh that
// fits one workgroup needs no sums: this launch alone (ALONE).
template <bool ALONE>
__global__ __launch_bounds__(TAB_THREADS) void k_tab_scan(TabArgs a) {
  __shared__ uint32_t s[TAB_WAVES];
  uint32_t pre[4] = {0, 0, 0, 0};
  uint32_t why = 0u;  // ALONE: what k_tab_reduce would have marked
  bool keep = false;
  if constexpr (!ALONE) {
    keep = a.may_keep && a.counters[CNT_KEEP] != 0u;
    if (keep && blockIdx.x != 0) return;
  }
  if (!keep) {
  if constexpr (!ALONE) {
    if (gridDim.x > SUMS_DIRECT) {
#pragma unroll
      for (int q = 0; q < 4; ++q) pre[q] = a.sums[4 * int64_t(blockIdx.x) + q];
    } else {
      for (int b = int(threadIdx.x); b < int(blockIdx.x); b += TAB_THREADS)
#pragma unroll
        for (int q = 0; q < 4; ++q) pre[q] += a.sums[4 * b + q];
#pragma unroll
      for (int q = 0; q < 4; ++q) pre[q] = block_sum(pre[q], s);
    }
  }
  const int64_t t = int64_t(blockIdx.x) * TAB_THREADS + threadIdx.x;
  const bool ok = t < a.ntiles;
  const uint32_t ti = ok ? a.tin[t] : 0u, ct = ok ? a.stay[t] + ti : 0u;
  uint32_t fl = 0u;
  if constexpr (ALONE) {
    uint32_t w = 0u;
    if (ok) {
      fl = ct != 0 || touched(a, t) ? 1u : 0u;
      a.nb_flag[t] = fl;
      w = crowded(a, t, ti, ct);
    }
    // (a barrier: the neighbours' arrivals have been read; they are reset below)
    if (__syncthreads_or(w != 0u))
      why = (__syncthreads_or(w & RESORT_CROWD) ? uint32_t(RESORT_CROWD) : 0u) |
            (__syncthreads_or(w & RESORT_TILE) ? uint32_t(RESORT_TILE) : 0u);
  } else {
    fl = ok ? a.nb_flag[t] : 0u;
  }
  const uint32_t ec = pre[0] + block_scan_excl(ct, s), ei = pre[1] + block_scan_excl(ti, s);
  const uint32_t epk = block_scan_excl((ct ? 1u : 0u) | (fl << 16), s);
  const uint32_t ea = pre[2] + (epk & 0xffffu), en = pre[3] + (epk >> 16);
  if (ok) {
    a.start[t] = ec;
    a.end[t] = ec + ct;
    a.flag[t] = ct ? 1u : 0u;
    a.slot[t] = ea;
    a.seg[t] = ei;
    if (ct) a.active[ea] = uint32_t(t);
    if (fl) a.nb_list[en] = uint32_t(t);
    if (ti) a.tin[t] = 0u;
  }
  // the thread of the last tile: totals, and the particles outside the mesh
  // (the entry past the tiles)
  if (t == a.ntiles - 1) {
    const uint32_t inside = ec + ct, arrive = ei + ti, act = ea + (ct ? 1u : 0u), nb = en + fl;
    const uint32_t out_in = a.tin[a.ntiles];
    a.seg[a.ntiles] = arrive;
    a.start[a.ntiles] = inside;
    a.stay[a.ntiles] += out_in;
    a.tin[a.ntiles] = 0u;
    a.counters[CNT_PREV_ACTIVE] = a.counters[CNT_ACTIVE];
    a.counters[CNT_INSIDE] = inside;
    a.counters[CNT_ACTIVE] = act;
    a.counters[CNT_NB] = nb;
    a.counters[CNT_OUTIN] = out_in;
    a.counters[CNT_MANY] = arrive + out_in > a.many ? 1u : 0u;
    a.host[CNT_INSIDE] = inside;
    a.host[CNT_ACTIVE] = act;
    a.host[CNT_NB] = nb;
    a.host[CNT_OUTIN] = out_in;
    a.host[CNT_ARRIVE] = arrive + out_in;
    reported(a, LANE_GROUPS);
  }
  } else if (threadIdx.x == 0) {
    reported(a, LANE_GROUPS);  // the totals of the last report stand
  }
  if (blockIdx.x == 0) {
    // one wave per group of lanes
    const int g = int(threadIdx.x >> 6), i = int(threadIdx.x & 63);
    uint32_t x = 0, err = 0, resort = 0;
    if (g == LANE_NODES && i == 0) {  // loaded with the lanes
      err = a.counters[CNT_ERR];
      resort = a.counters[CNT_RESORT] | why;
    }
    if (g < LANE_GROUPS && i < LANES) {
      uint32_t* lane = a.lanes + (g * LANES + i) * LANE_STRIDE;
      x = *lane;
      if (x) *lane = 0u;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, 64);
    if (i == 0 && g < LANE_GROUPS) {
      a.host[g == LANE_MOVED ? CNT_MOVED : g == LANE_BROKEN ? CNT_MISPLACED : CNT_NODES] = x;
      if (g == LANE_MOVED) a.counters[CNT_MOVED] = x;
      if (g == LANE_NODES) {
        a.counters[CNT_NODES] = x;
        a.counters[CNT_RESORTED] = resort;
        a.counters[CNT_RESORT] = 0u;
        a.counters[CNT_SCATTERED] = 0u;
        a.host[CNT_ERR] = err;
        a.host[CNT_RESORT] = resort;
        if (!a.keep_err) a.counters[CNT_ERR] = 0u;
      }
      reported(a, g);
    }
  }
}

// Particles of each tile in a freshly sorted order (binary searches of the
// keys; the entry past the tiles counts the particles outside the mesh).
__global__ __launch_bounds__(256) void k_tile_counts(const uint32_t* __restrict__ skeys, int64_t n, int64_t ntiles,
                                                     uint32_t* __restrict__ stay, uint32_t* __restrict__ tin) {
  __shared__ uint32_t s_bound[257];
  auto bound = [&](int64_t t) {  // first position whose key is not below tile t's
    int64_t lo = 0, hi = n;
    const uint32_t key = uint32_t(t) * 64u;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (skeys[mid] < key) lo = mid + 1;
      else hi = mid;
    }
    return uint32_t(lo);
  };
  const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (t <= ntiles) s_bound[threadIdx.x] = bound(t);
  if (threadIdx.x == 255 && t + 1 <= ntiles) s_bound[256] = bound(t + 1);
  __syncthreads();
  if (t > ntiles) return;
  const uint32_t hi = t == ntiles ? uint32_t(n) : s_bound[threadIdx.x + 1];
  stay[t] = hi - s_bound[threadIdx.x];
  tin[t] = 0u;
}

// A merge launched before the host has read the report: nothing to do when no key
// changed, or when the host sorts them all (CNT_RESORT, CNT_MANY).
__device__ __forceinline__ bool merge_gated(const MergeArgs& a) {
  if (!a.gate) return false;
  const uint32_t moved = a.gate[CNT_MOVED], resort = a.gate[CNT_RESORTED] | a.gate[CNT_MANY];  // read together
  return (moved == 0u) | (resort != 0u);
}

// The leavers of each previously active tile into the arrival segments of the
// tiles they enter (a leaver's rank there was drawn when its key was computed).
__global__ __launch_bounds__(64) void k_scatter_out(MergeArgs a) {
  if (merge_gated(a)) return;
  const int64_t count = int64_t(a.old_count ? *a.old_count : a.old_active_n);
  for (int64_t j = blockIdx.x; j < count; j += gridDim.x) {
    const uint32_t t = a.old_active[j];
    const uint32_t start = a.old_start[t], cnt = a.old_end[t] - start;
    const uint32_t leave = cnt - a.stay[t];
    for (uint32_t i = threadIdx.x; i < leave; i += 64) {
      const uint2 o = a.out[start + i];
      const uint32_t key = a.nk[o.x];
      a.seg[a.seg_off[key >> 6] + o.y] = make_uint2(key, o.x);
    }
  }
}

// The merge runs one workgroup per tile, of 4 waves also where tiles hold few
// particles: one wave for each of the batch's 215 k tiles of 45 particles made a
// call of 8 steps 0.26 ms longer, and a binning of the two disks 3 us.  Arrivals
// up to the LDS list are sorted there.
constexpr int MERGE_WAVES = 4, MERGE_THREADS = 64 * MERGE_WAVES;
constexpr uint32_t MERGE_CAP = 512;

// Sorts k (key, position) pairs of a segment by position with one workgroup:
// 8-bit digits of the position, `bits` low bits, between seg and alt; returns
// the buffer that holds the result.  For segments past the LDS list.
__device__ uint2* segment_sort(uint2* seg, uint2* alt, uint32_t k, int bits, uint32_t* s_hist, uint32_t (*s_wc)[256]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int shift = 0; shift < bits; shift += 8) {
    __syncthreads();
    for (int d = int(threadIdx.x); d < 256; d += MERGE_THREADS) s_hist[d] = 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < k; i += MERGE_THREADS) atomicAdd(&s_hist[(seg[i].y >> shift) & 255u], 1u);
    __syncthreads();
    if (wave == 0) {  // exclusive prefix of the 256 digits, four per lane
      uint32_t h[4], tot = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        h[q] = s_hist[4 * lane + q];
        tot += h[q];
      }
      uint32_t run = wave_scan_incl(tot) - tot;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s_hist[4 * lane + q] = run;
        run += h[q];
      }
    }
    __syncthreads();
    for (uint32_t b = 0; b < k; b += MERGE_THREADS) {
      const uint32_t i = b + threadIdx.x;
      const bool valid = i < k;
      const uint2 e = valid ? seg[i] : make_uint2(0u, 0u);
      const uint32_t d = (e.y >> shift) & 255u;
      for (int q = int(threadIdx.x); q < 256; q += MERGE_THREADS)
#pragma unroll
        for (int w = 0; w < MERGE_WAVES; ++w) s_wc[w][q] = 0;
      __syncthreads();
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const bool bit = (d >> q) & 1u;
        const uint64_t m = __ballot(valid && bit);
        peers &= bit ? m : ~m;
      }
      const uint32_t below = uint32_t(__popcll(peers & ((uint64_t(1) << lane) - 1)));
      if (valid && below == 0) s_wc[wave][d] = uint32_t(__popcll(peers));
      __syncthreads();
      if (valid) {
        uint32_t pos = s_hist[d] + below;
        for (int w = 0; w < wave; ++w) pos += s_wc[w][d];
        alt[pos] = e;
      }
      __syncthreads();
      for (int q = int(threadIdx.x); q < 256; q += MERGE_THREADS) {
        uint32_t add = 0;
#pragma unroll
        for (int w = 0; w < MERGE_WAVES; ++w) add += s_wc[w][q];
        s_hist[q] += add;
      }
      __syncthreads();
    }
    __threadfence_block();
    __syncthreads();
    uint2* const x = seg;
    seg = alt;
    alt = x;
  }
  return seg;
}

// One workgroup per tile that holds particles now.  The tile's new run is the
// stable counting sort, by class, of a sequence in order of previous position:
// arrivals from below its old run, the old run without its leavers, arrivals
// from above.  The waves take consecutive parts of the sequence.
__global__ __launch_bounds__(MERGE_THREADS) void k_merge_tiles(MergeArgs a) {
  __shared__ uint2 s_raw[MERGE_CAP], s_in[MERGE_CAP];
  __shared__ uint32_t s_hist[256], s_wc[MERGE_WAVES][256];
  __shared__ uint32_t s_base[MERGE_WAVES][64], s_low;
  const int64_t jt = a.first_tile + int64_t(blockIdx.x);
  const uint32_t t = a.new_active[jt];  // (ntiles entries: in range whether or not jt is active)
  if (jt >= int64_t(a.new_count ? *a.new_count : a.new_active_n) || merge_gated(a)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const uint32_t os = a.old_start[t], oc = a.old_end[t] - os;
  const uint32_t ns = a.new_start[t], k = a.new_end[t] - ns - a.stay[t];
  const uint2* in = s_in;
  if (threadIdx.x == 0) s_low = 0;
  s_base[wave][lane] = 0;
  if (k > 0 && k <= MERGE_CAP) {
    const uint2* seg = a.seg + a.seg_off[t];
    for (uint32_t i = threadIdx.x; i < k; i += MERGE_THREADS) s_raw[i] = seg[i];
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < k; i += MERGE_THREADS) {
      const uint2 e = s_raw[i];
      uint32_t r = 0;
      for (uint32_t q = 0; q < k; ++q) r += s_raw[q].y < e.y ? 1u : 0u;
      s_in[r] = e;
    }
  } else if (k > 0) {
    in = segment_sort(a.seg + a.seg_off[t], a.seg_alt + a.seg_off[t], k, a.pos_bits, s_hist, s_wc);
  }
  __syncthreads();
  if (k > 0) {
    uint32_t low = 0;
    for (uint32_t i = threadIdx.x; i < k; i += MERGE_THREADS) low += in[i].y < os ? 1u : 0u;
    if (low) atomicAdd(&s_low, low);
    __syncthreads();
  }
  const uint32_t klow = s_low, len = k + oc;
  // element i of the sequence: its key (in *valid elements) and previous position
  auto element = [&](uint32_t i, uint32_t& key, uint32_t& pos) {
    if (i >= len) return false;
    if (i >= klow && i < klow + oc) {
      pos = os + (i - klow);
      key = a.nk[pos];
      return (key >> 6) == t;
    }
    const uint2 e = in[i < klow ? i : i - oc];
    key = e.x;
    pos = e.y;
    return true;
  };
  const uint32_t quarter = ((len + MERGE_THREADS - 1) / MERGE_THREADS) * 64u;  // a wave's part
  const uint32_t i0 = uint32_t(wave) * quarter;
  auto match = [&](uint32_t c, bool valid) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const bool bit = (c >> b) & 1u;
      const uint64_t m = __ballot(valid && bit);
      peers &= bit ? m : ~m;
    }
    return peers;
  };
  const uint64_t lt = (uint64_t(1) << lane) - 1;
  // class counts of the wave's quarter; the first chunks stay in registers
  constexpr int KEEP = 4;
  uint32_t kk[KEEP], kp[KEEP];
  bool kv[KEEP];
#pragma unroll
  for (int r = 0; r < KEEP; ++r) {
    kk[r] = kp[r] = 0u;
    kv[r] = uint32_t(r) * 64u < quarter && element(i0 + uint32_t(r) * 64u + uint32_t(lane), kk[r], kp[r]);
  }
  uint32_t* mine = s_base[wave];
#pragma unroll
  for (int r = 0; r < KEEP; ++r) {
    if (uint32_t(r) * 64u >= quarter) break;  // uniform
    const uint64_t peers = match(kk[r] & 63u, kv[r]);
    if (kv[r] && (peers & lt) == 0) mine[kk[r] & 63u] += uint32_t(__popcll(peers));
    __asm__ volatile("" ::: "memory");  // the next chunk's counts in program order
  }
  for (uint32_t o = KEEP * 64u; o < quarter; o += 64u) {
    uint32_t key = 0u, pos = 0u;
    const bool v = element(i0 + o + uint32_t(lane), key, pos);
    const uint64_t peers = match(key & 63u, v);
    if (v && (peers & lt) == 0) mine[key & 63u] += uint32_t(__popcll(peers));
    __asm__ volatile("" ::: "memory");
  }
  __syncthreads();
  // where each (class, wave) starts: classes ascending, waves in order
  if (wave == 0) {
    uint32_t tot = 0, w[MERGE_WAVES];
#pragma unroll
    for (int q = 0; q < MERGE_WAVES; ++q) {
      w[q] = s_base[q][lane];
      tot += w[q];
    }
    uint32_t run = wave_scan_incl(tot) - tot;
#pragma unroll
    for (int q = 0; q < MERGE_WAVES; ++q) {
      s_base[q][lane] = run;
      run += w[q];
    }
  }
  __syncthreads();
  auto place = [&](uint32_t key, uint32_t pos, bool v) {
    const uint64_t peers = match(key & 63u, v);
    const uint32_t below = uint32_t(__popcll(peers & lt));
    // the leader of each class draws its peers' slots (the LDS executes one
    // wave's accesses in order; the shuffle hands the base to the peers)
    uint32_t base = 0u;
    if (v && below == 0) {
      base = mine[key & 63u];
      mine[key & 63u] = base + uint32_t(__popcll(peers));
    }
    __asm__ volatile("" ::: "memory");  // the next chunk draws after this one
    base = __shfl(base, v ? __ffsll((unsigned long long)peers) - 1 : lane, 64);
    if (v) {
      a.keys_new[ns + base + below] = key;
      a.perm_new[ns + base + below] = a.perm_old[pos];
    }
  };
#pragma unroll
  for (int r = 0; r < KEEP; ++r) {
    if (uint32_t(r) * 64u >= quarter) break;  // uniform
    place(kk[r], kp[r], kv[r]);
  }
  for (uint32_t o = KEEP * 64u; o < quarter; o += 64u) {
    uint32_t key = 0u, pos = 0u;
    const bool v = element(i0 + o + uint32_t(lane), key, pos);
    place(key, pos, v);
  }
}

// Arrivals outside the mesh, many of them, in order of previous position: each of
// `parts` workgroups counts those at positions before its part (reading them all,
// so that no workgroup waits for another) and places its own.
constexpr uint32_t OUTSIDE_PARTS = 128;
__device__ void place_outside(const MergeArgs& a, uint32_t ns, uint32_t os, uint32_t parts, uint32_t* s_sum) {
  constexpr uint32_t STEP = 4 * MERGE_THREADS;  // positions of a workgroup at a time, four a thread
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t out = uint32_t(a.ntiles);
  const uint32_t part = ((os + parts - 1) / parts + STEP - 1) / STEP * STEP;
  const uint32_t lo = blockIdx.x * part, hi = min(os, lo + part);
  if (lo >= os) return;  // uniform
  const uint4* nk4 = reinterpret_cast<const uint4*>(a.nk);
  uint32_t before = 0;
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < lo / 4; i += MERGE_THREADS) {
    const uint4 q = nk4[i];
    before += (q.x >> 6 == out) + (q.y >> 6 == out) + (q.z >> 6 == out) + (q.w >> 6 == out);
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) before += __shfl_xor(before, off, 64);
  if (lane == 0) s_sum[wave] = before;
  __syncthreads();
  uint32_t at = ns;
#pragma unroll
  for (int w = 0; w < MERGE_WAVES; ++w) at += s_sum[w];
  for (uint32_t b = lo; b < hi; b += STEP) {
    const uint32_t i = b + 4 * threadIdx.x;
    uint32_t key[4], mine = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      key[q] = i + q < hi ? a.nk[i + q] : 0u;
      mine += i + q < hi && key[q] >> 6 == out ? 1u : 0u;
    }
    const uint32_t incl = wave_scan_incl(mine);
    __syncthreads();  // the sums have been read
    if (lane == 63) s_sum[wave] = incl;
    __syncthreads();
    uint32_t r = at + incl - mine;
#pragma unroll
    for (int w = 0; w < MERGE_WAVES; ++w) {
      if (w < wave) r += s_sum[w];
      at += s_sum[w];
    }
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      if (i + q < hi && key[q] >> 6 == out) {
        a.keys_new[r] = key[q];
        a.perm_new[r++] = a.perm_old[i + q];
      }
    }
  }
}

// Particles outside the mesh: those that were outside keep their order behind
// the arrivals (whose previous positions are all lower).  Workgroup 0 places
// the arrivals, sorted by previous position; a captured step, which merges
// whatever their number, shares many among its workgroups from where the host would
// sort every key (six steps, 800 k particles that leave in three of them: 2D 13.0
// and 1.8 ms, 3D 13.7 and 1.6 ms).
__global__ __launch_bounds__(MERGE_THREADS) void k_merge_outside(MergeArgs a) {
  __shared__ uint32_t s_hist[256], s_wc[MERGE_WAVES][256];
  const uint32_t k = a.counters ? a.counters[CNT_OUTIN] : a.out_in;
  const uint32_t ns = a.new_start[a.ntiles], os = a.old_start[a.ntiles];
  const uint32_t parts = min(gridDim.x, OUTSIDE_PARTS);
  if (k > a.crowd) {
    if (blockIdx.x < parts) place_outside(a, ns, os, parts, s_hist);
  } else if (blockIdx.x == 0 && k > 0) {
    const uint32_t off = a.seg_off[a.ntiles];
    const uint2* in = segment_sort(a.seg + off, a.seg_alt + off, k, a.pos_bits, s_hist, s_wc);
    for (uint32_t i = threadIdx.x; i < k; i += MERGE_THREADS) {
      a.keys_new[ns + i] = in[i].x;
      a.perm_new[ns + i] = a.perm_old[in[i].y];
    }
  }
  const uint32_t stayed = uint32_t(a.n) - os;
  for (uint32_t i = blockIdx.x * MERGE_THREADS + threadIdx.x; i < stayed; i += gridDim.x * MERGE_THREADS) {
    a.keys_new[ns + k + i] = a.nk[os + i];
    a.perm_new[ns + k + i] = a.perm_old[os + i];
  }
}

}  // namespace

int64_t tab_blocks(int64_t ntiles) { return ceil_div(ntiles, int64_t(TAB_THREADS)); }

void launch_tables(hipStream_t st, const TabArgs& a) {
  const unsigned nb = unsigned(tab_blocks(a.ntiles));
  if (nb == 1) {
    hipLaunchKernelGGL(k_tab_scan<true>, dim3(1), dim3(TAB_THREADS), 0, st, a);
    TESS_HIP(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(k_tab_reduce, dim3(nb), dim3(TAB_THREADS), 0, st, a);
  TESS_HIP(hipGetLastError());
  if (int64_t(nb) > SUMS_DIRECT) {
    hipLaunchKernelGGL(k_tab_prefix, dim3(1), dim3(TAB_THREADS), 0, st, a.sums, int64_t(nb));
    TESS_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_tab_scan<false>, dim3(nb), dim3(TAB_THREADS), 0, st, a);
  TESS_HIP(hipGetLastError());
}

void launch_tile_counts(hipStream_t st, const uint32_t* skeys, int64_t n, int64_t ntiles, uint32_t* stay, uint32_t* tin) {
  hipLaunchKernelGGL(k_tile_counts, dim3(unsigned(ceil_div(ntiles + 1, int64_t(256)))), dim3(256), 0, st, skeys, n, ntiles,
                     stay, tin);
  TESS_HIP(hipGetLastError());
}

// workgroups of k_scatter_out: one per tile cost 56 us for 258 k tiles (0.2 ns of
// dispatch each), 16 k that walk them 19 us
constexpr int64_t SCATTER_GRID = 16384;

// The launch counts are those of the host, or upper bounds of the device counts
// the args point at.
void launch_merge(hipStream_t st, const MergeArgs& a, unsigned outside_blocks) {
  if (a.old_active_n > 0) {
    hipLaunchKernelGGL(k_scatter_out, dim3(unsigned(std::min<int64_t>(a.old_active_n, SCATTER_GRID))), dim3(64), 0, st,
                       a);
    TESS_HIP(hipGetLastError());
  }
  launch_merge_tiles(st, a, a.new_active_n);
  if (outside_blocks > 0) launch_merge_outside(st, a, outside_blocks);
}

// The tiles from a.first_tile on, one workgroup each.
void launch_merge_tiles(hipStream_t st, const MergeArgs& a, int64_t tiles) {
  if (tiles <= 0) return;
  hipLaunchKernelGGL(k_merge_tiles, dim3(unsigned(tiles)), dim3(MERGE_THREADS), 0, st, a);
  TESS_HIP(hipGetLastError());
}

void launch_merge_outside(hipStream_t st, const MergeArgs& a, unsigned blocks) {
  hipLaunchKernelGGL(k_merge_outside, dim3(blocks), dim3(256), 0, st, a);
  TESS_HIP(hipGetLastError());
}

}  // namespace tess
