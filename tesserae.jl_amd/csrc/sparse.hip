// SpIndices block activation and numbering from particle positions
// (update_sparsity!(spinds, xₚ, mesh), src/Grids/sparsity.jl:23-40,53-60,
// 120-238).  Blocks of 2^L nodes per axis; a block holding a particle is
// occupied, every block within ±1 block of an occupied one is active, and the
// active blocks are numbered 1, 2, ... in column-major block order.
#include <hip/hip_runtime.h>

#include "tess_device.hpp"
#include "tess_internal.hpp"

namespace tess {
namespace {

// words of the pinned readback slots this file reports to
enum { SP_COUNT = 32, SP_CHANGED = 33 };

template <int D>
struct BlockGrid {
  int32_t nb[D];
  int64_t total;
};

// occupied[b] = 1 for the block of every particle inside the mesh
// (findblock, src/Mesh/cartesian.jl:277-285: cell0 = floor((x-xmin)h⁻¹),
// inside iff 0 <= cell0 <= dims-2, block = cell0 >> L).
template <typename T, int D>
__global__ __launch_bounds__(256) void k_sp_occupied(DField<T> x, int64_t n, DMesh<T, D> mesh, int L,
                                                     BlockGrid<D> bg, uint32_t* __restrict__ occ) {
  const int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int64_t b = 0;
  bool inside = true;
#pragma unroll
  for (int d = D - 1; d >= 0; --d) {
    const T f = floor((x(p, d) - mesh.xmin[d]) * mesh.h_inv);
    inside = inside && T(0) <= f && f <= T(mesh.dims[d] - 2);
    const int c = inside ? int(f) : 0;
    b = b * bg.nb[d] + (c >> L);
  }
  if (inside) occ[b] = 1u;  // every writer stores the same value
}

// act[b] = 1 if any block of the 3^dim neighbourhood is occupied
// (_activate_block_neighborhood!, sparsity.jl:141-145), with the workgroup's
// count of active blocks and whether its part of the active set differs from
// the numbering passed in (sparsity.jl:262-267).
constexpr int SP_THREADS = 256;
template <int D>
__global__ __launch_bounds__(SP_THREADS) void k_sp_activity(const uint32_t* __restrict__ occ, BlockGrid<D> bg,
                                                            const int32_t* __restrict__ old_numbering,
                                                            uint32_t* __restrict__ act,
                                                            uint2* __restrict__ sums) {
  __shared__ uint32_t s_n[SP_THREADS / 64], s_c[SP_THREADS / 64];
  const int64_t b = int64_t(blockIdx.x) * SP_THREADS + threadIdx.x;
  bool a = false, diff = false;
  if (b < bg.total) {
    int I[D];
    int64_t r = b;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      I[d] = int(r % bg.nb[d]);
      r /= bg.nb[d];
    }
    constexpr int NN = (D == 3) ? 27 : 9;
    uint32_t any = 0;  // the neighbours' flags loaded together, clamped at the faces
#pragma unroll
    for (int k = 0; k < NN; ++k) {
      int q = k;
      int J[D];
#pragma unroll
      for (int d = 0; d < D; ++d) {
        J[d] = min(max(I[d] + q % 3 - 1, 0), bg.nb[d] - 1);
        q /= 3;
      }
      int64_t nb = J[D - 1];
#pragma unroll
      for (int d = D - 2; d >= 0; --d) nb = nb * bg.nb[d] + J[d];
      any |= occ[nb];
    }
    a = any != 0;
    act[b] = a ? 1u : 0u;
    diff = (old_numbering[b] != 0) != a;
  }
  const uint64_t m = __ballot(a), dm = __ballot(diff);
  if ((threadIdx.x & 63) == 0) {
    s_n[threadIdx.x >> 6] = uint32_t(__popcll(m));
    s_c[threadIdx.x >> 6] = dm ? 1u : 0u;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint2 t = make_uint2(0u, 0u);
    for (int w = 0; w < SP_THREADS / 64; ++w) {
      t.x += s_n[w];
      t.y |= s_c[w];
    }
    sums[blockIdx.x] = t;
  }
}

// Exclusive prefix of the workgroups' counts (and the OR of their changes) in
// place, by one workgroup, where there are more of them than k_sp_number should
// add up by itself.  Entry `wgs` receives the total.
constexpr int64_t SUMS_DIRECT = 1024;
__global__ __launch_bounds__(64) void k_sp_prefix(uint2* __restrict__ sums, int64_t wgs) {
  uint32_t carry = 0, ch = 0;
  for (int64_t b0 = 0; b0 < wgs; b0 += 64) {
    const int64_t b = b0 + threadIdx.x;
    const uint2 v = b < wgs ? sums[b] : make_uint2(0u, 0u);
    uint32_t inc = v.x;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t u = __shfl_up(inc, off, 64);
      if (int(threadIdx.x) >= off) inc += u;
    }
    if (__ballot(v.y != 0)) ch = 1u;
    if (b < wgs) sums[b].x = carry + inc - v.x;
    carry += __shfl(inc, 63, 64);
  }
  if (threadIdx.x == 0) sums[wgs] = make_uint2(carry, ch);
}

// The numbers of a workgroup's active blocks after the counts of the workgroups
// before it; clears the occupied flags for the next update.  The last workgroup
// reports the totals to pinned host memory.
__global__ __launch_bounds__(SP_THREADS) void k_sp_number(const uint32_t* __restrict__ act,
                                                          const uint2* __restrict__ sums, int64_t total,
                                                          int32_t* __restrict__ numbering, uint32_t* __restrict__ occ,
                                                          uint32_t* __restrict__ host) {
  __shared__ uint32_t s_n[SP_THREADS / 64], s_c[SP_THREADS / 64], s_w[SP_THREADS / 64];
  const bool last = blockIdx.x == gridDim.x - 1;
  uint32_t pre = 0, ch = 0;
  if (int64_t(gridDim.x) > SUMS_DIRECT) {
    if (threadIdx.x == 0) {
      pre = sums[blockIdx.x].x;
      ch = sums[gridDim.x].y;
    }
  } else {
    for (int i = int(threadIdx.x); i < int(blockIdx.x); i += SP_THREADS) {
      const uint2 t = sums[i];
      pre += t.x;
      ch |= t.y;
    }
    if (last && threadIdx.x == 0) ch |= sums[blockIdx.x].y;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    pre += __shfl_xor(pre, off, 64);
    ch |= __shfl_xor(ch, off, 64);
  }
  const int64_t b = int64_t(blockIdx.x) * SP_THREADS + threadIdx.x;
  const bool a = b < total && act[b] != 0;
  const uint64_t m = __ballot(a);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    s_n[wave] = pre;
    s_c[wave] = ch;
    s_w[wave] = uint32_t(__popcll(m));
  }
  __syncthreads();
  uint32_t base = 0, own = 0, changed = 0;
  for (int w = 0; w < SP_THREADS / 64; ++w) {
    base += s_n[w];
    changed |= s_c[w];
    own += s_w[w];
  }
  for (int w = 0; w < wave; ++w) base += s_w[w];
  if (b < total) {
    numbering[b] = a ? int32_t(base + uint32_t(__popcll(m & ((uint64_t(1) << lane) - 1))) + 1u) : 0;
    occ[b] = 0u;
  }
  if (last && threadIdx.x == 0) {
    host[SP_COUNT] = base + own;  // thread 0 is in wave 0: base holds the workgroups before
    host[SP_CHANGED] = changed;
    __threadfence_system();
  }
}

template <int D>
BlockGrid<D> block_grid(const tess_mesh& mesh) {
  BlockGrid<D> bg;
  bg.total = 1;
  for (int d = 0; d < D; ++d) {
    bg.nb[d] = int32_t(((mesh.dims[d] - 1) >> mesh.block_size_log2) + 1);
    bg.total *= bg.nb[d];
  }
  return bg;
}

}  // namespace

// The totals of an update whose kernels have run.
void take_sparsity(tess_ctx* ctx, const tess_mesh& mesh, tess_sparsity& sp, int32_t* changed) {
  const uint32_t* hc = reinterpret_cast<const uint32_t*>(ctx->counters_host);
  sp.storage_len = int64_t(hc[SP_COUNT]) << (mesh.block_size_log2 * mesh.dim);
  if (changed) *changed = hc[SP_CHANGED] ? 1 : 0;
}

namespace {

template <typename T, int D>
void sparsity_impl(tess_ctx* ctx, const tess_mesh& mesh, tess_field x, int64_t n, tess_sparsity& sp,
                   int32_t* changed, bool defer) {
  const BlockGrid<D> bg = block_grid<D>(mesh);
  const int L = mesh.block_size_log2;
  const int64_t nbt = bg.total;
  if (nbt >= (int64_t(1) << 31)) raise(TESS_ERR_UNSUPPORTED, "block table larger than 2^31 blocks");
  uint32_t* act = ctx->sp_act.as<uint32_t>(size_t(nbt));
  const int64_t wgs = ceil_div(nbt, int64_t(SP_THREADS));
  uint2* sums = ctx->sp_sums.as<uint2>(size_t(wgs) + 1);
  uint32_t* occ = static_cast<uint32_t*>(ctx->sp_occ.ptr);
  if (ctx->sp_clean != nbt || !occ) {
    // the first update of this many blocks, or one that was cut short
    occ = ctx->sp_occ.as<uint32_t>(size_t(nbt));
    TESS_HIP(hipMemsetAsync(occ, 0, size_t(nbt) * sizeof(uint32_t), ctx->stream));
  }
  ctx->sp_clean = -1;
  if (n > 0) {
    const DMesh<T, D> dm = dmesh<T, D>(mesh);
    hipLaunchKernelGGL((k_sp_occupied<T, D>), dim3(unsigned(ceil_div(n, 256))), dim3(256), 0, ctx->stream,
                       dfield<T>(x), n, dm, L, bg, occ);
    TESS_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL((k_sp_activity<D>), dim3(unsigned(wgs)), dim3(SP_THREADS), 0, ctx->stream, occ, bg,
                     static_cast<const int32_t*>(sp.blocknumbering), act, sums);
  TESS_HIP(hipGetLastError());
  if (wgs > SUMS_DIRECT) {
    hipLaunchKernelGGL(k_sp_prefix, dim3(1), dim3(64), 0, ctx->stream, sums, wgs);
    TESS_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_sp_number, dim3(unsigned(wgs)), dim3(SP_THREADS), 0, ctx->stream, act, sums, nbt,
                     sp.blocknumbering, occ, reinterpret_cast<uint32_t*>(ctx->counters_host));
  TESS_HIP(hipGetLastError());
  ctx->sp_clean = nbt;
  if (defer) return;
  TESS_HIP(hipStreamSynchronize(ctx->stream));
  take_sparsity(ctx, mesh, sp, changed);
}

}  // namespace

void run_sparsity_update(tess_ctx* ctx, const tess_mesh& mesh, tess_field x, int64_t n, tess_sparsity& sp,
                         int32_t* changed, bool defer) {
  if (mesh.dtype == TESS_FLOAT32) {
    if (mesh.dim == 2) sparsity_impl<float, 2>(ctx, mesh, x, n, sp, changed, defer);
    else sparsity_impl<float, 3>(ctx, mesh, x, n, sp, changed, defer);
  } else {
    if (mesh.dim == 2) sparsity_impl<double, 2>(ctx, mesh, x, n, sp, changed, defer);
    else sparsity_impl<double, 3>(ctx, mesh, x, n, sp, changed, defer);
  }
}

}  // namespace tess
