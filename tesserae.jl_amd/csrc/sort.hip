// Device-wide exclusive scan and stable LSD radix sort (keys: uint32, values:
// uint32) used for particle binning.  Integer-only, so results are
// deterministic; ranking inside a workgroup is stable (index order).
//
// Sort pass structure (one digit of 8 to 10 bits per pass, sort_digit_bits):
//   1. k_radix_hist   per-workgroup digit histogram of a chunk, stored
//                     digit-major: hist[digit * nchunks + chunk]
//   2. k_radix_rows   one workgroup per digit: exclusive scan of its row, and
//                     its total
//   3. k_radix_scatter re-reads the chunk, each wave a consecutive part of it,
//                     ranks each key among equal digits (wave match via
//                     ballots and running counts per wave, no barrier between
//                     rounds), and writes (key, value) to offset + rank.
//
// What bounds it: up to a million particles the launches and the few hundred
// workgroups, each a serial chain of rounds; past that the scattered writes of 4
// bytes.  1.67 M particles with 20-bit keys, unsorted: three passes took 12 us for
// the histogram, 14 us for a scan of three launches and 22 us with four barriers
// per 256 keys each; now they take 8 + 4 + 15 us, and the block partition that
// they serve 115 us instead of 188.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "tess_internal.hpp"

namespace tess {
namespace {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_CHUNK = SCAN_THREADS * SCAN_ITEMS;  // 4096

constexpr int RADIX_BITS_MAX = 10;
constexpr int SORT_THREADS = 256;
constexpr int SORT_WAVES = SORT_THREADS / 64;
// Keys per thread: 16 fill the chip from 4 M keys on (1024 chunks); below, 8.
constexpr int SORT_ROUNDS_LARGE = 16, SORT_ROUNDS_SMALL = 8;
constexpr int64_t SORT_LARGE = int64_t(4) << 20;
inline int64_t sort_chunk(int64_t n) {
  return int64_t(SORT_THREADS) * (n >= SORT_LARGE ? SORT_ROUNDS_LARGE : SORT_ROUNDS_SMALL);
}
// Digit bits: as few passes as 10-bit digits give, of equal width, while launches
// are what a pass costs; 8-bit digits from SORT_NARROW keys on, where a wider
// digit leaves a chunk two keys of each and its writes share no line.  A block
// partition of particles in no order, 10-bit and 8-bit digits: 0.05 M 68 and 79 us,
// 0.8 M 84 and 102, 1.67 M 137 and 133, 3.3 M 205 and 182.
constexpr int64_t SORT_NARROW = int64_t(1) << 20;
inline int sort_passes(int key_bits, int64_t n) {
  const int widest = n < SORT_NARROW ? RADIX_BITS_MAX : 8;
  return key_bits <= 0 ? 1 : (key_bits + widest - 1) / widest;
}
inline int sort_digit_bits(int key_bits, int64_t n) {
  const int p = sort_passes(key_bits, n);
  const int b = (key_bits + p - 1) / p;
  return b < 8 ? 8 : b;
}

__device__ __forceinline__ uint32_t wave_inclusive_scan(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  return v;
}

// Block-wide exclusive scan of one value per thread (256 threads); returns the
// exclusive prefix and the block total.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t& total, uint32_t* s_wave) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t inc = wave_inclusive_scan(v);
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  uint32_t wave_off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < SCAN_THREADS / 64; ++w) {
    const uint32_t s = s_wave[w];
    if (w < wave) wave_off += s;
    tot += s;
  }
  total = tot;
  __syncthreads();
  return wave_off + inc - v;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const uint32_t* __restrict__ data, int64_t n,
                                                               uint32_t* __restrict__ block_sums) {
  __shared__ uint32_t s_wave[SCAN_THREADS / 64];
  const int64_t base = int64_t(blockIdx.x) * SCAN_CHUNK;
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const int64_t i = base + int64_t(k) * SCAN_THREADS + threadIdx.x;
    if (i < n) s += data[i];
  }
  uint32_t total;
  block_exclusive_scan(s, total, s_wave);
  if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

// In-place exclusive scan of each chunk, offset by block_offsets[chunk].
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_apply(uint32_t* __restrict__ data, int64_t n,
                                                              const uint32_t* __restrict__ block_offsets,
                                                              uint32_t* __restrict__ total_out) {
  __shared__ uint32_t s_items[SCAN_CHUNK];
  __shared__ uint32_t s_wave[SCAN_THREADS / 64];
  const int64_t base = int64_t(blockIdx.x) * SCAN_CHUNK;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const int64_t i = base + int64_t(k) * SCAN_THREADS + threadIdx.x;
    s_items[k * SCAN_THREADS + threadIdx.x] = i < n ? data[i] : 0u;
  }
  __syncthreads();
  uint32_t local[SCAN_ITEMS];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    local[k] = s_items[threadIdx.x * SCAN_ITEMS + k];
    sum += local[k];
  }
  uint32_t total;
  uint32_t run = block_exclusive_scan(sum, total, s_wave) + (block_offsets ? block_offsets[blockIdx.x] : 0u);
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    s_items[threadIdx.x * SCAN_ITEMS + k] = run;
    run += local[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const int64_t i = base + int64_t(k) * SCAN_THREADS + threadIdx.x;
    if (i < n) data[i] = s_items[k * SCAN_THREADS + threadIdx.x];
  }
  if (total_out && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
    // last chunk: offset + chunk total = grand total
    *total_out = (block_offsets ? block_offsets[blockIdx.x] : 0u) + total;
  }
}

__device__ __forceinline__ uint64_t lanemask_lt() {
  const int lane = threadIdx.x & 63;
  return (uint64_t(1) << lane) - 1;
}

// Lanes of the wave whose digit equals this lane's (among `valid` lanes).
template <int RB>
__device__ __forceinline__ uint64_t match_digit(uint32_t digit, bool valid) {
  uint64_t peers = __ballot(valid);
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const bool bit = (digit >> b) & 1u;
    const uint64_t m = __ballot(valid && bit);
    peers &= bit ? m : ~m;
  }
  return peers;
}

template <int RB, int ROUNDS>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_hist(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                              uint32_t* __restrict__ hist, int64_t nchunks) {
  constexpr int RADIX = 1 << RB;
  __shared__ uint32_t s_hist[RADIX];
  const int64_t base = int64_t(blockIdx.x) * (SORT_THREADS * ROUNDS);
  uint32_t k[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = base + r * SORT_THREADS + threadIdx.x;
    k[r] = i < n ? keys[i] : 0u;
  }
  for (int d = int(threadIdx.x); d < RADIX; d += SORT_THREADS) s_hist[d] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = base + r * SORT_THREADS + threadIdx.x;
    const bool valid = i < n;
    // integer adds, whose order does not matter; a wave whose keys share one
    // digit (nearly sorted input) adds once
    const uint32_t digit = (k[r] >> shift) & (RADIX - 1);
    const uint64_t live = __ballot(valid);
    if (live == 0) continue;
    const uint32_t d0 = uint32_t(__shfl(int(digit), __ffsll((unsigned long long)live) - 1, 64));
    if (__ballot(valid && digit != d0) == 0) {
      if ((threadIdx.x & 63) == 0) atomicAdd(&s_hist[d0], uint32_t(__popcll(live)));
    } else if (valid) {
      atomicAdd(&s_hist[digit], 1u);
    }
  }
  __syncthreads();
  for (int d = int(threadIdx.x); d < RADIX; d += SORT_THREADS) hist[int64_t(d) * nchunks + blockIdx.x] = s_hist[d];
}

// Exclusive scan of each digit's row of chunk counts in place; the row total
// goes to totals[digit].
__global__ __launch_bounds__(SORT_THREADS) void k_radix_rows(uint32_t* __restrict__ hist, int64_t nchunks,
                                                              uint32_t* __restrict__ totals) {
  __shared__ uint32_t s_wave[SORT_THREADS / 64];
  uint32_t* row = hist + int64_t(blockIdx.x) * nchunks;
  uint32_t carry = 0;
  for (int64_t c0 = 0; c0 < nchunks; c0 += SORT_THREADS) {
    const int64_t c = c0 + threadIdx.x;
    const uint32_t v = c < nchunks ? row[c] : 0u;
    uint32_t total;
    const uint32_t e = block_exclusive_scan(v, total, s_wave);
    if (c < nchunks) row[c] = carry + e;
    carry += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

template <int RB, int ROUNDS>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_scatter(const uint32_t* __restrict__ keys_in,
                                                                 const uint32_t* __restrict__ vals_in,
                                                                 uint32_t* __restrict__ keys_out,
                                                                 uint32_t* __restrict__ vals_out, int64_t n,
                                                                 int shift, const uint32_t* __restrict__ rows,
                                                                 const uint32_t* __restrict__ totals,
                                                                 int64_t nchunks) {
  constexpr int RADIX = 1 << RB, PER = RADIX / SORT_THREADS;
  __shared__ uint32_t s_cnt[SORT_WAVES][RADIX];
  __shared__ uint32_t s_wave[SORT_THREADS / 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int64_t base = int64_t(blockIdx.x) * (SORT_THREADS * ROUNDS);
  // wave w takes the keys [w*64*ROUNDS, (w+1)*64*ROUNDS) of the chunk in order
  const int64_t first = base + int64_t(wave) * (64 * ROUNDS) + lane;
  uint32_t k[ROUNDS], v[ROUNDS], rank[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int64_t i = first + r * 64;
    k[r] = i < n ? keys_in[i] : 0u;
    v[r] = i < n ? (vals_in ? vals_in[i] : uint32_t(i)) : 0u;
  }
  // each thread's digits: where the chunk's keys of a digit go
  uint32_t dbase[PER], tot = 0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    dbase[q] = totals[int(threadIdx.x) * PER + q];
    tot += dbase[q];
  }
#pragma unroll
  for (int w = 0; w < SORT_WAVES; ++w)
    for (int d = int(threadIdx.x); d < RADIX; d += SORT_THREADS) s_cnt[w][d] = 0;
  uint32_t all;
  uint32_t run = block_exclusive_scan(tot, all, s_wave);  // barriers after the clearing
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const uint32_t t = dbase[q];
    dbase[q] = run + rows[int64_t(int(threadIdx.x) * PER + q) * nchunks + blockIdx.x];
    run += t;
  }
  // ranks within the wave, in order (the LDS executes one wave's accesses in order)
  uint32_t* mine = s_cnt[wave];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const bool valid = first + r * 64 < n;
    const uint32_t digit = (k[r] >> shift) & (RADIX - 1);
    const uint64_t peers = match_digit<RB>(digit, valid);
    const uint32_t below = uint32_t(__popcll(peers & lanemask_lt()));
    uint32_t b = 0;
    if (valid && below == 0) {
      b = mine[digit];
      mine[digit] = b + uint32_t(__popcll(peers));
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the next round's counts after this one's
    rank[r] = uint32_t(__shfl(int(b), valid ? __ffsll((unsigned long long)peers) - 1 : lane, 64)) + below;
  }
  __syncthreads();
  // counts -> where each (digit, wave) starts
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int d = int(threadIdx.x) * PER + q;
    uint32_t at = dbase[q];
#pragma unroll
    for (int w = 0; w < SORT_WAVES; ++w) {
      const uint32_t c = s_cnt[w][d];
      s_cnt[w][d] = at;
      at += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    if (first + r * 64 < n) {
      const uint32_t pos = mine[(k[r] >> shift) & (RADIX - 1)] + rank[r];
      keys_out[pos] = k[r];
      vals_out[pos] = v[r];
    }
  }
}

// *out += sum of v[0..n): grid-stride partial sums, one atomic add per
// workgroup (integer, so the result does not depend on the order)
constexpr int SUM_THREADS = 256;
__global__ __launch_bounds__(SUM_THREADS) void k_sum_u32(const uint32_t* __restrict__ v, int64_t n,
                                                         uint32_t* __restrict__ out) {
  __shared__ uint32_t s[SUM_THREADS / 64];
  uint32_t acc = 0;
  for (int64_t i = int64_t(blockIdx.x) * SUM_THREADS + threadIdx.x; i < n; i += int64_t(gridDim.x) * SUM_THREADS)
    acc += v[i];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (int w = 0; w < SUM_THREADS / 64; ++w) t += s[w];
    if (t) atomicAdd(out, t);
  }
}

// Copy of n 16-byte words, one per thread (the form that measured fastest
// against grid-stride loops with several loads in flight per thread).
__global__ __launch_bounds__(256) void k_stream_copy(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                      int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

}  // namespace

void run_device_copy(tess_ctx* ctx, const void* src, void* dst, int64_t bytes) {
  const int64_t n = bytes / 16;
  if (n == 0) return;
  if (n > int64_t(UINT32_MAX) * 256) raise(TESS_ERR_ARGUMENT, "device copy larger than one launch");
  const int64_t blocks = ceil_div(n, int64_t(256));
  hipLaunchKernelGGL(k_stream_copy, dim3(unsigned(blocks)), dim3(256), 0, ctx->stream,
                     static_cast<const uint4*>(src), static_cast<uint4*>(dst), n);
  TESS_HIP(hipGetLastError());
}

void sum_u32(tess_ctx* ctx, const uint32_t* v, int64_t n, uint32_t* out) {
  TESS_HIP(hipMemsetAsync(out, 0, sizeof(uint32_t), ctx->stream));
  if (n <= 0) return;
  // about 8 values per thread, at most 512 workgroups
  const int64_t blocks = std::min<int64_t>(512, std::max<int64_t>(1, ceil_div(n, int64_t(SUM_THREADS) * 8)));
  hipLaunchKernelGGL(k_sum_u32, dim3(unsigned(blocks)), dim3(SUM_THREADS), 0, ctx->stream, v, n, out);
  TESS_HIP(hipGetLastError());
}

size_t scan_work_bytes(int64_t n) {
  size_t bytes = 256;
  for (int64_t m = ceil_div(n, SCAN_CHUNK); m > 1; m = ceil_div(m, SCAN_CHUNK)) bytes += size_t(m) * sizeof(uint32_t) + 256;
  return bytes;
}

void exclusive_scan_u32_ws(hipStream_t stream, uint8_t* tmp, uint32_t* data, int64_t n, uint32_t* total_dev) {
  if (n <= 0) return;
  const int64_t nchunks = ceil_div(n, SCAN_CHUNK);
  if (nchunks == 1) {
    hipLaunchKernelGGL(k_scan_apply, dim3(1), dim3(SCAN_THREADS), 0, stream, data, n, nullptr, total_dev);
    TESS_HIP(hipGetLastError());
    return;
  }
  // block sums live in a per-level slice of tmp (levels shrink by 4096x)
  struct Level {
    uint32_t* data;
    int64_t n;
  };
  Level lv[8];
  int nl = 0;
  lv[nl++] = {data, n};
  size_t off = 0;
  while (ceil_div(lv[nl - 1].n, SCAN_CHUNK) > 1) {
    const int64_t m = ceil_div(lv[nl - 1].n, SCAN_CHUNK);
    uint32_t* sums = reinterpret_cast<uint32_t*>(tmp + off);
    off += size_t(m) * sizeof(uint32_t) + 256;
    hipLaunchKernelGGL(k_scan_reduce, dim3(unsigned(m)), dim3(SCAN_THREADS), 0, stream, lv[nl - 1].data,
                       lv[nl - 1].n, sums);
    TESS_HIP(hipGetLastError());
    lv[nl++] = {sums, m};
  }
  // top level fits one chunk
  hipLaunchKernelGGL(k_scan_apply, dim3(1), dim3(SCAN_THREADS), 0, stream, lv[nl - 1].data, lv[nl - 1].n, nullptr,
                     nl == 1 ? total_dev : nullptr);
  TESS_HIP(hipGetLastError());
  for (int l = nl - 2; l >= 0; --l) {
    const int64_t m = ceil_div(lv[l].n, SCAN_CHUNK);
    hipLaunchKernelGGL(k_scan_apply, dim3(unsigned(m)), dim3(SCAN_THREADS), 0, stream, lv[l].data, lv[l].n,
                       lv[l + 1].data, l == 0 ? total_dev : nullptr);
    TESS_HIP(hipGetLastError());
  }
}

void exclusive_scan_u32(tess_ctx* ctx, uint32_t* data, int64_t n, uint32_t* total_dev) {
  if (n <= 0) {
    if (total_dev) TESS_HIP(hipMemsetAsync(total_dev, 0, sizeof(uint32_t), ctx->stream));
    return;
  }
  uint8_t* tmp = ceil_div(n, SCAN_CHUNK) > 1 ? static_cast<uint8_t*>(ctx->scan_tmp.get(scan_work_bytes(n))) : nullptr;
  exclusive_scan_u32_ws(ctx->stream, tmp, data, n, total_dev);
}

size_t sort_hist_words(int64_t n) {
  // a row of chunk counts and a total for each digit of the widest kind
  return (size_t(ceil_div(n, sort_chunk(n))) + 1) << RADIX_BITS_MAX;
}

namespace {
template <int RB, int ROUNDS>
void sort_pass(const SortWork& w, const uint32_t* kin, const uint32_t* vin, uint32_t* kout, uint32_t* vout, int64_t n,
               int shift, int64_t nchunks) {
  uint32_t* totals = w.hist + (nchunks << RB);
  hipLaunchKernelGGL((k_radix_hist<RB, ROUNDS>), dim3(unsigned(nchunks)), dim3(SORT_THREADS), 0, w.stream, kin, n, shift,
                     w.hist, nchunks);
  TESS_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_radix_rows, dim3(1u << RB), dim3(SORT_THREADS), 0, w.stream, w.hist, nchunks, totals);
  TESS_HIP(hipGetLastError());
  hipLaunchKernelGGL((k_radix_scatter<RB, ROUNDS>), dim3(unsigned(nchunks)), dim3(SORT_THREADS), 0, w.stream, kin, vin,
                     kout, vout, n, shift, w.hist, totals, nchunks);
  TESS_HIP(hipGetLastError());
}
}  // namespace

void radix_sort_pairs_ws(const SortWork& w, const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                         uint32_t* vals_out, int64_t n, int key_bits) {
  if (n <= 0) return;
  if (n > int64_t(UINT32_MAX)) raise(TESS_ERR_ARGUMENT, "radix sort: more than 2^32-1 elements");
  const int passes = sort_passes(key_bits, n), bits = sort_digit_bits(key_bits, n);
  const int64_t nchunks = ceil_div(n, sort_chunk(n));
  const bool large = n >= SORT_LARGE;
  // ping-pong so that the last pass writes (keys_out, vals_out)
  const uint32_t* kin = keys_in;
  const uint32_t* vin = vals_in;
  for (int p = 0; p < passes; ++p) {
    const bool to_out = ((passes - 1 - p) % 2) == 0;
    uint32_t* kout = to_out ? keys_out : w.keys_alt;
    uint32_t* vout = to_out ? vals_out : w.vals_alt;
    auto run = [&](auto rb) {
      constexpr int RB = decltype(rb)::value;
      if (large) sort_pass<RB, SORT_ROUNDS_LARGE>(w, kin, vin, kout, vout, n, p * bits, nchunks);
      else sort_pass<RB, SORT_ROUNDS_SMALL>(w, kin, vin, kout, vout, n, p * bits, nchunks);
    };
    if (bits == 8) run(std::integral_constant<int, 8>{});
    else if (bits == 9) run(std::integral_constant<int, 9>{});
    else run(std::integral_constant<int, 10>{});
    kin = kout;
    vin = vout;
  }
}

void radix_sort_pairs(tess_ctx* ctx, const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                      uint32_t* vals_out, int64_t n, int key_bits) {
  if (n <= 0) return;
  if (n > int64_t(UINT32_MAX)) raise(TESS_ERR_ARGUMENT, "radix sort: more than 2^32-1 elements");
  SortWork w;
  w.stream = ctx->stream;
  w.hist = ctx->hist.as<uint32_t>(sort_hist_words(n));
  w.keys_alt = ctx->keys_alt.as<uint32_t>(size_t(n));
  w.vals_alt = ctx->vals_alt.as<uint32_t>(size_t(n));
  radix_sort_pairs_ws(w, keys_in, vals_in, keys_out, vals_out, n, key_bits);
}

}  // namespace tess
