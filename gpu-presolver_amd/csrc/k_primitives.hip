// Primitive kernels of the presolve library: fills, scans, row activity,
// column max-abs, CSR statistics, mask compaction, LSD radix sort and the
// transpose built on it.  gfx950, wave64, 256-thread blocks.
#include <hip/hip_runtime.h>

#include <cmath>
#include <climits>
#include <cstdint>

#include "gp_device.hpp"
#include "gp_kernels.h"

using namespace gpdev;

namespace {

// ---------------------------------------------------------------- fills ----
template <class T>
__global__ void k_fill(T* dst, T v, int64_t n) {
  for (int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x)
    dst[i] = v;
}

__global__ void k_iota(int32_t* dst, int32_t n) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = i;
}

// ---------------------------------------------------------------- scans ----
// Reduce-then-scan: tile sums, one-block scan of tile sums, tile downsweep.
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;  // 2048

template <class In>
__device__ inline int32_t scan_value(const In* in, int64_t i);
template <>
__device__ inline int32_t scan_value<int32_t>(const int32_t* in, int64_t i) { return in[i]; }
template <>
__device__ inline int32_t scan_value<uint8_t>(const uint8_t* in, int64_t i) { return in[i] != 0 ? 1 : 0; }

template <class In>
__global__ __launch_bounds__(kBlock) void k_scan_tiles(const In* in, int64_t n, int32_t* tile_sums) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int32_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k)
    if (base + k < n) s += scan_value(in, base + k);
  int32_t total;
  (void)block_exclusive_sum(s, &total);
  if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// One block scans `tiles` tile sums in place (exclusive) and stores the grand total in out[n].
__global__ __launch_bounds__(kBlock) void k_scan_tile_sums(int32_t* tile_sums, int64_t tiles, int32_t* out_total) {
  __shared__ int32_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  for (int64_t b = 0; b < tiles; b += kBlock) {
    const int64_t i = b + threadIdx.x;
    const int32_t v = i < tiles ? tile_sums[i] : 0;
    int32_t total;
    const int32_t ex = block_exclusive_sum(v, &total);
    const int32_t carry = s_carry;
    if (i < tiles) tile_sums[i] = carry + ex;
    __syncthreads();
    if (threadIdx.x == 0) s_carry = carry + total;
    __syncthreads();
  }
  if (threadIdx.x == 0) *out_total = s_carry;
}

template <class In>
__global__ __launch_bounds__(kBlock) void k_scan_down(const In* in, int32_t* out, int64_t n, const int32_t* tile_prefix) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kScanTile + threadIdx.x * kScanItems;
  int32_t v[kScanItems];
  int32_t s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    v[k] = base + k < n ? scan_value(in, base + k) : 0;
    s += v[k];
  }
  int32_t total;
  int32_t run = block_exclusive_sum(s, &total) + tile_prefix[blockIdx.x];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    if (base + k < n) out[base + k] = run;
    run += v[k];
  }
}

// -------------------------------------------------------- row activity ----
// One thread per row, 256 consecutive rows per block.  The block's CSR
// segment is streamed through LDS in windows: all threads cooperatively load
// coalesced (col, a) entries, then gather the packed (l, u) pairs (all loads
// of a window issued before any is used), form the min/max terms and stage
// them; each thread then adds its own row's terms in CSR order, so every row
// sum has exactly the sequential rounding of the reference kernel
// (gpu_presolve_kernels.cu:18-66) for any row length.
// A row of more than kLongRow entries is left to act_long_row: its one
// thread would add thousands of terms from LDS while the other 255 wait, and
// neighbouring long rows (linking rows come last in most models) would queue
// in one block.  200 adjacent rows of 3,000 entries behind 80,000 short rows
// took 67 ms per call that way, and 42 us with a wave each.  The windows of a
// block with long rows skip them (their entries were read by the tile and
// by the wave before: 50,000 rows of 200 to 300 entries scattered among a million
// short ones 570 -> 386 us, 100,000 rows of 129 580 -> 395).
constexpr int kActRows = kBlock;
constexpr int kActCap = 2048;
constexpr int kActItems = kActCap / kBlock;

// (l, u) interleaved, so an activity term needs one 16-byte gather.
__global__ void k_pack_lu(const double* __restrict__ l, const double* __restrict__ u, int32_t n,
                          double2* __restrict__ lu) {
  const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) lu[j] = make_double2(l[j], u[j]);
}

// A term of the activity sums; b = (l, u) of the entry's column.
__device__ inline double act_min(double a, double2 b, bool on) { return on ? (a >= 0.0 ? a * b.x : a * b.y) : 0.0; }
__device__ inline double act_max(double a, double2 b, bool on) { return on ? (a >= 0.0 ? a * b.y : a * b.x) : 0.0; }

// One of the rows of more than kLongRow entries, by a wave; lane 0 adds the min
// terms and lane 1 the max terms.
static_assert(kWaves * 2 * kRowPitch <= kActCap + 16, "the long rows' terms fit the tile's LDS");

__device__ __forceinline__ void act_long_row(const int32_t* __restrict__ col_idx, const double* __restrict__ val,
                                             int64_t row, int32_t b, int32_t e, const double2* __restrict__ lu,
                                             double ztol, double* __restrict__ min_fin, double* __restrict__ max_fin,
                                             int32_t* __restrict__ neg_inf, int32_t* __restrict__ pos_inf,
                                             double* s_t) {
  int32_t ni = 0, pi = 0;
  const double acc = wave_row_sums<2, double2>(
      col_idx, val, b, e, s_t,
      [&](int32_t j, double a, bool in) { return lu[in && fabs(a) > ztol ? j : 0]; },
      [&](double a, double2 lub, bool in, double* t) {
        const bool on = in && fabs(a) > ztol;
        const double tn = act_min(a, lub, on), tx = act_max(a, lub, on);
        const bool fn = isfinite(tn), fx = isfinite(tx);
        ni += static_cast<int32_t>(__popcll(__ballot(!fn && tn < 0.0)));
        pi += static_cast<int32_t>(__popcll(__ballot(!fx && tx > 0.0)));
        t[0] = fn ? tn : 0.0;
        t[1] = fx ? tx : 0.0;
        return true;
      });
  const int lane = lane_id();
  if (lane == 0) {
    min_fin[row] = acc;
    neg_inf[row] = ni;
    pos_inf[row] = pi;
  } else if (lane == 1) {
    max_fin[row] = acc;
  }
}

// At least six waves a SIMD: the gathers of the tiles are bound by how many
// are in flight.
__global__ __launch_bounds__(kBlock, 6) void k_row_activity_lu(const int32_t* __restrict__ row_ptr,
                                                            const int32_t* __restrict__ col_idx,
                                                            const double* __restrict__ val, int32_t m,
                                                            const double2* __restrict__ lu, double ztol,
                                                            double* __restrict__ min_fin,
                                                            double* __restrict__ max_fin,
                                                            int32_t* __restrict__ neg_inf,
                                                            int32_t* __restrict__ pos_inf,
                                                            int32_t tiles) {
  // One term array (the min terms, then the max terms): with the runs 18 KB of
  // LDS per block, so LDS has room for eight blocks a CU (the registers for six).
  __shared__ __align__(16) double s_t[kActCap + 16];
  __shared__ int32_t s_run[kActRows], s_at[kActRows];
  if (static_cast<int32_t>(blockIdx.x) >= tiles) {
    double* s_row = s_t + (threadIdx.x >> 6) * 2 * kRowPitch;
    wave_long_rows(row_ptr, m, kLongRow, tiles, [&](int64_t row, int32_t b, int32_t e) {
      act_long_row(col_idx, val, row, b, e, lu, ztol, min_fin, max_fin, neg_inf, pos_inf, s_row);
    });
    return;
  }
  const int32_t r0 = static_cast<int32_t>(blockIdx.x) * kActRows;
  const int32_t rows = min(kActRows, m - r0);
  const int tid = threadIdx.x;
  const int32_t seg_b = row_ptr[r0], seg_e = row_ptr[r0 + rows];
  const int32_t row_b = row_ptr[r0 + min(tid, rows)], row_e = row_ptr[r0 + min(tid + 1, rows)];
  const bool is_long = row_e - row_b > kLongRow;
  // The windows go over the block's entries less those of its long rows: entry
  // t of them stands at t + seg_b, or where there are long rows at t + s_at of
  // the last run of rows between them that begins at or before t (s_run).
  int32_t my_b = row_b - seg_b, my_e = row_e - seg_b, total = seg_e - seg_b, runs = 0;
  if (__syncthreads_or(is_long) != 0) {
    const int32_t len = is_long ? 0 : row_e - row_b;
    my_b = block_exclusive_sum(len, &total);
    my_e = my_b + len;
    const bool head = tid < rows && !is_long && (tid == 0 || row_b - row_ptr[r0 + tid - 1] > kLongRow);
    const int32_t run = block_exclusive_sum(head ? 1 : 0, &runs);
    if (head) {
      s_run[run] = my_b;
      s_at[run] = row_b - my_b;
    }
    __syncthreads();
  }
  double mn = 0.0, mx = 0.0;
  int32_t ni = 0, pi = 0;
  for (int32_t w = 0, we; w < total; w = we) {
    we = total - w > kActCap ? w + kActCap : total;
    const int32_t rb = max(my_b, w), re = min(my_e, we);
    double a[kActItems];
    double2 b[kActItems];
    int32_t j[kActItems], pc[kActItems];
#pragma unroll
    for (int k = 0; k < kActItems; ++k) pc[k] = row_entry(w, we, tid + k * kBlock);
    if (runs > 0) {
#pragma unroll
      for (int k = 0; k < kActItems; ++k) {
        int lo = 0, hi = runs;  // s_run[lo] <= pc[k] < s_run[hi]
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (s_run[mid] <= pc[k]) lo = mid; else hi = mid;
        }
        pc[k] += s_at[lo];
      }
    } else {
#pragma unroll
      for (int k = 0; k < kActItems; ++k) pc[k] += seg_b;
    }
    // Every load is issued unconditionally (positions past the window read
    // its last entry and are discarded), so the compiler emits the 16 loads
    // back to back and then the 8 gathers, with no wait in between.
#pragma unroll
    for (int k = 0; k < kActItems; ++k) {
      a[k] = val[pc[k]];
      j[k] = col_idx[pc[k]];
    }
#pragma unroll
    for (int k = 0; k < kActItems; ++k) {
      if (tid + k * kBlock >= we - w) a[k] = 0.0;
      b[k] = lu[fabs(a[k]) > ztol ? j[k] : 0];
    }
    double tmx[kActItems];  // the max terms wait in registers while the min terms are summed
#pragma unroll
    for (int k = 0; k < kActItems; ++k) {
      const int t = tid + k * kBlock;
      const bool on = fabs(a[k]) > ztol;
      tmx[k] = act_max(a[k], b[k], on);
      if (t < we - w) s_t[t] = act_min(a[k], b[k], on);
    }
    __syncthreads();
    for (int32_t p = rb; p < re; ++p) {
      const double t = s_t[p - w];
      if (isfinite(t)) mn += t; else if (t < 0.0) ++ni;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kActItems; ++k) {
      const int t = tid + k * kBlock;
      if (t < we - w) s_t[t] = tmx[k];
    }
    __syncthreads();
    for (int32_t p = rb; p < re; ++p) {
      const double t = s_t[p - w];
      if (isfinite(t)) mx += t; else if (t > 0.0) ++pi;
    }
    if (we < total) __syncthreads();  // the next window restages
  }
  if (tid < rows && !is_long) {
    min_fin[r0 + tid] = mn;
    max_fin[r0 + tid] = mx;
    neg_inf[r0 + tid] = ni;
    pos_inf[r0 + tid] = pi;
  }
}

__global__ void k_col_max_abs(const int32_t* at_ptr, const double* at_val, int32_t n, double* out) {
  const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  double v = 0.0;
  for (int32_t p = at_ptr[j]; p < at_ptr[j + 1]; ++p) v = fmax(v, fabs(at_val[p]));
  out[j] = v;
}

__global__ void k_csr_stats(const int32_t* ptr, const int32_t* idx, const double* val, int32_t rows,
                            int32_t* nnz_out, uint8_t* empty_mask, uint8_t* singleton_mask,
                            int32_t* singleton_idx, double* singleton_val) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows) return;
  const int32_t b = ptr[i];
  const int32_t cnt = ptr[i + 1] - b;
  if (nnz_out) nnz_out[i] = cnt;
  if (empty_mask) empty_mask[i] = cnt == 0 ? 1 : 0;
  if (singleton_mask) singleton_mask[i] = cnt == 1 ? 1 : 0;
  if (singleton_idx) singleton_idx[i] = cnt == 1 ? idx[b] : -1;
  if (singleton_val) singleton_val[i] = cnt == 1 ? val[b] : 0.0;
}

// ---------------------------------------------------------- compaction ----
__device__ inline int find_row(const int32_t* s_ptr, int rows, int32_t p) {
  int lo = 0, hi = rows;  // s_ptr[lo] <= p < s_ptr[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (s_ptr[mid] <= p) lo = mid; else hi = mid;
  }
  return lo;
}

// ------------------------------------------------ decoupled look-back ----
constexpr uint64_t kLbSpinLimit = 1ull << 20;

__device__ inline uint64_t lb_word(uint32_t epoch, uint32_t flag, int32_t value) {
  return (static_cast<uint64_t>(epoch) << 34) | (static_cast<uint64_t>(flag) << 32) |
         static_cast<uint64_t>(static_cast<uint32_t>(value));
}

// Called by the first wave of the tile (all 64 lanes).  Publishes the tile's
// aggregate, then looks back over kLbWindow predecessors at a time, lane l
// watching kLbPerLane consecutive ones (nearest first): every lane waits for
// its predecessors' words, the nearest inclusive prefix in the window ends the
// walk, otherwise the window's aggregates are summed and the walk moves a
// window further back.  A wide window matters on this GPU: a status word
// written on one XCD is read through memory by the others, so each step
// costs a memory round trip, and the walk's depth is tiles / window.
// Publishes the tile's inclusive prefix and returns its exclusive prefix (in
// every lane).  Tile ids are tickets taken in dispatch order, so every
// predecessor is already running and each wait ends; the spin limit only
// guards a broken invariant (*error is set and the result is meaningless).
// The status words carry all the data a reader needs, so relaxed
// device-scope atomics suffice: acquire/release would add cache
// invalidation / write-back on every poll.
constexpr int kLbPerLane = 4;
constexpr int kLbWindow = 64 * kLbPerLane;

__device__ inline uint64_t lb_wait(const gpk_lookback& lb, int32_t j, int32_t first = 0) {
  if (j < first) return lb_word(lb.epoch, 2u, 0);  // before the chain's first tile: an inclusive prefix of 0
  uint64_t spins = 0;
  while (true) {
    const uint64_t w = __hip_atomic_load(lb.status + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((w >> 34) == lb.epoch && ((w >> 32) & 3u) != 0) return w;
    if (++spins > kLbSpinLimit) {
      __hip_atomic_store(lb.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return lb_word(lb.epoch, 2u, 0);
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

// `first`: the first tile of this tile's chain (several independent scans
// can share one launch and one status array, chain after chain in ticket
// order).
__device__ int32_t lb_exclusive(const gpk_lookback& lb, int32_t tile, int32_t aggregate, int32_t first = 0) {
  const int lane = lane_id();
  if (lane == 0)
    __hip_atomic_store(lb.status + tile, lb_word(lb.epoch, tile == first ? 2u : 1u, aggregate), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  if (tile == first) return 0;
  int32_t excl = 0;
  for (int32_t j0 = tile - 1;; j0 -= kLbWindow) {
    uint64_t w[kLbPerLane];
#pragma unroll
    for (int q = 0; q < kLbPerLane; ++q) w[q] = lb_wait(lb, j0 - lane * kLbPerLane - q, first);
    int q_incl = kLbPerLane;  // this lane's nearest inclusive prefix
#pragma unroll
    for (int q = kLbPerLane - 1; q >= 0; --q)
      if (((w[q] >> 32) & 3u) == 2u) q_incl = q;
    const uint64_t incl = __ballot(q_incl < kLbPerLane);
    const int first = incl ? __ffsll(static_cast<unsigned long long>(incl)) - 1 : 64;
    int32_t v = 0;
    if (lane <= first) {
      const int last_q = lane < first ? kLbPerLane - 1 : q_incl;
#pragma unroll
      for (int q = 0; q < kLbPerLane; ++q)
        if (q <= last_q) v += static_cast<int32_t>(static_cast<uint32_t>(w[q]));
    }
    excl += __shfl(wave_inclusive_sum(v), 63, 64);
    if (incl) break;
  }
  if (lane == 0)
    __hip_atomic_store(lb.status + tile, lb_word(lb.epoch, 2u, excl + aggregate), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  return excl;
}

__device__ inline int32_t lb_ticket(const gpk_lookback& lb) {
  __shared__ int32_t s_tile;
  if (threadIdx.x == 0) s_tile = atomicAdd(lb.ticket, 1);
  __syncthreads();
  return s_tile;
}

// Exclusive scan, 2048 items per tile (8 consecutive per thread); out[n] =
// total.
template <class In>
__global__ __launch_bounds__(kBlock) void k_scan_lb(const In* in, int32_t* out, int64_t n, gpk_lookback lb) {
  __shared__ int32_t s_wbase[kScanItems * kWaves];
  __shared__ int32_t s_excl;
  const int32_t tile = lb_ticket(lb);
  if (tile >= static_cast<int32_t>(gridDim.x)) {  // the ticket word was not zeroed
    if (threadIdx.x == 0) __hip_atomic_store(lb.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  // Striped items: element base + 256k + t belongs to thread t, so every load
  // and store instruction of a wave covers 64 consecutive elements.  Each
  // slice k is scanned across the wave with shuffles; the (slice, wave)
  // totals, in element order, give each wave-slice its offset in the tile.
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int64_t base = static_cast<int64_t>(tile) * kScanTile + tid;
  int32_t v[kScanItems], inc[kScanItems];
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k * kBlock;
    v[k] = i < n ? scan_value(in, i) : 0;
  }
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    inc[k] = wave_inclusive_sum(v[k]);
    if (lane == 63) s_wbase[k * kWaves + wave] = inc[k];
  }
  __syncthreads();
  if (tid < 64) {
    const int32_t c = tid < kScanItems * kWaves ? s_wbase[tid] : 0;
    const int32_t ci = wave_inclusive_sum(c);
    if (tid < kScanItems * kWaves) s_wbase[tid] = ci - c;
    const int32_t total = __shfl(ci, 63, 64);
    const int32_t e = lb_exclusive(lb, tile, total);
    if (tid == 0) s_excl = e;
    const int64_t tiles = (n + kScanTile - 1) / kScanTile;
    if (tid == 0 && tile == tiles - 1) out[n] = e + total;
  }
  __syncthreads();
  const int32_t excl = s_excl;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    const int64_t i = base + k * kBlock;
    const int32_t prefix = excl + s_wbase[k * kWaves + wave] + inc[k] - v[k];
    if (i < n) out[i] = prefix;
  }
}

// Bit b of the result: byte b of the word is not zero.
__device__ inline uint32_t nonzero_bytes(uint64_t x) {
  constexpr uint64_t k7f = 0x7f7f7f7f7f7f7f7full;
  const uint64_t hi = (((x & k7f) + k7f) | x) & ~k7f;  // bit 7 of every byte that is set
  return static_cast<uint32_t>(((hi >> 7) * 0x0102040810204080ull) >> 56);
}

// Eight mask entries from i on as bits (none past n); mask + i is 8-byte
// aligned when `aligned`.
__device__ inline uint32_t mask_bits8(const uint8_t* __restrict__ mask, int64_t i, int64_t n, bool aligned) {
  if (aligned && i + 8 <= n) return nonzero_bytes(*reinterpret_cast<const uint64_t*>(mask + i));
  uint32_t b = 0;
#pragma unroll 1
  for (int k = 0; k < 8 && i + k < n; ++k) b |= (mask[i + k] != 0 ? 1u : 0u) << k;
  return b;
}

// Set entries of mask[0, n), n a multiple of 16 and mask 16-byte aligned,
// counted by the thread's share of the block; four loads on their way at a
// time.
__device__ inline int32_t mask_count_share(const uint8_t* __restrict__ mask, int64_t n) {
  constexpr int U = 4;
  const ulonglong2* w = reinterpret_cast<const ulonglong2*>(mask);
  const int64_t words = n / 16;
  int32_t c = 0;
#pragma unroll 1
  for (int64_t i = threadIdx.x; i < words; i += U * kBlock) {
    ulonglong2 v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = i + k * kBlock < words ? w[i + k * kBlock] : make_ulonglong2(0, 0);
#pragma unroll
    for (int k = 0; k < U; ++k) c += __popc(nonzero_bytes(v[k].x)) + __popc(nonzero_bytes(v[k].y));
  }
  return c;
}

// The two keep maps of one plan application in one launch (build_old_to_new
// for rows and columns, gpu_presolve.cu:878-934): chains of 2048-item tiles,
// rows, then columns, eight consecutive items a thread (one 8-byte load of the
// mask, two 16-byte stores of the map; these kernels are bound by their chain
// of loads and by fetching their code, so both are kept short).  With l, the
// column tiles also mark the removed columns with a fixed interval, store how
// many each tile has and add them up.  A tile's offset comes from (kMode)
//   kMapRecount  the tile counting the chain's mask up to itself: one byte an
//                item, so at 262,144 items (GPK_MAP_RECOUNT_MAX) the last tile
//                reads 64 16-byte words a thread.  No tile waits for another,
//                as in look-back, whose status words cross the XCDs through
//                memory: 10.3 us on average over the applications of the 1M x
//                1.5M presolve, 13.5 before (8.7 at 12,000 x 23,000);
//   kMapCounts   the counts that k_apply_counts left, summed by the tile
//                (up to GPK_MAP_COUNT_TILES of them), 17.4 us for both launches
//                at 1M x 1.5M against 57 with look-back; at 200,000 items both
//                routes take 13 us;
//   kMapLookback decoupled look-back, for more tiles than that.
// The row pointers of the matrices to compact are walked on the way: entry
// q << chunk_shift of A lies in row a_chunk[q] (and of AT in row at_chunk[q]).
enum { kMapLookback = 0, kMapRecount = 1, kMapCounts = 2 };

__global__ __launch_bounds__(kBlock) void k_apply_counts(gpk_apply_maps_args a, int32_t row_tiles, int32_t aligned) {
  const int32_t tile = static_cast<int32_t>(blockIdx.x);
  const bool rows = tile < row_tiles;
  const int64_t i0 = static_cast<int64_t>(rows ? tile : tile - row_tiles) * kScanTile + 8 * threadIdx.x;
  int32_t total;
  (void)block_exclusive_sum(__popc(mask_bits8(rows ? a.keep_row : a.keep_col, i0, rows ? a.m : a.n, aligned != 0)),
                            &total);
  if (threadIdx.x == 0) a.tile_counts[tile] = total;
}

template <int kMode>
__global__ __launch_bounds__(kBlock) void k_apply_maps(gpk_apply_maps_args a, int32_t row_tiles, int32_t aligned,
                                                       gpk_lookback lb) {
  __shared__ int32_t s_excl;
  __shared__ __align__(8) uint8_t s_bits[kBlock];
  __shared__ int32_t s_first[kBlock / 8];
  int32_t tile = static_cast<int32_t>(blockIdx.x);
  if constexpr (kMode == kMapLookback) {
    tile = lb_ticket(lb);
    if (tile >= static_cast<int32_t>(gridDim.x)) {  // the ticket word was not zeroed
      if (threadIdx.x == 0) __hip_atomic_store(lb.error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
  }
  const bool rows = tile < row_tiles;
  const int32_t first = rows ? 0 : row_tiles, last = rows ? row_tiles - 1 : static_cast<int32_t>(gridDim.x) - 1;
  const int64_t n = rows ? a.m : a.n;
  const uint8_t* mask = rows ? a.keep_row : a.keep_col;
  const int32_t* ptr = rows ? a.a_ptr : a.at_ptr;
  const int tid = threadIdx.x;
  const int64_t base = static_cast<int64_t>(tile - first) * kScanTile, i0 = base + 8 * tid;
  const int64_t i1 = i0 + 8 < n ? i0 + 8 : n;
  const bool any = i0 < n;
  const int32_t pb = ptr != nullptr && any ? ptr[i0] : 0, pe = ptr != nullptr && any ? ptr[i1] : 0;
  const uint32_t bits = mask_bits8(mask, i0, n, aligned != 0);
  int32_t share = 0;  // of the set entries before the tile
  if constexpr (kMode == kMapRecount) {
    share = mask_count_share(mask, base);
  } else if constexpr (kMode == kMapCounts) {
#pragma unroll 1
    for (int32_t t = first + tid; t < tile; t += kBlock) share += a.tile_counts[t];
  }
  int32_t total, excl = 0;
  const int32_t before = block_exclusive_sum(__popc(bits), &total);  // in the tile
  if constexpr (kMode == kMapLookback) {
    if (tid < 64) {
      const int32_t e = lb_exclusive(lb, tile, total, first);
      if (tid == 0) s_excl = e;
    }
    __syncthreads();
    excl = s_excl;
  } else {
    (void)block_exclusive_sum(share, &excl);
  }
  if (tid == 0 && tile == last) a.counts[rows ? 0 : 1] = excl + total;
  if (ptr != nullptr) {
    // Chunk starts among the thread's entries: each lies in the last row that
    // begins at or before it.
    int32_t* chunk_row = rows ? a.a_chunk : a.at_chunk;
    const int shift = a.chunk_shift;
    int64_t r = i0;
#pragma unroll 1
    for (int64_t q = (pb + (int64_t{1} << shift) - 1) >> shift; q << shift < pe && q < a.chunks; ++q) {
#pragma unroll 1
      while (r + 1 < i1 && ptr[r + 1] <= q << shift) ++r;
      chunk_row[q] = static_cast<int32_t>(r);
    }
    // Chunks that start before the first row's entries or past the last row's.
    const int64_t round = (int64_t{1} << shift) - 1;
    if (tile == first)
      for (int64_t q = tid, lead = (ptr[0] + round) >> shift; q < lead && q < a.chunks; q += kBlock) chunk_row[q] = 0;
    if (tile == last)
      for (int64_t q = ((ptr[n] + round) >> shift) + tid; q <= a.chunks; q += kBlock)
        chunk_row[q] = static_cast<int32_t>(n) - 1;
  }
  if (!rows && a.l != nullptr) {
    // Removed, both bounds finite and within 1e-9 of each other.
    uint32_t fixed = 0;
    if (bits != 255u && any) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int64_t i = i0 + k < n ? i0 + k : n - 1;
        const double lo = a.l[i], hi = a.u[i];
        fixed |= (isfinite(lo) && isfinite(hi) && fabs(lo - hi) <= 1.0e-9 ? 1u : 0u) << k;
      }
      fixed &= ~bits & (i1 - i0 == 8 ? 255u : (1u << (i1 - i0)) - 1u);
    }
    if (i1 - i0 == 8) {  // the mask is the library's own (aligned)
      uint64_t bytes = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) bytes |= static_cast<uint64_t>((fixed >> k) & 1u) << (8 * k);
      *reinterpret_cast<uint64_t*>(a.fixed_mask + i0) = bytes;
    } else {
#pragma unroll 1
      for (int64_t i = i0; i < i1; ++i) a.fixed_mask[i] = (fixed >> (i - i0)) & 1u;
    }
    int32_t c;
    (void)block_exclusive_sum(__popc(fixed), &c);
    if (tid == 0) {
      a.fixed_tiles[tile - first] = c;
      if (c != 0) atomicAdd(&a.counts[2], c);
    }
  }
  int32_t* out = rows ? a.row_map : a.col_map;
  int32_t v[8], run = excl + before;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    v[k] = (bits >> k) & 1u ? run : -1;
    run += (bits >> k) & 1u;
  }
  if (i1 - i0 == 8) {  // the maps are the library's own (16-byte aligned)
    reinterpret_cast<int4*>(out + i0)[0] = make_int4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<int4*>(out + i0)[1] = make_int4(v[4], v[5], v[6], v[7]);
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (i0 + k < n) out[i0 + k] = v[k];
  }
  gpk_rank_word* rank = rows ? a.row_rank : a.col_rank;
  if (rank == nullptr) return;
  // Eight threads make a rank word: kept bits and the new index of the first
  // kept one.
  s_bits[tid] = static_cast<uint8_t>(bits);
  if ((tid & 7) == 0) s_first[tid >> 3] = excl + before;
  __syncthreads();
  if (tid < kBlock / 8 && base + 64 * tid < n) {
    const uint64_t b = reinterpret_cast<const uint64_t*>(s_bits)[tid];
    gpk_rank_word w;
    w.bits = b;
    w.base = b ? s_first[tid] : 0;
    w.pad = 0;
    rank[(base >> 6) + tid] = w;
  }
}

// Exclusive scan (out[n] = total) of a 16-byte aligned mask of up to
// GPK_MAP_RECOUNT_MAX entries, a tile's offset as in k_apply_maps with
// kMapRecount: 5.1 us at 23,000 entries against 9.9 with look-back, and 4.4 at
// 12,000 against 9.4 in one workgroup.  `out` holds n + 1 entries and may
// start anywhere.
__global__ __launch_bounds__(kBlock) void k_mask_scan(const uint8_t* __restrict__ mask, int32_t* __restrict__ out,
                                                      int32_t n) {
  const int tid = threadIdx.x;
  const int32_t base = static_cast<int32_t>(blockIdx.x) * kScanTile, i0 = base + 8 * tid;
  const uint32_t bits = mask_bits8(mask, i0, n, true);
  const int32_t share = mask_count_share(mask, base);
  int32_t total, excl;
  int32_t run = block_exclusive_sum(__popc(bits), &total);
  (void)block_exclusive_sum(share, &excl);
  run += excl;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    if (i0 + k < n) out[i0 + k] = run;
    run += (bits >> k) & 1u;
  }
  if (blockIdx.x == gridDim.x - 1 && tid == 0) out[n] = excl + total;
}

// Small scans in one workgroup (no tickets, no look-back): 1024 threads walk
// the array in chunks of 8192 with a running carry, each chunk striped and
// scanned like a look-back tile.  Same outputs as k_scan_lb.
constexpr int kSmallBlock = 1024;
constexpr int64_t kSmallScanMax = 16384;

template <class In>
__global__ __launch_bounds__(kSmallBlock) void k_scan_small(const In* in, int32_t* out, int64_t n) {
  constexpr int kWaves = kSmallBlock / 64;
  constexpr int kSlots = kScanItems * kWaves;  // 128
  __shared__ int32_t s_w[kSlots];
  __shared__ int32_t s_total;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  int32_t carry = 0;
  for (int64_t c = 0; c < n; c += static_cast<int64_t>(kScanItems) * kSmallBlock) {
    int32_t v[kScanItems], inc[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      const int64_t i = c + k * kSmallBlock + tid;
      v[k] = i < n ? scan_value(in, i) : 0;
    }
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      inc[k] = wave_inclusive_sum(v[k]);
      if (lane == 63) s_w[k * kWaves + wave] = inc[k];
    }
    __syncthreads();
    if (tid < 64) {  // exclusive prefix of the 128 (slice, wave) totals, two per lane
      const int32_t a = s_w[2 * tid], b = s_w[2 * tid + 1];
      const int32_t pi = wave_inclusive_sum(a + b);
      s_w[2 * tid] = pi - a - b;
      s_w[2 * tid + 1] = pi - b;
      if (tid == 63) s_total = pi;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
      const int64_t i = c + k * kSmallBlock + tid;
      const int32_t prefix = carry + s_w[k * kWaves + wave] + inc[k] - v[k];
      if (i < n) out[i] = prefix;
    }
    carry += s_total;
    __syncthreads();  // s_w and s_total are rewritten by the next chunk
  }
  if (tid == 0) out[n] = carry;
}

// Compaction (gpu_presolve.cu:1881-1978) over chunks of entries, whatever the
// rows: a tile of 256 rows gives a block-structured LP's 200 linking rows of
// 3,000 entries to one block (1.58 ms a map pass, 0.59 ms a write pass on
// 80,200 x 120,000; 14.5 and 15.4 us by chunks), and the popular columns of AT
// to few (121 us the map pass of the pair on 1M x 1.5M; 67 by chunks).
//   k_compact_map    maps every entry once (row kept and column rank, one
//     cache-resident rank gather per entry; with no rank words, when no column
//     is dropped, the column keeps its index), stores the new column index or
//     -1 per entry, the chunk's kept entries as words of bits with their
//     prefix sums, and its kept count;
//   k_compact_write  moves the chunk's kept entries to their places (chunk
//     offset, word prefix, bits below), staged in LDS for coalesced stores;
//     further blocks turn every kept row's first entry into its row pointer
//     through the same words, and gather the LP's vectors on the way.
// A chunk's offset is the sum of the counts before it: added up by each block
// from the raw counts (up to GPK_COMPACT_COUNT_CHUNKS a side), or scanned by a
// launch in between.
// kI entries a thread: 8 (chunks of 2048) on large matrices, 2 (chunks of 512)
// up to GPK_COMPACT_SMALL_NNZ entries, where the chip is far from full and a
// block's own chain of loads is what counts (26,000 entries: 4.2 us a map pass
// against 8.7 with 2048).

// One 16-byte load of the word, then the rank; -1 when entry j is dropped.
__device__ inline uint4 rank_word(const gpk_rank_word* __restrict__ rank, int32_t j) {
  return *reinterpret_cast<const uint4*>(rank + (j >> 6));
}
__device__ inline int32_t rank_of(uint4 w, int32_t j) {
  const uint64_t bits = static_cast<uint64_t>(w.x) | (static_cast<uint64_t>(w.y) << 32);
  const uint64_t bit = 1ull << (j & 63);
  const int32_t r = static_cast<int32_t>(w.z) + static_cast<int32_t>(__popcll(bits & (bit - 1)));
  return (bits & bit) ? r : -1;
}

// Sets bits [b, e) of an LDS bitmap.
__device__ inline void set_bits(uint32_t* words, int b, int e) {
  for (int w = b >> 5; w <= (e - 1) >> 5; ++w) {
    const int lo = max(b - 32 * w, 0), hi = min(e - 32 * w, 32);
    atomicOr(&words[w], (hi == 32 ? ~0u : (1u << hi) - 1u) & ~((1u << lo) - 1u));
  }
}

// Rows of a chunk (its entries' rows and the empty ones between) up to which
// the block marks kept rows in the bitmap; past that every entry looks its row
// up by bisection, so a chunk that spans a million empty rows costs 20 loads
// an entry instead of 4,000 a thread.
constexpr int kCompMarkRows = 8192;

template <int kI>
__device__ __forceinline__ void compact_map_chunk(int32_t q, const gpk_compact_side& s, int32_t* __restrict__ chunk_cnt,
                                                  int32_t* __restrict__ kept_total) {
  constexpr int kChunk = kBlock * kI, kWords = kChunk / 64, kAhead = 2;
  __shared__ uint32_t s_live[2 * kWords];
  __shared__ uint64_t s_mask[kWords];
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int32_t c0 = q * kChunk;
  const int32_t c1 = min(s.nnz - c0, kChunk);  // entries of the chunk
  const int32_t r_lo = s.chunk_row[q], r_hi = s.chunk_row[q + 1];
  int32_t cj[kI];
#pragma unroll
  for (int k = 0; k < kI; ++k) cj[k] = s.idx[c0 + min(k * kBlock + tid, c1 - 1)];
  if (tid < 2 * kWords) s_live[tid] = 0;
  if (r_hi - r_lo < kCompMarkRows) {
    // The first rows' pointers and fates are loaded together.
    int32_t b[kAhead], e[kAhead], to[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int32_t r = min(r_lo + tid + k * kBlock, r_hi);
      b[k] = s.ptr[r];
      e[k] = s.ptr[r + 1];
      to[k] = s.row_map[r];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int lo = max(b[k] - c0, 0), hi = min(e[k] - c0, c1);
      if (r_lo + tid + k * kBlock <= r_hi && lo < hi && to[k] >= 0) set_bits(s_live, lo, hi);
    }
    for (int32_t r = r_lo + tid + kAhead * kBlock; r <= r_hi; r += kBlock) {
      const int lo = max(s.ptr[r] - c0, 0), hi = min(s.ptr[r + 1] - c0, c1);
      if (lo < hi && s.row_map[r] >= 0) set_bits(s_live, lo, hi);
    }
  } else {
    __syncthreads();
    for (int k = 0; k < kI; ++k) {
      const int32_t p = k * kBlock + tid;
      if (p >= c1) break;
      int32_t lo = r_lo, hi = r_hi + 1;  // ptr[lo] <= c0 + p < ptr[hi]
      while (hi - lo > 1) {
        const int32_t mid = lo + (hi - lo) / 2;
        if (s.ptr[mid] <= c0 + p) lo = mid; else hi = mid;
      }
      const bool held = s.ptr[lo] <= c0 + p && c0 + p < s.ptr[lo + 1];
      if (held && s.row_map[lo] >= 0) atomicOr(&s_live[p >> 5], 1u << (p & 31));
    }
  }
  __syncthreads();
  // Slice k of a wave is word k * kWaves + wave of the chunk.
  bool live[kI];
  uint4 w[kI];
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int p = k * kBlock + tid;
    live[k] = (s_live[p >> 5] >> (p & 31)) & 1u;
  }
  if (s.col_rank != nullptr) {
#pragma unroll
    for (int k = 0; k < kI; ++k) w[k] = rank_word(s.col_rank, live[k] ? cj[k] : 0);
  }
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int p = k * kBlock + tid;
    const int32_t jn = !live[k] ? -1 : s.col_rank != nullptr ? rank_of(w[k], cj[k]) : cj[k];
    if (p < c1) s.jn[c0 + p] = jn;
    const uint64_t kept = __ballot(jn >= 0);  // entries past the chunk are not live
    if (lane == 0) s_mask[k * kWaves + wave] = kept;
  }
  __syncthreads();
  if (tid < 64) {
    const uint64_t bits = tid < kWords ? s_mask[tid] : 0ull;
    const int32_t c = static_cast<int32_t>(__popcll(bits));
    const int32_t inc = wave_inclusive_sum(c);
    if (tid < kWords) {
      s.mask[static_cast<int64_t>(q) * kWords + tid] = bits;
      s.word_pre[static_cast<int64_t>(q) * kWords + tid] = inc - c;
    }
    if (tid == 63) {
      chunk_cnt[q] = inc;
      if (kept_total != nullptr && inc != 0) atomicAdd(kept_total, inc);  // integer: order-free
    }
  }
}

// A's chunks, then those of its transpose, compacted with the same maps.
template <int kI>
__global__ __launch_bounds__(kBlock) void k_compact_map(gpk_compact_side a, gpk_compact_side t, int32_t chunks_a,
                                                        int32_t* __restrict__ chunk_cnt,
                                                        int32_t* __restrict__ kept_total) {
  const int32_t b = static_cast<int32_t>(blockIdx.x);
  if (b < chunks_a) compact_map_chunk<kI>(b, a, chunk_cnt, kept_total);
  else compact_map_chunk<kI>(b - chunks_a, t, chunk_cnt + chunks_a, nullptr);
}

// The vector gathers of one plan application: c, l, u, the column
// reduced-to-original map and the record of a removed fixed column for column
// i (fixed_at: its place among them, or -1); AL, AU and the row map for row i
// (dst[map[i]] = src[i] for map[i] >= 0; a null destination is skipped).
__device__ __forceinline__ void gather_col(const gpk_apply_gathers_args& a, int32_t i, int32_t j, int32_t fixed_at) {
  if (j >= 0) {
    a.c_out[j] = a.c_in[i];
    a.l_out[j] = a.l_in[i];
    a.u_out[j] = a.u_in[i];
    if (a.col_r2o_out) a.col_r2o_out[j] = a.col_r2o_in[i];
  } else if (fixed_at >= 0) {
    a.fixed_idx[fixed_at] = a.col_r2o_in[i];
    a.fixed_val[fixed_at] = 0.5 * (a.l_in[i] + a.u_in[i]);
  }
}
__device__ __forceinline__ void gather_row(const gpk_apply_gathers_args& a, int32_t i, int32_t r) {
  if (r < 0) return;
  a.al_out[r] = a.al_in[i];
  a.au_out[r] = a.au_in[i];
  if (a.row_r2o_out) a.row_r2o_out[r] = a.row_r2o_in[i];
}

// The column's place among the removed fixed columns (-1: not one), for the
// kBlock columns from block * kBlock on: the tiles' counts before its map
// tile, the mask up to the block, then the block's own prefix.
static_assert(kScanTile % kBlock == 0, "a block of columns lies in one map tile");
__device__ __forceinline__ int32_t fixed_place(const gpk_apply_gathers_args& a, int32_t block) {
  const int tid = threadIdx.x;
  const int64_t at = static_cast<int64_t>(block) * kBlock;
  const int32_t j0 = at < a.n ? static_cast<int32_t>(at) : a.n, tile = j0 / kScanTile;  // past the columns: none
  const int32_t f = at + tid < a.n ? a.fixed_mask[at + tid] : 0;
  int32_t c = 0, before, mine;
#pragma unroll 1
  for (int32_t t = tid; t < tile; t += kBlock) c += a.fixed_tiles[t];
#pragma unroll 1
  for (int32_t j = tile * kScanTile + tid; j < j0; j += kBlock) c += a.fixed_mask[j];
  (void)block_exclusive_sum(c, &before);
  const int32_t excl = block_exclusive_sum(f, &mine);
  return f ? before + excl : -1;
}

__global__ __launch_bounds__(kBlock) void k_apply_gathers(gpk_apply_gathers_args a) {
  const int32_t b = static_cast<int32_t>(blockIdx.x);
  const int64_t i = static_cast<int64_t>(b) * kBlock + threadIdx.x;
  const int32_t at = a.fixed_mask != nullptr ? fixed_place(a, b) : -1;
  if (i < a.n) gather_col(a, static_cast<int32_t>(i), a.col_map[i], at);
  if (i < a.m) gather_row(a, static_cast<int32_t>(i), a.row_map[i]);
}

// The kept entries of chunk q; off: the side's raw chunk counts (from_counts)
// or their exclusive scan (whose first word is subtracted: a segment of a
// longer scan).
template <int kI>
__device__ __forceinline__ void compact_write_chunk(int32_t q, bool from_counts, const gpk_compact_side& s,
                                                    const int32_t* __restrict__ off, double* s_oval, int32_t* s_oidx) {
  constexpr int kChunk = kBlock * kI, kWords = kChunk / 64;
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
  const int32_t c0 = q * kChunk;
  const int32_t c1 = min(s.nnz - c0, kChunk);
  const int64_t word0 = static_cast<int64_t>(q) * kWords + wave;
  int32_t jn[kI], pre[kI];
  uint64_t bits[kI];
  double v[kI];
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    const int32_t p = c0 + min(k * kBlock + tid, c1 - 1);
    jn[k] = s.jn[p];
    v[k] = s.val[p];
    bits[k] = s.mask[word0 + k * kWaves];
    pre[k] = s.word_pre[word0 + k * kWaves];
  }
  int32_t base, total;
  if (from_counts) {
    int32_t c = 0;
    total = off[q];
    for (int32_t i = tid; i < q; i += kBlock) c += off[i];
    (void)block_exclusive_sum(c, &base);
  } else {
    const int32_t first = off[0];
    base = off[q] - first;
    total = off[q + 1] - first - base;
  }
  if (total == 0) return;
  const uint64_t below = lanemask_lt(lane);
#pragma unroll
  for (int k = 0; k < kI; ++k) {
    if ((bits[k] >> lane) & 1ull) {
      const int32_t pos = pre[k] + static_cast<int32_t>(__popcll(bits[k] & below));
      s_oidx[pos] = jn[k];
      s_oval[pos] = v[k];
    }
  }
  __syncthreads();
  for (int t = tid; t < total; t += kBlock) {
    s.out_idx[base + t] = s_oidx[t];
    s.out_val[base + t] = s_oval[t];
  }
}

// The row pointers of kBlock old rows; returns the thread's new row (-1:
// dropped or past the end).
template <int kI>
__device__ __forceinline__ int32_t compact_row(int32_t block, int32_t chunks, bool from_counts,
                                               const gpk_compact_side& s, const int32_t* __restrict__ off,
                                               int32_t* s_off) {
  constexpr int kChunk = kBlock * kI;
  const int tid = threadIdx.x;
  const int64_t r = static_cast<int64_t>(block) * kBlock + tid;
  const int32_t nr = r < s.m_old ? s.row_map[r] : -1;
  const int32_t p = r < s.m_old ? s.ptr[r] : s.nnz;
  int32_t local = 0;
  if (p < s.nnz)
    local = s.word_pre[p >> 6] + static_cast<int32_t>(__popcll(s.mask[p >> 6] & ((1ull << (p & 63)) - 1ull)));
  int32_t first = 0;  // the word subtracted from an offset
  if (from_counts) {
    constexpr int kPer = GPK_COMPACT_COUNT_CHUNKS / kBlock;
    int32_t c[kPer], sum = 0, all;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      c[k] = tid * kPer + k < chunks ? off[tid * kPer + k] : 0;
      sum += c[k];
    }
    int32_t run = block_exclusive_sum(sum, &all);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      s_off[tid * kPer + k] = run;
      run += c[k];
    }
    if (tid == 0) s_off[GPK_COMPACT_COUNT_CHUNKS] = all;
    __syncthreads();
  } else {
    first = off[0];
  }
  auto offset = [&](int32_t q) {
    return from_counts ? s_off[q < chunks ? q : GPK_COMPACT_COUNT_CHUNKS] : off[q] - first;
  };
  // empty rows at the end start at the kept count
  if (nr >= 0) s.out_ptr[nr] = offset(p < s.nnz ? p / kChunk : chunks) + local;
  if (block == 0 && tid == 0) s.out_ptr[s.m_new] = offset(chunks);
  return nr;
}

// Blocks: A's chunks, AT's chunks, A's rows, AT's rows.
template <int kI>
__global__ __launch_bounds__(kBlock) void k_compact_write(gpk_compact_side a, gpk_compact_side t, int32_t chunks_a,
                                                          int32_t chunks_t, int32_t row_blocks_a,
                                                          const int32_t* __restrict__ off, int32_t from_counts,
                                                          gpk_apply_gathers_args g) {
  constexpr int kChunk = kBlock * kI;
  constexpr int kLds = kChunk * 12 > (GPK_COMPACT_COUNT_CHUNKS + 1) * 4 ? kChunk * 12 : (GPK_COMPACT_COUNT_CHUNKS + 2) * 4;
  __shared__ __align__(16) char s_buf[kLds];
  double* s_oval = reinterpret_cast<double*>(s_buf);
  int32_t* s_oidx = reinterpret_cast<int32_t*>(s_buf + sizeof(double) * kChunk);
  int32_t* s_off = reinterpret_cast<int32_t*>(s_buf);
  int32_t b = static_cast<int32_t>(blockIdx.x);
  if (b < chunks_a) {
    compact_write_chunk<kI>(b, from_counts != 0, a, off, s_oval, s_oidx);
    return;
  }
  b -= chunks_a;
  if (b < chunks_t) {
    compact_write_chunk<kI>(b, from_counts != 0, t, off + chunks_a, s_oval, s_oidx);
    return;
  }
  b -= chunks_t;
  const bool rows = b < row_blocks_a;
  if (!rows) b -= row_blocks_a;
  const int32_t to = rows ? compact_row<kI>(b, chunks_a, from_counts != 0, a, off, s_off)
                          : compact_row<kI>(b, chunks_t, from_counts != 0, t, off + chunks_a, s_off);
  const int64_t i = static_cast<int64_t>(b) * kBlock + threadIdx.x;
  if (rows) {
    if (g.m > 0) gather_row(g, static_cast<int32_t>(i), to);
  } else if (g.n > 0) {
    const int32_t at = g.fixed_mask != nullptr ? fixed_place(g, b) : -1;
    if (i < g.n) gather_col(g, static_cast<int32_t>(i), to, at);
  }
}

__global__ void k_mail(const uint32_t* __restrict__ src, int32_t words, uint32_t* mail, uint32_t seq) {
  const int t = threadIdx.x;
  if (t < words) mail[4 + t] = src[t];
  __threadfence_system();
  __syncthreads();
  if (t == 0) *reinterpret_cast<volatile uint32_t*>(mail) = seq;
}

struct CopyList {
  gpk_copy_seg seg[GPK_COPY_MAX];
};

template <class U>
__device__ inline void copy_units(const gpk_copy_seg& g) {
  const int64_t units = g.bytes / static_cast<int64_t>(sizeof(U));
  U* d = static_cast<U*>(g.dst);
  const U* src = static_cast<const U*>(g.src);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < units; i += stride)
    d[i] = src ? src[i] : U{};
}

__global__ __launch_bounds__(kBlock) void k_copy_many(CopyList list) {
  const gpk_copy_seg g = list.seg[blockIdx.y];
  const uint64_t a = reinterpret_cast<uint64_t>(g.dst) | reinterpret_cast<uint64_t>(g.src) |
                     static_cast<uint64_t>(g.bytes);
  if ((a & 15u) == 0) copy_units<uint4>(g);
  else if ((a & 7u) == 0) copy_units<uint2>(g);
  else if ((a & 3u) == 0) copy_units<uint32_t>(g);
  else copy_units<uint8_t>(g);
}

__global__ void k_gather_i32(const int32_t* map, int32_t n_old, const int32_t* src, int32_t* dst) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_old) return;
  const int32_t t = map[i];
  if (t >= 0) dst[t] = src[i];
}

// ------------------------------------------------------------ radix sort ----
// Stable LSD radix sort, 8-bit digits.  Tile = 2048 keys; wave w of a block
// owns the contiguous keys [w*512, w*512+512) of the tile, read 64 at a time.
// Per 64-key step the lanes holding the same digit are found with eight
// ballots, ranked by lane order, and appended to a per-wave digit counter in
// LDS; digit offsets across waves and tiles come from the global histogram
// scan, so equal digits keep their input order.  The ranked tile is staged
// in LDS in digit order and stored run by run.
constexpr int kRsTile = 2048;
constexpr int kRsWaveItems = 512;
constexpr int kRsWaves = kBlock / 64;
// Up to this many tiles, each scatter block reads the whole histogram
// (256 x tiles words) instead of waiting for a scan launch.
constexpr int kRsHistTilesMax = 64;

// kTileMajor: one tile's 256 counts together (for k_radix_scatter from the raw
// histogram), else one digit's tiles together (for the scan).
template <class K, bool kTileMajor>
__global__ __launch_bounds__(kBlock) void k_radix_hist(const K* __restrict__ keys, int32_t n, int shift,
                                                      int32_t tiles, int32_t* __restrict__ hist) {
  __shared__ int32_t s_h[256];
  s_h[threadIdx.x] = 0;
  __syncthreads();
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kRsTile;
  for (int k = 0; k < kRsTile / kBlock; ++k) {
    const int64_t e = base + k * kBlock + threadIdx.x;
    if (e < n) atomicAdd(&s_h[static_cast<int>((keys[e] >> shift) & 255u)], 1);
  }
  __syncthreads();
  hist[kTileMajor ? static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x
                  : static_cast<int64_t>(threadIdx.x) * tiles + blockIdx.x] = s_h[threadIdx.x];
}

// kFromHist: offs is the raw histogram (tile-major) and every block derives its
// own digit offsets from it, 16 tiles' loads on their way at a time (for few
// tiles, this saves the separate scan launch; one load after the other took
// 18 us at 59 tiles, 11 now); otherwise offs is the scanned histogram
// (digit-major).
template <class K, bool kFromHist>
__global__ __launch_bounds__(kBlock) void k_radix_scatter(const K* __restrict__ kin, const int32_t* __restrict__ vin,
                                                         K* __restrict__ kout, int32_t* __restrict__ vout,
                                                         int32_t n, int shift, int32_t tiles,
                                                         const int32_t* __restrict__ offs) {
  __shared__ int32_t s_cnt[kRsWaves][256];
  __shared__ int32_t s_off[kRsWaves][256];
  __shared__ int32_t s_base[256];
  __shared__ int32_t s_start[256];
  __shared__ int32_t s_wsum[kRsWaves];
  __shared__ K s_key[kRsTile];
  __shared__ int32_t s_val[kRsTile];
  const int tid = threadIdx.x;
  for (int i = tid; i < kRsWaves * 256; i += kBlock) s_cnt[i >> 8][i & 255] = 0;
  if (kFromHist) {
    static_assert(kBlock == 256, "one thread per digit");
    constexpr int U = 16;
    int32_t total = 0, before = 0;
#pragma unroll 1
    for (int32_t t0 = 0; t0 < tiles; t0 += U) {
      int32_t h[U];
#pragma unroll
      for (int k = 0; k < U; ++k) h[k] = t0 + k < tiles ? offs[(t0 + k) * 256 + tid] : 0;
#pragma unroll
      for (int k = 0; k < U; ++k) {
        total += h[k];
        before += t0 + k < static_cast<int32_t>(blockIdx.x) ? h[k] : 0;
      }
    }
    const int32_t inc = wave_inclusive_sum(total);
    if ((tid & 63) == 63) s_wsum[tid >> 6] = inc;
    __syncthreads();
    int32_t wbase = 0;
    for (int w = 0; w < (tid >> 6); ++w) wbase += s_wsum[w];
    s_base[tid] = wbase + inc - total + before;
  }
  __syncthreads();
  const int wave = tid >> 6, lane = tid & 63;
  const uint64_t lt = lanemask_lt(lane);
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kRsTile + wave * kRsWaveItems;
  constexpr int kSteps = kRsWaveItems / 64;
  K kk[kSteps];
  int32_t vv[kSteps];
  int dig[kSteps];
  int rank[kSteps];
#pragma unroll
  for (int k = 0; k < kSteps; ++k) {
    const int64_t e = base + k * 64 + lane;
    const bool valid = e < n;
    int d = 0;
    if (valid) {
      kk[k] = kin[e];
      vv[k] = vin ? vin[e] : static_cast<int32_t>(e);  // no values: the input positions
      d = static_cast<int>((kk[k] >> shift) & 255u);
    }
    dig[k] = d;
    uint64_t match = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (d >> b) & 1;
      const uint64_t bal = __ballot(bit);
      match &= bit ? bal : ~bal;
    }
    rank[k] = 0;
    if (valid) {
      const int r = __popcll(match & lt);
      const int prev = s_cnt[wave][d];
      rank[k] = prev + r;
      if (r == 0) s_cnt[wave][d] = prev + __popcll(match);
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // Thread `tid` is digit tid: offsets of the waves' runs inside the tile's
  // run of the digit, and the digit's run start in the tile's digit-sorted
  // order.
  int32_t tile_cnt;
  {
    int32_t run = 0;
    for (int w = 0; w < kRsWaves; ++w) {
      s_off[w][tid] = run;
      run += s_cnt[w][tid];
    }
    s_start[tid] = block_exclusive_sum(run, &tile_cnt);
    if (!kFromHist) s_base[tid] = offs[static_cast<int64_t>(tid) * tiles + blockIdx.x];
  }
  __syncthreads();
  // The tile is staged in LDS in digit order, then written out by
  // consecutive threads to consecutive positions of each digit's run, so
  // the stores of a digit's run are contiguous.
#pragma unroll
  for (int k = 0; k < kSteps; ++k) {
    const int64_t e = base + k * 64 + lane;
    if (e < n) {
      const int d = dig[k];
      const int32_t local = s_start[d] + s_off[wave][d] + rank[k];
      s_key[local] = kk[k];
      s_val[local] = vv[k];
    }
  }
  __syncthreads();
  for (int i = tid; i < tile_cnt; i += kBlock) {
    const K key = s_key[i];
    const int d = static_cast<int>((key >> shift) & 255u);
    const int32_t pos = s_base[d] + (i - s_start[d]);
    kout[pos] = key;
    vout[pos] = s_val[i];
  }
}

// ------------------------------------------------------------- transpose ----
// (row, value) of every entry of A packed into 16 bytes, so that the
// transpose's gather reads one pair per entry instead of two scattered
// words: one thread per entry over tiles of 256 rows (an entry finds its row
// by a binary search of the tile's row pointers in LDS), so reads and writes
// stay coalesced whatever the row lengths.
__global__ __launch_bounds__(kBlock) void k_expand_rows(const int32_t* __restrict__ ptr,
                                                        const double* __restrict__ val, int32_t m,
                                                        gpk_row_val* __restrict__ rv) {
  __shared__ int32_t s_ptr[kBlock + 1];
  const int32_t r0 = blockIdx.x * kBlock;
  const int nr = min(kBlock, m - r0);
  for (int t = threadIdx.x; t <= nr; t += kBlock) s_ptr[t] = ptr[r0 + t];
  __syncthreads();
  const int32_t b = s_ptr[0];
  for (uint32_t o = threadIdx.x, n = row_length(b, s_ptr[nr]); o < n; o += kBlock) {
    const int32_t p = b + static_cast<int32_t>(o);
    const double v = val[p];
    reinterpret_cast<int4*>(rv)[p] =
        make_int4(r0 + find_row(s_ptr, nr, p), 0, __double2loint(v), __double2hiint(v));
  }
}

// Row pointers of the transpose from its sorted column keys: position p
// starts every column in (key[p-1], key[p]] (p = nnz closes the columns up
// to n), so each pointer is written once and no counter is shared.
__global__ void k_col_bounds(const uint32_t* keys, int32_t nnz, int32_t n, int32_t* ptr) {
  const int32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p > nnz) return;
  const int32_t hi = p < nnz ? static_cast<int32_t>(keys[p]) : n;
  const int32_t lo = p > 0 ? static_cast<int32_t>(keys[p - 1]) : -1;
  for (int32_t j = lo + 1; j <= hi; ++j) ptr[j] = p;
}

__global__ void k_transpose_gather(const int32_t* __restrict__ perm, const gpk_row_val* __restrict__ rv,
                                   int32_t nnz, int32_t* __restrict__ at_idx, double* __restrict__ at_val) {
  const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnz) return;
  const int4 w = reinterpret_cast<const int4*>(rv)[perm[k]];  // one 16-byte load
  at_idx[k] = w.x;
  at_val[k] = __hiloint2double(w.w, w.z);
}

// The transpose by buckets of 2^low columns (at most kTbBuckets of them): the
// entries are moved once, with their rows and values, into the buckets, and
// once more, by a workgroup for each bucket, to their columns.  Both moves keep
// the order of A, so every row of the transpose comes out sorted.  (The sort of
// the column indices alone reads and writes (key, position) three times and
// then gathers 16 bytes from a line of 128 for each entry: 493 us a call for the
// 1M x 1.5M LP's 8 million entries, of which 154 the gather; this takes 281: 34
// the counts and pieces, 90 the first move, 105 the second, the rest allocations
// and the call.  8 million entries with 100,000 to a million of them in one
// column: 395 to 402, 480 by the sort; 80 million 3.2 ms against 4.9.)  The moves are bound by their
// stores, a request to the L2 for each 16 bytes and for each 4 and 8.
constexpr int kTbBlock = 512;
constexpr int kTbWaves = kTbBlock / 64;
constexpr int kTbSteps = 8;  // of 64 consecutive entries, for a wave
constexpr int kTbTile = kTbBlock * kTbSteps;
constexpr int kTbBuckets = 1024;
constexpr int kTbLowMax = 11;
constexpr int kTbCols = 1 << kTbLowMax;

// Rows that a tile spans (its entries' and the empty ones between) up to which
// each marks its first entry; past that every entry looks its row up by
// bisection.  With 900,000 empty rows in one tile's span a transpose of 8 million
// entries takes 375 us, 1,190 with a mark for each of them (9 million: 375 against
// 8,670).
constexpr int32_t kTbMarkRows = 16 * kTbBlock;

// Blocks go to the XCDs in turn; neighbouring tiles write neighbouring words, so
// an XCD gets a stretch of tiles and its L2 joins them into whole lines.
constexpr int kXcds = 8;
__device__ __forceinline__ int32_t tb_tile(int32_t tiles) {
  const int32_t b = static_cast<int32_t>(blockIdx.x), x = b % kXcds, q = tiles / kXcds, r = tiles % kXcds;
  return x * q + min(x, r) + b / kXcds;
}

// A column outside the matrix counts as one of the last bucket.
__device__ __forceinline__ int tb_bucket(int32_t col, int low, int buckets) {
  return static_cast<int>(min(static_cast<uint32_t>(col) >> low, static_cast<uint32_t>(buckets - 1)));
}

// The place of each valid lane's entry among those of its digit that the wave
// has ranked so far, counted in cnt[digit].
__device__ __forceinline__ int tb_rank(uint16_t* cnt, int digit, int bits, bool valid, uint64_t below) {
  uint64_t match = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool bit = (digit >> b) & 1;
    const uint64_t bal = __ballot(bit);
    match &= bit ? bal : ~bal;
  }
  int rank = 0;
  if (valid) {
    const int r = __popcll(match & below);
    const int prev = cnt[digit];
    rank = prev + r;
    if (r == 0) cnt[digit] = static_cast<uint16_t>(prev + __popcll(match));
  }
  __builtin_amdgcn_wave_barrier();
  return rank;
}

__global__ __launch_bounds__(kTbBlock) void k_tb_hist(const int32_t* __restrict__ col, int32_t nnz, int low,
                                                      int32_t buckets, int32_t tiles, int32_t* __restrict__ hist) {
  __shared__ int32_t s_h[kTbBuckets];
  const int tid = static_cast<int>(threadIdx.x);
  const int32_t tile = tb_tile(tiles);
  for (int d = tid; d < buckets; d += kTbBlock) s_h[d] = 0;
  const int64_t c0 = static_cast<int64_t>(tile) * kTbTile;
  int32_t j[kTbSteps];
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k) j[k] = c0 + k * kTbBlock + tid < nnz ? col[c0 + k * kTbBlock + tid] : 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k)
    if (c0 + k * kTbBlock + tid < nnz) atomicAdd(&s_h[tb_bucket(j[k], low, buckets)], 1);
  __syncthreads();
  for (int d = tid; d < buckets; d += kTbBlock) hist[static_cast<int64_t>(d) * tiles + tile] = s_h[d];
}

// The second move takes a bucket by one workgroup, at about 1 us for 1,000
// entries, unless it holds more than tb_share(nnz): then by several, each a
// piece of its entries.  The share keeps a workgroup's time at what the whole
// chip needs for the others, so a bucket of ordinary size has one piece (8
// million entries: 62,500), and at most nnz / share + 1 buckets are split.
constexpr int32_t kTbShareMin = 16384;
constexpr int kTbMore = 128;              // pieces beyond one a bucket
constexpr int kTbSplit = 2 * kTbMore;     // pieces of split buckets
inline int32_t tb_share(int32_t nnz) {
  const int32_t part = nnz / kTbMore + 1;
  return part > kTbShareMin ? part : kTbShareMin;
}
struct TbPiece {
  int32_t bucket;      // -1: none
  int32_t begin, end;  // its entries
  int32_t piece, pieces;
  int32_t slot;  // of its column counts, the bucket's others next to it
};
static_assert(sizeof(TbPiece) == 6 * sizeof(int32_t), "laid out in 32-bit scratch");

// The pieces of all buckets, in their order; entries past them have no bucket.
// split[s]: the piece with slot s, -1 past the last.
__global__ __launch_bounds__(kTbBuckets) void k_tb_pieces(const int32_t* __restrict__ offs, int32_t buckets,
                                                          int32_t tiles, int32_t share, TbPiece* __restrict__ piece,
                                                          int32_t* __restrict__ split) {
  __shared__ int32_t s_all[kTbBuckets / 64], s_slots[kTbBuckets / 64];
  const int d = static_cast<int>(threadIdx.x), wave = d >> 6;
  const int32_t b = d < buckets ? offs[static_cast<int64_t>(d) * tiles] : 0;
  const int32_t e = d < buckets ? offs[static_cast<int64_t>(d + 1) * tiles] : 0;
  const int32_t n = d >= buckets ? 0 : e - b > share ? (e - b - 1) / share + 1 : 1;
  const int32_t many = n > 1 ? n : 0;
  const int32_t all = wave_inclusive_sum(n), slots = wave_inclusive_sum(many);
  if ((d & 63) == 63) {
    s_all[wave] = all;
    s_slots[wave] = slots;
  }
  __syncthreads();
  int32_t at = all - n, slot = slots - many, total = 0, total_slots = 0;
  for (int w = 0; w < kTbBuckets / 64; ++w) {
    at += w < wave ? s_all[w] : 0;
    slot += w < wave ? s_slots[w] : 0;
    total += s_all[w];
    total_slots += s_slots[w];
  }
  for (int32_t k = 0; k < n; ++k) {
    const int32_t from = b + k * share;
    piece[at + k] = TbPiece{d, from, k + 1 < n ? from + share : e, k, n, slot + k};
    if (many != 0) split[slot + k] = at + k;
  }
  for (int32_t k = total + d; k < buckets + kTbMore; k += kTbBuckets) piece[k] = TbPiece{-1, 0, 0, 0, 0, 0};
  for (int32_t k = total_slots + d; k < kTbSplit; k += kTbBuckets) split[k] = -1;
}

// The last row that starts at or before entry p, by a wave: a 64th of the rows
// is left after each look.
__device__ inline int32_t wave_row_of(const int32_t* __restrict__ ptr, int32_t m, int32_t p) {
  int32_t lo = 0, n = m;  // the row is one of [lo, lo + n)
  while (n > 1) {
    const int32_t step = (n + 63) / 64;
    const int64_t r = static_cast<int64_t>(lo) + static_cast<int64_t>(lane_id()) * step;
    const uint64_t before = __ballot(r < static_cast<int64_t>(lo) + n && ptr[r < m ? r : m] <= p);
    const int32_t at = max(static_cast<int32_t>(__popcll(before)) - 1, 0) * step;
    lo += at;
    n = min(step, n - at);
  }
  return lo;
}

__global__ __launch_bounds__(kTbBlock) void k_tb_partition(const int32_t* __restrict__ ptr,
                                                           const int32_t* __restrict__ col,
                                                           const double* __restrict__ val, int32_t m, int32_t nnz,
                                                           int low, int32_t buckets, int bits, int32_t tiles,
                                                           const int32_t* __restrict__ offs, int4* __restrict__ rec) {
  __shared__ uint16_t s_cnt[kTbWaves][kTbBuckets];
  __shared__ int32_t s_base[kTbBuckets];
  __shared__ int32_t s_row[kTbTile];  // row - first, of each entry
  __shared__ int32_t s_w[kTbWaves];
  __shared__ int32_t s_first, s_last;
  const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
  const int32_t tile = tb_tile(tiles);
  const int32_t c0 = tile * kTbTile;
  const int32_t cnt = min(kTbTile, nnz - c0);
  const int32_t mine = wave * (64 * kTbSteps) + lane;
  int32_t j[kTbSteps];
  double v[kTbSteps];
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k) {
    const int32_t p = c0 + min(mine + 64 * k, cnt - 1);
    j[k] = col[p];
    v[k] = val[p];
  }
  for (int i = tid; i < kTbWaves * kTbBuckets / 2; i += kTbBlock) reinterpret_cast<uint32_t*>(&s_cnt[0][0])[i] = 0;
  for (int i = tid; i < kTbTile; i += kTbBlock) s_row[i] = 0;
  for (int d = tid; d < buckets; d += kTbBlock) s_base[d] = offs[static_cast<int64_t>(d) * tiles + tile];
  if (wave < 2) {
    const int32_t r = wave_row_of(ptr, m, wave == 0 ? c0 : c0 + (cnt - 1));
    if (lane == 0) (wave == 0 ? s_first : s_last) = r;
  }
  __syncthreads();
  const int32_t first = s_first, last = s_last;
  if (last - first <= kTbMarkRows) {
    // Each further row marks its first entry (of rows that start together the
    // last one holds it); the running maximum is then every entry's row.
    for (int64_t r = static_cast<int64_t>(first) + 1 + tid; r <= last; r += kTbBlock) {
      const int32_t p = ptr[r] - c0;
      if (p >= 0) atomicMax(&s_row[p], static_cast<int32_t>(r - first));
    }
  } else {
    for (int i = tid; i < cnt; i += kTbBlock) {
      int32_t lo = first, hi = last;  // the last row that starts at or before the entry is one of [lo, hi]
      while (lo < hi) {
        const int32_t mid = hi - (hi - lo) / 2;
        if (ptr[mid] <= c0 + i) lo = mid; else hi = mid - 1;
      }
      s_row[i] = lo - first;
    }
  }
  __syncthreads();
  int32_t run[kTbSteps];
  int32_t most = 0;
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k) {
    most = max(most, s_row[tid * kTbSteps + k]);
    run[k] = most;
  }
  int32_t upto = most;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t o = __shfl_up(upto, d, 64);
    if (lane >= d) upto = max(upto, o);
  }
  if (lane == 63) s_w[wave] = upto;
  int32_t before = __shfl_up(upto, 1, 64);
  if (lane == 0) before = 0;
  __syncthreads();
  for (int w = 0; w < wave; ++w) before = max(before, s_w[w]);
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k) s_row[tid * kTbSteps + k] = max(before, run[k]);
  const uint64_t below = lanemask_lt(lane);
  int digit[kTbSteps], rank[kTbSteps];
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k) {
    digit[k] = tb_bucket(j[k], low, buckets);
    rank[k] = tb_rank(s_cnt[wave], digit[k], bits, mine + 64 * k < cnt, below);
  }
  __syncthreads();
  for (int d = tid; d < buckets; d += kTbBlock) {
    int32_t sum = 0;
#pragma unroll
    for (int w = 0; w < kTbWaves; ++w) {
      const int32_t c = s_cnt[w][d];
      s_cnt[w][d] = static_cast<uint16_t>(sum);
      sum += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kTbSteps; ++k)
    if (mine + 64 * k < cnt)
      rec[s_base[digit[k]] + s_cnt[wave][digit[k]] + rank[k]] =
          make_int4(j[k], first + s_row[mine + 64 * k], __double2loint(v[k]), __double2hiint(v[k]));
}

// s_count[c] = the entries of column c of the bucket among rec[b, e).
__device__ __forceinline__ void tb_count_columns(const int4* __restrict__ rec, int32_t b, int32_t e, int cols,
                                                 int32_t* s_count) {
  const int tid = static_cast<int>(threadIdx.x);
  for (int i = tid; i < kTbCols; i += kTbBlock) s_count[i] = 0;
  __syncthreads();
  for (int32_t p0 = b; p0 < e; p0 += kTbTile) {
    int32_t j[kTbSteps];
#pragma unroll
    for (int k = 0; k < kTbSteps; ++k) j[k] = rec[min(p0 + k * kTbBlock + tid, e - 1)].x;
#pragma unroll
    for (int k = 0; k < kTbSteps; ++k)
      if (p0 + k * kTbBlock + tid < e) atomicAdd(&s_count[j[k] & (cols - 1)], 1);
  }
  __syncthreads();
}

// The column counts of the split buckets' pieces, kTbCols words a slot.
__global__ __launch_bounds__(kTbBlock) void k_tb_piece_counts(const int4* __restrict__ rec, int low,
                                                              const TbPiece* __restrict__ piece,
                                                              const int32_t* __restrict__ split,
                                                              int32_t* __restrict__ counts) {
  __shared__ int32_t s_count[kTbCols];
  const int32_t at = split[blockIdx.x];
  if (at < 0) return;
  tb_count_columns(rec, piece[at].begin, piece[at].end, 1 << low, s_count);
  for (int i = static_cast<int>(threadIdx.x); i < kTbCols; i += kTbBlock)
    counts[static_cast<int64_t>(blockIdx.x) * kTbCols + i] = s_count[i];
}

// A piece (mostly a whole bucket): the bucket's entries counted by column, which
// gives the columns' row pointers of the transpose, then the piece's placed tile
// by tile in their order, after those of the pieces before it.
__global__ __launch_bounds__(kTbBlock) void k_tb_columns(const int4* __restrict__ rec, int32_t n, int32_t nnz, int low,
                                                         int32_t share, const TbPiece* __restrict__ piece,
                                                         const int32_t* __restrict__ counts,
                                                         int32_t* __restrict__ at_ptr, int32_t* __restrict__ at_idx,
                                                         double* __restrict__ at_val) {
  __shared__ uint16_t s_cnt[kTbWaves][kTbCols];
  __shared__ int32_t s_next[kTbCols];  // where a column's next entry goes
  __shared__ int32_t s_w[kTbWaves];
  constexpr int kPer = kTbCols / kTbBlock;
  const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6, lane = tid & 63;
  const int cols = 1 << low;
  const TbPiece me = piece[blockIdx.x];
  if (me.bucket < 0) return;
  const int32_t b = me.begin, e = me.end;
  int32_t c[kPer], before[kPer], sum = 0;  // of the whole bucket, of the pieces before
  if (me.pieces == 1) {
    tb_count_columns(rec, b, e, cols, s_next);
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      c[k] = s_next[tid * kPer + k];
      before[k] = 0;
    }
  } else {
    static_assert(kPer == 4, "a thread's columns in one load");
    const int4* __restrict__ of = reinterpret_cast<const int4*>(counts + static_cast<int64_t>(me.slot - me.piece) * kTbCols) + tid;
    int4 t{0, 0, 0, 0}, f{0, 0, 0, 0};
#pragma unroll 8
    for (int32_t k = 0; k < me.pieces; ++k) {
      const int4 v = of[static_cast<int64_t>(k) * (kTbCols / 4)];
      const int32_t on = k < me.piece ? 1 : 0;
      t.x += v.x, t.y += v.y, t.z += v.z, t.w += v.w;
      f.x += on * v.x, f.y += on * v.y, f.z += on * v.z, f.w += on * v.w;
    }
    c[0] = t.x, c[1] = t.y, c[2] = t.z, c[3] = t.w;
    before[0] = f.x, before[1] = f.y, before[2] = f.z, before[3] = f.w;
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) sum += c[k];
  const int32_t inc = wave_inclusive_sum(sum);
  if (lane == 63) s_w[wave] = inc;
  __syncthreads();
  int32_t at = b - me.piece * share + inc - sum;  // from where the bucket begins
  for (int w = 0; w < wave; ++w) at += s_w[w];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int64_t col = (static_cast<int64_t>(me.bucket) << low) + tid * kPer + k;
    if (me.piece == 0 && tid * kPer + k < cols && col < n) at_ptr[col] = at;
    s_next[tid * kPer + k] = at + before[k];
    at += c[k];
  }
  if (me.bucket == 0 && me.piece == 0 && tid == 0) at_ptr[n] = nnz;
  const uint64_t below = lanemask_lt(lane);
  const int32_t mine = wave * (64 * kTbSteps) + lane;
  for (int32_t p0 = b; p0 < e; p0 += kTbTile) {
    const int32_t cnt = min(kTbTile, e - p0);
    int4 w4[kTbSteps];
    int rank[kTbSteps];
#pragma unroll
    for (int k = 0; k < kTbSteps; ++k) w4[k] = rec[p0 + min(mine + 64 * k, cnt - 1)];
    for (int w = 0; w < kTbWaves; ++w)
      for (int i = tid; i < (cols + 1) / 2; i += kTbBlock) reinterpret_cast<uint32_t*>(s_cnt[w])[i] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTbSteps; ++k)
      rank[k] = tb_rank(s_cnt[wave], w4[k].x & (cols - 1), low, mine + 64 * k < cnt, below);
    __syncthreads();
    int32_t total[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      total[k] = 0;
      const int col = tid + k * kTbBlock;
      if (col < cols)
#pragma unroll
        for (int w = 0; w < kTbWaves; ++w) {
          const int32_t t = s_cnt[w][col];
          s_cnt[w][col] = static_cast<uint16_t>(total[k]);
          total[k] += t;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTbSteps; ++k)
      if (mine + 64 * k < cnt) {
        const int col = w4[k].x & (cols - 1);
        const int32_t to = s_next[col] + s_cnt[wave][col] + rank[k];
        at_idx[to] = w4[k].y;
        at_val[to] = __hiloint2double(w4[k].w, w4[k].z);
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (tid + k * kTbBlock < cols) s_next[tid + k * kTbBlock] += total[k];
    __syncthreads();
  }
}

// CSR checks.  The row pointers are checked first, one row a thread
// (flags[0]: not monotone, not from 0 to nnz), and leave the chunk rows of the
// matrix (its last row past the last chunk); then chunks of 2048 entries are
// checked, 8 a thread, whatever the rows (tiles of 256 rows, each entry
// finding its row by bisection, took 1.35 ms on 200 adjacent rows of 3,000
// entries, and 98 us for A and AT of the 1M x 1.5M LP; 10 and 37 us for both
// launches by chunks).  A
// chunk marks the first entry of each of its rows in a bitmap; every other
// entry is compared with the one before it: flags[1] a column outside
// [0, cols), flags[2] two equal neighbours, flags[3] a descending pair.  No
// entry is read of a matrix whose pointers are bad.
// Rows of a chunk (its entries' and the empty ones between) up to which they
// mark their first entries; past that every entry looks its row up by
// bisection.
constexpr int kChkMarkRows = 8192;
constexpr int kChkItems = 8;
constexpr int kChkChunk = kBlock * kChkItems;

__global__ __launch_bounds__(kBlock) void k_csr_check_ptr(gpk_csr_check_side a, gpk_csr_check_side t,
                                                          int32_t blocks_a) {
  const bool first = static_cast<int32_t>(blockIdx.x) < blocks_a;
  const gpk_csr_check_side& s = first ? a : t;
  const int64_t i = static_cast<int64_t>(first ? blockIdx.x : blockIdx.x - blocks_a) * kBlock + threadIdx.x;
  if (i >= s.rows) return;
  const int32_t b = s.ptr[i], e = s.ptr[i + 1];
  if ((i == 0 && b != 0) || (i == s.rows - 1 && e != s.nnz) || b > e || b < 0 || e > s.nnz) {
    wave_set_flag(s.flags);
    return;
  }
#pragma unroll 1
  for (int64_t q = (static_cast<int64_t>(b) + kChkChunk - 1) / kChkChunk; q * kChkChunk < e; ++q)
    s.chunk_row[q] = static_cast<int32_t>(i);
}

__global__ __launch_bounds__(kBlock) void k_csr_check_entries(gpk_csr_check_side a, gpk_csr_check_side t,
                                                              int32_t chunks_a, int32_t chunks_t) {
  __shared__ uint32_t s_head[kChkChunk / 32];
  const int32_t blk = static_cast<int32_t>(blockIdx.x);
  const bool first = blk < chunks_a;
  const gpk_csr_check_side& s = first ? a : t;
  const int32_t q = first ? blk : blk - chunks_a, chunks = first ? chunks_a : chunks_t;
  const int tid = threadIdx.x;
  if (*s.flags != 0) return;  // the pointers are bad (set by the launch before)
  const int32_t c0 = q * kChkChunk, c1 = min(s.nnz - c0, kChkChunk);
  int32_t j[kChkItems];
#pragma unroll
  for (int k = 0; k < kChkItems; ++k) j[k] = s.idx[c0 + min(k * kBlock + tid, c1 - 1)];
  const int32_t edge = s.idx[c0 > 0 ? c0 - 1 : 0];
  const int32_t r_lo = s.chunk_row[q], r_hi = q + 1 < chunks ? s.chunk_row[q + 1] : s.rows - 1;
  if (tid < kChkChunk / 32) s_head[tid] = 0;
  __syncthreads();
  if (r_hi - r_lo < kChkMarkRows) {
#pragma unroll 1
    for (int64_t r = static_cast<int64_t>(r_lo) + tid; r <= r_hi; r += kBlock) {
      const int32_t b = s.ptr[r] - c0;
      if (b >= 0 && b < c1) atomicOr(&s_head[b >> 5], 1u << (b & 31));  // empty rows mark their successor's
    }
  } else {
    for (int p = tid; p < c1; p += kBlock) {
      int32_t lo = r_lo, hi = r_hi;  // the last row that starts at or before the entry is one of [lo, hi]
      while (lo < hi) {
        const int32_t mid = hi - (hi - lo) / 2;
        if (s.ptr[mid] <= c0 + p) lo = mid; else hi = mid - 1;
      }
      if (s.ptr[lo] == c0 + p) atomicOr(&s_head[p >> 5], 1u << (p & 31));
    }
  }
  __syncthreads();
  bool range = false, equal = false, desc = false;
#pragma unroll
  for (int k = 0; k < kChkItems; ++k) {
    const int p = k * kBlock + tid;
    // The entry before: the lane below, or for a wave's first lane from memory.
    int32_t before = __shfl_up(j[k], 1, 64);
    if (lane_id() == 0 && p < c1) before = p == 0 ? edge : s.idx[c0 + p - 1];
    if (p >= c1) continue;
    range = range || j[k] < 0 || j[k] >= s.cols;
    if (((s_head[p >> 5] >> (p & 31)) & 1u) == 0) {
      equal = equal || j[k] == before;
      desc = desc || j[k] < before;
    }
  }
  if (range) wave_set_flag(s.flags + 1);
  if (equal) wave_set_flag(s.flags + 2);
  if (desc) wave_set_flag(s.flags + 3);
}

// Rows sorted by column, over tiles of 256 rows with one thread per entry (the
// pointers are trusted): every entry finds its row by a bisection of the tile's
// row pointers in LDS and is compared with the entry before it in the same
// row.
__global__ __launch_bounds__(kBlock) void k_csr_unsorted(const int32_t* __restrict__ ptr,
                                                         const int32_t* __restrict__ idx, int32_t rows,
                                                         int32_t* flag) {
  __shared__ int32_t s_ptr[kBlock + 1];
  const int32_t r0 = blockIdx.x * kBlock;
  const int nr = min(kBlock, rows - r0);
  const int tid = threadIdx.x;
  for (int t = tid; t <= nr; t += kBlock) s_ptr[t] = ptr[r0 + t];
  __syncthreads();
  bool desc = false;
  const int32_t b = s_ptr[0];
  for (uint32_t o = tid, n = row_length(b, s_ptr[nr]); o < n; o += kBlock) {
    const int32_t p = b + static_cast<int32_t>(o);
    if (p > s_ptr[find_row(s_ptr, nr, p)]) desc = desc || idx[p] < idx[p - 1];
  }
  if (desc) wave_set_flag(flag);
}

// Input check of a CSR matrix, one row per thread (for matrices whose rows
// arrive unsorted: a column can repeat at a distance): flags[0] row pointers
// that are not monotone or do not start at 0 / end at nnz, flags[1] a column
// index outside [0, cols), flags[2] a column repeated within a row, flags[3]
// a row whose columns are not ascending.  Sorted rows are checked for repeats
// by neighbours; an unsorted row compares every pair of its entries.
__global__ void k_csr_check(const int32_t* ptr, const int32_t* idx, int32_t rows, int32_t cols, int32_t nnz,
                            int32_t* flags) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows) return;
  const int32_t b = ptr[i], e = ptr[i + 1];
  if ((i == 0 && b != 0) || (i == rows - 1 && e != nnz) || b > e || b < 0 || e > nnz) {
    wave_set_flag(flags);
    return;
  }
  bool range = false, repeat = false, unsorted = false;
  int32_t prev = -1;
  for (int32_t p = b; p < e; ++p) {
    const int32_t j = idx[p];
    range = range || j < 0 || j >= cols;
    if (p > b) {
      repeat = repeat || j == prev;
      unsorted = unsorted || j < prev;
    }
    prev = j;
  }
  if (unsorted && !repeat) {
    for (int32_t p = b + 1; p < e && !repeat; ++p) {
      const int32_t j = idx[p];
      for (int32_t q = b; q < p; ++q)
        if (idx[q] == j) {
          repeat = true;
          break;
        }
    }
  }
  if (range) wave_set_flag(flags + 1);
  if (repeat) wave_set_flag(flags + 2);
  if (unsorted) wave_set_flag(flags + 3);
}

// Stable insertion sort of one row per thread (used only for inputs whose
// rows arrive unsorted).
__global__ void k_sort_rows(const int32_t* ptr, int32_t* idx, double* val, int32_t rows) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows) return;
  const int32_t b = ptr[i], e = ptr[i + 1];
  for (int32_t p = b + 1; p < e; ++p) {
    const int32_t key = idx[p];
    const double v = val[p];
    int32_t q = p - 1;
    while (q >= b && idx[q] > key) {
      idx[q + 1] = idx[q];
      val[q + 1] = val[q];
      --q;
    }
    idx[q + 1] = key;
    val[q + 1] = v;
  }
}

// Sorts up to kSortSmallMax (key, value) pairs in one workgroup: a bitonic
// network in LDS over (key, input position), so the order equals that of the
// stable radix sort; the values follow through the positions.
constexpr int kSortSmallMax = 4096;
constexpr int kSortSmallBlock = 1024;

template <class K>
__global__ __launch_bounds__(kSortSmallBlock) void k_sort_small(K* __restrict__ keys, int32_t* __restrict__ vals,
                                                               int32_t n) {
  __shared__ K s_k[kSortSmallMax];
  __shared__ int32_t s_v[kSortSmallMax];
  __shared__ int16_t s_p[kSortSmallMax];
  static_assert(kSortSmallMax <= 32768, "positions are stored in 16 bits");
  const int tid = threadIdx.x;
  int len = 1;
  while (len < n) len <<= 1;
  for (int i = tid; i < len; i += kSortSmallBlock) {
    s_k[i] = i < n ? keys[i] : static_cast<K>(~static_cast<K>(0));
    s_p[i] = static_cast<int16_t>(i);
    if (i < n) s_v[i] = vals[i];
  }
  __syncthreads();
  for (int size = 2; size <= len; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = tid; t < (len >> 1); t += kSortSmallBlock) {
        const int i = 2 * t - (t & (stride - 1));  // lower index of the pair
        const int j = i + stride;
        const bool up = (i & size) == 0;
        const K ki = s_k[i], kj = s_k[j];
        const int pi = s_p[i], pj = s_p[j];
        const bool gt = ki > kj || (ki == kj && pi > pj);
        if (gt == up) {
          s_k[i] = kj;
          s_k[j] = ki;
          s_p[i] = static_cast<int16_t>(pj);
          s_p[j] = static_cast<int16_t>(pi);
        }
      }
      // A stage with stride <= 64 only touches its wave's own 128-element
      // segments (pair t of thread t lies in [128 (t / 64), +128)), so between
      // two such stages the wave's LDS order suffices; any wider stage, before
      // or after, meets the other waves at the workgroup barrier.
      const int next = stride > 1 ? stride >> 1 : (size < len ? size : kSortSmallBlock);
      if (stride > 64 || next > 64) {
        __syncthreads();
      } else {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
  }
  for (int i = tid; i < n; i += kSortSmallBlock) {
    keys[i] = s_k[i];
    vals[i] = s_v[s_p[i]];
  }
}

// Words of scratch of a scan of n values.
int64_t scan_scratch_ints(int64_t n) { return (n + kScanTile - 1) / kScanTile + 1; }

template <class In>
hipError_t scan_impl(const In* in, int32_t* out, int64_t n, int32_t* scratch, hipStream_t s) {
  if (n <= 0) {
    return hipMemsetAsync(out, 0, sizeof(int32_t), s);
  }
  if (n <= kSmallScanMax) {
    hipLaunchKernelGGL((k_scan_small<In>), dim3(1), dim3(kSmallBlock), 0, s, in, out, n);
    return hipGetLastError();
  }
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL(k_scan_tiles<In>, dim3(static_cast<unsigned>(tiles)), dim3(kBlock), 0, s, in, n, scratch);
  hipLaunchKernelGGL(k_scan_tile_sums, dim3(1), dim3(kBlock), 0, s, scratch, tiles, out + n);
  hipLaunchKernelGGL(k_scan_down<In>, dim3(static_cast<unsigned>(tiles)), dim3(kBlock), 0, s, in, out, n,
                     static_cast<const int32_t*>(scratch));
  return hipGetLastError();
}

template <class K>
hipError_t radix_impl(K* keys, int32_t* vals, K* keys_alt, int32_t* vals_alt, int32_t n, int32_t key_bits,
                      int32_t* scratch, hipStream_t s) {
  if (n <= 1) return hipSuccess;
  if (n <= kSortSmallMax) {
    hipLaunchKernelGGL(k_sort_small<K>, dim3(1), dim3(kSortSmallBlock), 0, s, keys, vals, n);
    return hipGetLastError();
  }
  const int32_t tiles = (n + kRsTile - 1) / kRsTile;
  int32_t* hist = scratch;
  int32_t* scan_scratch = scratch + static_cast<int64_t>(256) * tiles + 1;
  const int passes = key_bits <= 0 ? 1 : (key_bits + 7) / 8;
  const bool from_hist = tiles <= kRsHistTilesMax;
  K* ka = keys;
  int32_t* va = vals;
  K* kb = keys_alt;
  int32_t* vb = vals_alt;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = pass * 8;
    if (from_hist) {
      hipLaunchKernelGGL((k_radix_hist<K, true>), dim3(tiles), dim3(kBlock), 0, s, ka, n, shift, tiles, hist);
      hipLaunchKernelGGL((k_radix_scatter<K, true>), dim3(tiles), dim3(kBlock), 0, s, ka, va, kb, vb, n, shift,
                         tiles, static_cast<const int32_t*>(hist));
    } else {
      hipLaunchKernelGGL((k_radix_hist<K, false>), dim3(tiles), dim3(kBlock), 0, s, ka, n, shift, tiles, hist);
      hipError_t e = scan_impl<int32_t>(hist, hist, static_cast<int64_t>(256) * tiles, scan_scratch, s);
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL((k_radix_scatter<K, false>), dim3(tiles), dim3(kBlock), 0, s, ka, va, kb, vb, n, shift,
                         tiles, static_cast<const int32_t*>(hist));
    }
    K* tk = ka; ka = kb; kb = tk;
    int32_t* tv = va; va = vb; vb = tv;
  }
  if (ka != keys) {
    hipError_t e = hipMemcpyAsync(keys, ka, sizeof(K) * n, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
    e = hipMemcpyAsync(vals, va, sizeof(int32_t) * n, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
  }
  return hipGetLastError();
}

inline unsigned grid_fill(int64_t n) {
  const unsigned g = grid_for(n);
  return g > 65535u ? 65535u : g;
}

}  // namespace

extern "C" {

hipError_t gpk_fill_u8(uint8_t* dst, uint8_t v, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<uint8_t>, dim3(grid_fill(n)), dim3(kBlock), 0, s, dst, v, n);
  return hipGetLastError();
}
hipError_t gpk_fill_i32(int32_t* dst, int32_t v, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<int32_t>, dim3(grid_fill(n)), dim3(kBlock), 0, s, dst, v, n);
  return hipGetLastError();
}
hipError_t gpk_fill_f64(double* dst, double v, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_fill<double>, dim3(grid_fill(n)), dim3(kBlock), 0, s, dst, v, n);
  return hipGetLastError();
}
hipError_t gpk_iota_i32(int32_t* dst, int32_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_iota, dim3(grid_for(n)), dim3(kBlock), 0, s, dst, n);
  return hipGetLastError();
}

int64_t gpk_lookback_tiles(int64_t n) { return n > 0 ? (n + kScanTile - 1) / kScanTile : 1; }

hipError_t gpk_scan_lb_i32(const int32_t* in, int32_t* out, int64_t n, gpk_lookback lb, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (n <= kSmallScanMax) {
    hipLaunchKernelGGL((k_scan_small<int32_t>), dim3(1), dim3(kSmallBlock), 0, s, in, out, n);
    return hipGetLastError();
  }
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL((k_scan_lb<int32_t>), dim3(static_cast<unsigned>(tiles)), dim3(kBlock), 0, s, in, out, n,
                     lb);
  return hipGetLastError();
}

hipError_t gpk_scan_lb_mask(const uint8_t* mask, int32_t* out, int64_t n, gpk_lookback lb, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (n <= GPK_MAP_RECOUNT_MAX && (reinterpret_cast<uintptr_t>(mask) & 15u) == 0) {
    hipLaunchKernelGGL(k_mask_scan, dim3(grid_for(n, kScanTile)), dim3(kBlock), 0, s, mask, out,
                       static_cast<int32_t>(n));
    return hipGetLastError();
  }
  if (n <= kSmallScanMax) {
    hipLaunchKernelGGL((k_scan_small<uint8_t>), dim3(1), dim3(kSmallBlock), 0, s, mask, out, n);
    return hipGetLastError();
  }
  const int64_t tiles = (n + kScanTile - 1) / kScanTile;
  hipLaunchKernelGGL((k_scan_lb<uint8_t>), dim3(static_cast<unsigned>(tiles)), dim3(kBlock), 0, s, mask, out, n,
                     lb);
  return hipGetLastError();
}

int64_t gpk_apply_maps_tiles(int32_t m, int32_t n) {
  const int64_t rt = m > 0 ? (static_cast<int64_t>(m) + kScanTile - 1) / kScanTile : 0;
  const int64_t ct = n > 0 ? (static_cast<int64_t>(n) + kScanTile - 1) / kScanTile : 0;
  return rt + ct;
}

hipError_t gpk_apply_maps(gpk_apply_maps_args args, gpk_lookback lb, hipStream_t s) {
  const int64_t tiles = gpk_apply_maps_tiles(args.m, args.n);
  if (tiles == 0) return hipSuccess;
  const dim3 grid(static_cast<unsigned>(tiles));
  const int32_t r = static_cast<int32_t>(gpk_apply_maps_tiles(args.m, 0));
  const bool aligned =
      ((reinterpret_cast<uintptr_t>(args.keep_row) | reinterpret_cast<uintptr_t>(args.keep_col)) & 15u) == 0;
  const int32_t al = aligned ? 1 : 0;
  if (aligned && args.m <= GPK_MAP_RECOUNT_MAX && args.n <= GPK_MAP_RECOUNT_MAX) {
    hipLaunchKernelGGL(k_apply_maps<kMapRecount>, grid, dim3(kBlock), 0, s, args, r, al, lb);
  } else if (tiles <= GPK_MAP_COUNT_TILES) {
    hipLaunchKernelGGL(k_apply_counts, grid, dim3(kBlock), 0, s, args, r, al);
    hipLaunchKernelGGL(k_apply_maps<kMapCounts>, grid, dim3(kBlock), 0, s, args, r, al, lb);
  } else {
    hipLaunchKernelGGL(k_apply_maps<kMapLookback>, grid, dim3(kBlock), 0, s, args, r, al, lb);
  }
  return hipGetLastError();
}

int32_t gpk_compact_shift(int32_t nnz) { return nnz <= GPK_COMPACT_SMALL_NNZ ? 9 : 11; }

int32_t gpk_compact_chunks(int32_t nnz) {
  const int32_t shift = gpk_compact_shift(nnz);
  return (nnz >> shift) + ((nnz & ((1 << shift) - 1)) != 0 ? 1 : 0);
}

hipError_t gpk_compact_map(gpk_compact_side a, gpk_compact_side t, int32_t* chunk_cnt, int32_t* kept_total,
                           hipStream_t s) {
  const int32_t ca = gpk_compact_chunks(a.nnz), ct = gpk_compact_chunks(t.nnz);
  if (ca + ct == 0) return hipSuccess;
  if (gpk_compact_shift(a.nnz > t.nnz ? a.nnz : t.nnz) == 9)
    hipLaunchKernelGGL(k_compact_map<2>, dim3(ca + ct), dim3(kBlock), 0, s, a, t, ca, chunk_cnt, kept_total);
  else
    hipLaunchKernelGGL(k_compact_map<8>, dim3(ca + ct), dim3(kBlock), 0, s, a, t, ca, chunk_cnt, kept_total);
  return hipGetLastError();
}

hipError_t gpk_compact_write(gpk_compact_side a, gpk_compact_side t, const int32_t* chunk_off, int32_t from_counts,
                             gpk_apply_gathers_args gathers, hipStream_t s) {
  if (a.nnz > 0 && t.nnz > 0 && a.nnz != t.nnz) return hipErrorInvalidValue;
  const int32_t ca = gpk_compact_chunks(a.nnz), ct = gpk_compact_chunks(t.nnz);
  if (from_counts && (ca > GPK_COMPACT_COUNT_CHUNKS || ct > GPK_COMPACT_COUNT_CHUNKS)) return hipErrorInvalidValue;
  const int32_t ra = ca > 0 ? static_cast<int32_t>(grid_for(a.m_old)) : 0;
  const int32_t rt = ct > 0 ? static_cast<int32_t>(grid_for(t.m_old)) : 0;
  if (ca + ct == 0) return hipSuccess;
  const dim3 grid(ca + ct + ra + rt);
  if (gpk_compact_shift(a.nnz > t.nnz ? a.nnz : t.nnz) == 9)
    hipLaunchKernelGGL(k_compact_write<2>, grid, dim3(kBlock), 0, s, a, t, ca, ct, ra, chunk_off, from_counts, gathers);
  else
    hipLaunchKernelGGL(k_compact_write<8>, grid, dim3(kBlock), 0, s, a, t, ca, ct, ra, chunk_off, from_counts, gathers);
  return hipGetLastError();
}

hipError_t gpk_pack_lu(const double* l, const double* u, int32_t n, double* lu, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pack_lu, dim3(grid_for(n)), dim3(kBlock), 0, s, l, u, n, reinterpret_cast<double2*>(lu));
  return hipGetLastError();
}

hipError_t gpk_row_activity_lu(const int32_t* row_ptr, const int32_t* col_idx, const double* val, int32_t m,
                               int32_t nnz, const double* lu, double ztol, double* min_fin, double* max_fin, int32_t* neg_inf,
                               int32_t* pos_inf, hipStream_t s) {
  if (m <= 0) return hipSuccess;
  // The tiles, then the blocks that look for long rows: on a matrix without
  // one those end while the last tiles run.  (A launch of their own cost 2.6
  // us more at 1M rows, and in front of the tiles they cost 1 us.)
  const unsigned tiles = grid_for(m, kActRows);
  hipLaunchKernelGGL(k_row_activity_lu, dim3(tiles + long_row_blocks(m, nnz)), dim3(kBlock), 0, s, row_ptr, col_idx, val, m,
                     reinterpret_cast<const double2*>(lu), ztol, min_fin, max_fin, neg_inf, pos_inf,
                     static_cast<int32_t>(tiles));
  return hipGetLastError();
}

hipError_t gpk_col_max_abs(const int32_t* at_ptr, const double* at_val, int32_t n, double* out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_col_max_abs, dim3(grid_for(n)), dim3(kBlock), 0, s, at_ptr, at_val, n, out);
  return hipGetLastError();
}

hipError_t gpk_csr_stats(const int32_t* ptr, const int32_t* idx, const double* val, int32_t rows, int32_t* nnz_out,
                         uint8_t* empty_mask, uint8_t* singleton_mask, int32_t* singleton_idx,
                         double* singleton_val, hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_csr_stats, dim3(grid_for(rows)), dim3(kBlock), 0, s, ptr, idx, val, rows, nnz_out,
                     empty_mask, singleton_mask, singleton_idx, singleton_val);
  return hipGetLastError();
}

hipError_t gpk_mail(const uint32_t* src, int32_t words, uint32_t* mail, uint32_t seq, hipStream_t s) {
  if (words < 0 || words > 28 || (words > 0 && src == nullptr) || mail == nullptr) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_mail, dim3(1), dim3(64), 0, s, src, words, mail, seq);
  return hipGetLastError();
}

hipError_t gpk_copy_many(const gpk_copy_seg* segs, int32_t count, hipStream_t s) {
  if (count < 0 || count > GPK_COPY_MAX) return hipErrorInvalidValue;
  CopyList list{};
  int32_t used = 0;
  int64_t most = 0;
  for (int32_t k = 0; k < count; ++k) {
    if (segs[k].bytes <= 0) continue;
    list.seg[used++] = segs[k];
    most = segs[k].bytes > most ? segs[k].bytes : most;
  }
  if (used == 0) return hipSuccess;
  const int64_t per_block = static_cast<int64_t>(kBlock) * 16;
  const int64_t blocks = (most + per_block - 1) / per_block;
  hipLaunchKernelGGL(k_copy_many, dim3(static_cast<unsigned>(blocks < 1024 ? blocks : 1024), used), dim3(kBlock), 0,
                     s, list);
  return hipGetLastError();
}

hipError_t gpk_apply_gathers(gpk_apply_gathers_args args, hipStream_t s) {
  const int32_t len = args.m > args.n ? args.m : args.n;
  if (len <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_apply_gathers, dim3(grid_for(len)), dim3(kBlock), 0, s, args);
  return hipGetLastError();
}

hipError_t gpk_gather_i32(const int32_t* map, int32_t n_old, const int32_t* src, int32_t* dst, hipStream_t s) {
  if (n_old <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_gather_i32, dim3(grid_for(n_old)), dim3(kBlock), 0, s, map, n_old, src, dst);
  return hipGetLastError();
}

int64_t gpk_radix_scratch_ints(int64_t n) {
  const int64_t tiles = (n + kRsTile - 1) / kRsTile;
  return 256 * tiles + 1 + scan_scratch_ints(256 * tiles) + 1;
}

hipError_t gpk_radix_sort_u64_i32(uint64_t* keys, int32_t* vals, uint64_t* keys_alt, int32_t* vals_alt, int32_t n,
                                  int32_t key_bits, int32_t* scratch, hipStream_t s) {
  return radix_impl<uint64_t>(keys, vals, keys_alt, vals_alt, n, key_bits, scratch, s);
}

hipError_t gpk_radix_sort_u32_i32(uint32_t* keys, int32_t* vals, uint32_t* keys_alt, int32_t* vals_alt, int32_t n,
                                  int32_t key_bits, int32_t* scratch, hipStream_t s) {
  return radix_impl<uint32_t>(keys, vals, keys_alt, vals_alt, n, key_bits, scratch, s);
}

hipError_t gpk_transpose_sort(const int32_t* col, int32_t nnz, int32_t key_bits, uint32_t* ka, int32_t* va,
                              uint32_t* kb, int32_t* vb, int32_t* scratch, int32_t* result_in_b, hipStream_t s) {
  *result_in_b = 0;
  if (nnz <= 0) return hipSuccess;
  if (nnz <= kSortSmallMax) {
    hipError_t e = hipMemcpyAsync(ka, col, sizeof(uint32_t) * nnz, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_iota, dim3(grid_for(nnz)), dim3(kBlock), 0, s, va, nnz);
    hipLaunchKernelGGL(k_sort_small<uint32_t>, dim3(1), dim3(kSortSmallBlock), 0, s, ka, va, nnz);
    return hipGetLastError();
  }
  // Stable LSD passes; the first reads the column indices in place with the
  // entry positions as values.
  const int32_t tiles = (nnz + kRsTile - 1) / kRsTile;
  int32_t* hist = scratch;
  int32_t* scan_scratch = scratch + static_cast<int64_t>(256) * tiles + 1;
  const int passes = key_bits <= 0 ? 1 : (key_bits + 7) / 8;
  const bool from_hist = tiles <= kRsHistTilesMax;
  const uint32_t* kin = reinterpret_cast<const uint32_t*>(col);
  const int32_t* vin = nullptr;
  uint32_t* kout = ka;
  int32_t* vout = va;
  for (int pass = 0; pass < passes; ++pass) {
    const int shift = pass * 8;
    if (from_hist) {
      hipLaunchKernelGGL((k_radix_hist<uint32_t, true>), dim3(tiles), dim3(kBlock), 0, s, kin, nnz, shift, tiles, hist);
      hipLaunchKernelGGL((k_radix_scatter<uint32_t, true>), dim3(tiles), dim3(kBlock), 0, s, kin, vin, kout, vout, nnz,
                         shift, tiles, static_cast<const int32_t*>(hist));
    } else {
      hipLaunchKernelGGL((k_radix_hist<uint32_t, false>), dim3(tiles), dim3(kBlock), 0, s, kin, nnz, shift, tiles, hist);
      hipError_t e = scan_impl<int32_t>(hist, hist, static_cast<int64_t>(256) * tiles, scan_scratch, s);
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL((k_radix_scatter<uint32_t, false>), dim3(tiles), dim3(kBlock), 0, s, kin, vin, kout, vout,
                         nnz, shift, tiles, static_cast<const int32_t*>(hist));
    }
    kin = kout;
    vin = vout;
    const bool to_b = kout == ka;
    kout = to_b ? kb : ka;
    vout = to_b ? vb : va;
  }
  *result_in_b = kin == kb ? 1 : 0;
  return hipGetLastError();
}

int32_t gpk_transpose_buckets(int32_t n, int32_t nnz, int32_t* low) {
  // At 1,048,576 entries the buckets take 99 to 107 us where the sort takes 117
  // to 147 (128 against 190 at twice that).  Up to 256 columns the sort has one
  // pass.
  *low = 0;
  if (nnz < GPK_TRANSPOSE_BUCKETS_MIN_NNZ || nnz > INT_MAX - 2 * kTbTile || n <= 256) return 0;
  while (*low < kTbLowMax && ((n - 1) >> *low) >= kTbBuckets) ++*low;
  const int32_t buckets = ((n - 1) >> *low) + 1;
  return buckets <= kTbBuckets ? buckets : 0;
}

namespace {
// The scratch of a transpose by buckets, 16 bytes to a line of counts.
struct TbScratch {
  int32_t* offs;  // buckets x tiles counts, then their exclusive scan and total
  int32_t* scan;
  TbPiece* piece;
  int32_t* split;
  int32_t* counts;
  int64_t ints;
};
TbScratch tb_scratch(int32_t* base, int32_t buckets, int32_t nnz) {
  const int64_t words = static_cast<int64_t>(buckets) * grid_for(nnz, kTbTile);
  int64_t used = 0;
  const auto take = [&](int64_t ints) {
    int32_t* p = base + used;
    used += (ints + 3) / 4 * 4;
    return p;
  };
  TbScratch t{};
  t.offs = take(words + 1);
  t.scan = take(scan_scratch_ints(words));
  t.piece = reinterpret_cast<TbPiece*>(take((buckets + kTbMore) * static_cast<int64_t>(sizeof(TbPiece) / sizeof(int32_t))));
  t.split = take(kTbSplit);
  t.counts = take(static_cast<int64_t>(kTbSplit) * kTbCols);
  t.ints = used;
  return t;
}
}  // namespace

int64_t gpk_transpose_buckets_scratch_ints(int32_t buckets, int32_t nnz) {
  return tb_scratch(nullptr, buckets, nnz).ints;
}

hipError_t gpk_transpose_buckets_count(const int32_t* col, int32_t nnz, int32_t low, int32_t buckets, int32_t* scratch,
                                       hipStream_t s) {
  if (nnz <= 0 || buckets <= 0 || buckets > kTbBuckets || low < 0 || low > kTbLowMax) return hipErrorInvalidValue;
  const int32_t tiles = static_cast<int32_t>(grid_for(nnz, kTbTile));
  const int64_t words = static_cast<int64_t>(buckets) * tiles;
  const TbScratch t = tb_scratch(scratch, buckets, nnz);
  hipLaunchKernelGGL(k_tb_hist, dim3(tiles), dim3(kTbBlock), 0, s, col, nnz, low, buckets, tiles, t.offs);
  const hipError_t e = scan_impl<int32_t>(t.offs, t.offs, words, t.scan, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_tb_pieces, dim3(1), dim3(kTbBuckets), 0, s, static_cast<const int32_t*>(t.offs), buckets, tiles,
                     tb_share(nnz), t.piece, t.split);
  return hipGetLastError();
}

hipError_t gpk_transpose_buckets_move(const int32_t* ptr, const int32_t* col, const double* val, int32_t m, int32_t n,
                                      int32_t nnz, int32_t low, int32_t buckets, int32_t* scratch,
                                      gpk_row_val* rec, int32_t* at_ptr, int32_t* at_idx, double* at_val,
                                      hipStream_t s) {
  if (nnz <= 0 || buckets <= 0 || buckets > kTbBuckets || low < 0 || low > kTbLowMax) return hipErrorInvalidValue;
  const int32_t tiles = static_cast<int32_t>(grid_for(nnz, kTbTile));
  int bits = 0;
  while ((1 << bits) < buckets) ++bits;
  const TbScratch t = tb_scratch(scratch, buckets, nnz);
  hipLaunchKernelGGL(k_tb_partition, dim3(tiles), dim3(kTbBlock), 0, s, ptr, col, val, m, nnz, low,
                     buckets, bits, tiles, static_cast<const int32_t*>(t.offs), reinterpret_cast<int4*>(rec));
  hipLaunchKernelGGL(k_tb_piece_counts, dim3(kTbSplit), dim3(kTbBlock), 0, s, reinterpret_cast<const int4*>(rec), low,
                     static_cast<const TbPiece*>(t.piece), static_cast<const int32_t*>(t.split), t.counts);
  hipLaunchKernelGGL(k_tb_columns, dim3(buckets + kTbMore), dim3(kTbBlock), 0, s, reinterpret_cast<const int4*>(rec), n,
                     nnz, low, tb_share(nnz), static_cast<const TbPiece*>(t.piece),
                     static_cast<const int32_t*>(t.counts), at_ptr, at_idx, at_val);
  return hipGetLastError();
}

hipError_t gpk_col_bounds(const uint32_t* sorted_keys, int32_t nnz, int32_t n, int32_t* ptr, hipStream_t s) {
  hipLaunchKernelGGL(k_col_bounds, dim3(grid_for(static_cast<int64_t>(nnz) + 1)), dim3(kBlock), 0, s, sorted_keys,
                     nnz, n, ptr);
  return hipGetLastError();
}

hipError_t gpk_expand_rows(const int32_t* ptr, const double* val, int32_t m, gpk_row_val* rv, hipStream_t s) {
  if (m <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_expand_rows, dim3(grid_for(m)), dim3(kBlock), 0, s, ptr, val, m, rv);
  return hipGetLastError();
}

hipError_t gpk_transpose_gather(const int32_t* perm, const gpk_row_val* rv, int32_t nnz, int32_t* at_idx,
                                double* at_val, hipStream_t s) {
  if (nnz <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_transpose_gather, dim3(grid_for(nnz)), dim3(kBlock), 0, s, perm, rv, nnz, at_idx, at_val);
  return hipGetLastError();
}

hipError_t gpk_rows_unsorted(const int32_t* ptr, const int32_t* idx, int32_t rows, int32_t* flag, hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_csr_unsorted, dim3(grid_for(rows)), dim3(kBlock), 0, s, ptr, idx, rows, flag);
  return hipGetLastError();
}

int32_t gpk_csr_check_chunks(int32_t nnz) { return nnz > 0 ? static_cast<int32_t>(grid_for(nnz, kChkChunk)) : 0; }

hipError_t gpk_csr_check(gpk_csr_check_side a, gpk_csr_check_side t, hipStream_t s) {
  const int32_t ba = a.rows > 0 ? static_cast<int32_t>(grid_for(a.rows)) : 0;
  const int32_t bt = t.rows > 0 ? static_cast<int32_t>(grid_for(t.rows)) : 0;
  if (ba + bt == 0) return hipSuccess;
  hipLaunchKernelGGL(k_csr_check_ptr, dim3(ba + bt), dim3(kBlock), 0, s, a, t, ba);
  const int32_t ca = ba > 0 ? gpk_csr_check_chunks(a.nnz) : 0, ct = bt > 0 ? gpk_csr_check_chunks(t.nnz) : 0;
  if (ca + ct > 0)
    hipLaunchKernelGGL(k_csr_check_entries, dim3(ca + ct), dim3(kBlock), 0, s, a, t, ca, ct);
  return hipGetLastError();
}

hipError_t gpk_csr_check_rows(const int32_t* ptr, const int32_t* idx, int32_t rows, int32_t cols, int32_t nnz,
                              int32_t* flags, hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_csr_check, dim3(grid_for(rows)), dim3(kBlock), 0, s, ptr, idx, rows, cols, nnz, flags);
  return hipGetLastError();
}

hipError_t gpk_sort_rows_in_place(const int32_t* ptr, int32_t* idx, double* val, int32_t rows, hipStream_t s) {
  if (rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_sort_rows, dim3(grid_for(rows)), dim3(kBlock), 0, s, ptr, idx, val, rows);
  return hipGetLastError();
}

}  // extern "C"
