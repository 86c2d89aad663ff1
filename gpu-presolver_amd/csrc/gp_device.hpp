// Device-side helpers shared by the HIP kernel files (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "gp_walk.hpp"

namespace gpdev {

constexpr int kBlock = 256;  // 4 waves of 64 lanes
constexpr int kWaves = kBlock / 64;

__host__ inline unsigned grid_for(int64_t n, int block = kBlock) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > 0x7fffffff) g = 0x7fffffff;
  return static_cast<unsigned>(g);
}

__device__ inline int lane_id() { return static_cast<int>(threadIdx.x & 63); }

__device__ inline uint64_t lanemask_lt(int lane) {
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Flag and counter updates aggregated per wave: the calling lanes (those for
// which the event happened) elect their lowest lane, which issues a single
// atomic for the whole wave.  Safe in divergent code: only the lanes that
// reach the call take part.
__device__ inline bool wave_leader(uint64_t* active) {
  const uint64_t m = __ballot(1);
  *active = m;
  return lane_id() == __ffsll(static_cast<unsigned long long>(m)) - 1;
}
// A yes/no flag word (0 until some thread sets it to 1, read only after the
// kernel): the wave's leader stores 1 with a plain store, which lands in its
// XCD's L2 and is written back at the end of the kernel.  No read-modify-
// write and no device-coherent load: when most waves of a large grid set the
// same flag, those would all queue on one address at one memory channel.
__device__ inline void wave_set_flag(int32_t* addr) {
  uint64_t m;
  if (wave_leader(&m)) __hip_atomic_store(addr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Max only ever grows the word, so a leader that reads a value at least its
// own skips the atomic.
__device__ inline void wave_max(int32_t* addr, int32_t v) {
  uint64_t m;
  if (wave_leader(&m) && __hip_atomic_load(addr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < v)
    atomicMax(addr, v);
}
__device__ inline void wave_add1(int32_t* addr) {
  uint64_t m;
  if (wave_leader(&m)) atomicAdd(addr, static_cast<int32_t>(__popcll(m)));
}

// Orders a wave's LDS stores before its own later loads (and the reverse);
// no other wave is met.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// s + t[0] + t[1] + ..., added one after the other; t is 16-byte aligned LDS,
// and where n is odd t[n] holds +0.  Eight pairs are on their way at a time.
__device__ inline double add_in_order(double s, const double* t, int n) {
  const double2* p = reinterpret_cast<const double2*>(t);
  const int pairs = (n + 1) / 2;
  int i = 0;
  for (; i + 8 <= pairs; i += 8) {
    double2 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = p[i + k];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      s += v[k].x;
      s += v[k].y;
    }
  }
  for (; i < pairs; ++i) {
    const double2 v = p[i];
    s += v.x;
    s += v.y;
  }
  return s;
}

// Rows of more entries than this get a wave each in the kernels that otherwise
// give a row to a thread: a thread walks a row at a few hundred ns an entry
// (1.3 ms for 3,000), a wave needs about 3 us for a row and 10 ns an entry.
constexpr int kLongRow = 128;

// Calls f(row, begin, end) in all lanes of a wave for every row of more than
// `longer` entries that falls to it, in a launch whose blocks from
// `first_block` on are given to long rows.  A wave looks at every waves-th group of g
// neighbouring rows, so neighbouring long rows go to different waves: g = 1
// up to 262,144 rows (a line of row pointers read for each, 16 MB of L2 reads
// in all), past that the 16 rows of a line.  The row pointers of kLook groups
// are loaded together: without a long row these blocks are gone in a few
// memory round trips.
// There are waves for as many long rows as the entries can make, up to eight
// blocks a CU: 50,000 rows of 200 to 300 entries among a million short ones
// are six for each wave (row activity 386 us, presolve 20.7 ms; 470 us and 25 ms
// with one block a CU, 525 us and 26 ms with a thread or tile for every row).  On
// 1M rows with no long one the blocks cost 2 us of 170.  nnz only sets the
// number: every long row is found by one block as well.
inline unsigned long_row_blocks(int32_t m, int64_t nnz) {
  const int64_t most = nnz / (kLongRow + 1) + 1;
  const unsigned b = grid_for(most < m ? most : m, kWaves);
  return b < 2048 ? b : 2048;
}

template <class F>
__device__ __forceinline__ void wave_long_rows(const int32_t* __restrict__ ptr, int32_t m, int32_t longer,
                                               int32_t first_block, F&& f) {
  constexpr int kLook = 8;
  const int lane = lane_id();
  const int g = m <= 262144 ? 1 : 16;
  const int64_t waves = static_cast<int64_t>(static_cast<int32_t>(gridDim.x) - first_block) * kWaves;
  const int64_t w0 = (static_cast<int64_t>(static_cast<int32_t>(blockIdx.x) - first_block) * kWaves + (threadIdx.x >> 6)) * g;
  const int64_t mine = (lane / g) * waves * g + lane % g;
  for (int64_t look = w0; look < m; look += kLook * 64 * waves) {
    bool any = false;
#pragma unroll
    for (int u = 0; u < kLook; ++u) {
      const int64_t r = look + u * 64 * waves + mine;
      any = any || (r < m && ptr[r + 1] - ptr[r] > longer);
    }
    if (__ballot(any) == 0) continue;
#pragma unroll 1
    for (int u = 0; u < kLook; ++u) {
      const int64_t first = look + u * 64 * waves, r = first + mine;
      const int32_t rb = r < m ? ptr[r] : 0, re = r < m ? ptr[r + 1] : 0;
      uint64_t todo = __ballot(re - rb > longer);
      while (todo) {
        const int q = __ffsll(static_cast<unsigned long long>(todo)) - 1;
        todo &= todo - 1;
        f(first + (q / g) * waves * g + q % g, __shfl(rb, q, 64), __shfl(re, q, 64));
      }
    }
  }
}

// The entries [b, e) of a row walked by a wave, kRowChunk at a time (the next
// ones on their way meanwhile): load(column, in_range) gathers, term(value,
// gathered, in_range, t) forms kSums terms of the entry, each kind of which is
// added in the order of the entries; lane k < kSums returns the sum of kind k.
// term returns false for an entry that adds nothing: its terms must be +0,
// which leaves a sum that started at +0 as it is (no such sum is -0).
// s_t: kSums * kRowPitch doubles of LDS, 16-byte aligned, the wave's own.
// Bound by the chain of adds, about 3 ns an entry.
constexpr int kRowSteps = 4;
constexpr int kRowChunk = 64 * kRowSteps;
constexpr int kRowPitch = kRowChunk + 2;  // the kinds start in different banks

template <int kSums, class G, class Load, class Term>
__device__ __forceinline__ double wave_row_sums(const int32_t* __restrict__ idx, const double* __restrict__ val,
                                                int32_t b, int32_t e, double* s_t, Load&& load, Term&& term) {
  const uint32_t lane = static_cast<uint32_t>(lane_id()), n = row_length(b, e);
  double a[kRowSteps], acc = 0.0;
  int32_t j[kRowSteps];
#pragma unroll
  for (int k = 0; k < kRowSteps; ++k) {
    const int32_t p = row_entry(b, e, 64 * k + lane);
    a[k] = val[p];
    j[k] = idx[p];
  }
#pragma unroll 1
  for (uint32_t c = 0; c < n; c += kRowChunk) {
    G g[kRowSteps];
#pragma unroll
    for (int k = 0; k < kRowSteps; ++k) g[k] = load(j[k], a[k], c + 64 * k + lane < n);
    double t[kRowSteps][kSums];
    bool any = false;
#pragma unroll
    for (int k = 0; k < kRowSteps; ++k) any = term(a[k], g[k], c + 64 * k + lane < n, t[k]) || any;
#pragma unroll
    for (int k = 0; k < kRowSteps; ++k) {  // the last entry again past the row's end
      const int32_t p = row_entry(b, e, c + kRowChunk + 64 * k + lane);
      a[k] = val[p];
      j[k] = idx[p];
    }
    if (__ballot(any) == 0) continue;
#pragma unroll
    for (int k = 0; k < kRowSteps; ++k)
#pragma unroll
      for (int q = 0; q < kSums; ++q) s_t[q * kRowPitch + 64 * k + lane] = t[k][q];
    wave_lds_fence();
    if (lane < kSums) acc = add_in_order(acc, s_t + lane * kRowPitch, static_cast<int>(min(static_cast<uint32_t>(kRowChunk), n - c)));
    wave_lds_fence();
  }
  return acc;
}

// Inclusive wave64 prefix sum of an int32.
__device__ inline int32_t wave_inclusive_sum(int32_t v) {
  const int lane = lane_id();
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  return v;
}

// Exclusive block prefix sum of one int32 per thread (blockDim.x == kBlock).
// Returns the thread's exclusive prefix; *total gets the block sum.
__device__ inline int32_t block_exclusive_sum(int32_t v, int32_t* total) {
  __shared__ int32_t s_wave[kBlock / 64];
  const int lane = lane_id();
  const int wave = static_cast<int>(threadIdx.x >> 6);
  const int32_t inc = wave_inclusive_sum(v);
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  int32_t wave_base = 0;
  int32_t sum = 0;
#pragma unroll
  for (int w = 0; w < kBlock / 64; ++w) {
    const int32_t t = s_wave[w];
    if (w < wave) wave_base += t;
    sum += t;
  }
  __syncthreads();
  *total = sum;
  return wave_base + inc - v;
}

// Replace-unless-dominated semantics of the reference's double CAS loops
// (rules/rule_singleton_rows.cu:18-50): slot := v unless slot >= v (max) or
// slot <= v (min).
__device__ inline void atomic_max_f64(double* addr, double v) {
  unsigned long long* a = reinterpret_cast<unsigned long long*>(addr);
  unsigned long long old = __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (true) {
    const double cur = __longlong_as_double(static_cast<long long>(old));
    if (cur >= v) return;
    const unsigned long long want = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned long long prev = atomicCAS(a, old, want);
    if (prev == old) return;
    old = prev;
  }
}

__device__ inline void atomic_min_f64(double* addr, double v) {
  unsigned long long* a = reinterpret_cast<unsigned long long*>(addr);
  unsigned long long old = __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  while (true) {
    const double cur = __longlong_as_double(static_cast<long long>(old));
    if (cur <= v) return;
    const unsigned long long want = static_cast<unsigned long long>(__double_as_longlong(v));
    const unsigned long long prev = atomicCAS(a, old, want);
    if (prev == old) return;
    old = prev;
  }
}

}  // namespace gpdev
