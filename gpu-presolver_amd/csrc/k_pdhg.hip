// Kernels of the on-device LP solver that takes the reduced LP from presolve
// (restarted primal-dual hybrid gradient, PDHG, on the Ruiz-scaled LP):
// the two half steps of an iteration, Ruiz scaling, sparse products for the
// norm estimate, and the residual sums of the KKT check.
//
// Every kernel that walks the rows of a CSR matrix (A, or AT for the
// columns) runs over row blocks built once per solve, of at most
// GPK_PDHG_ENTRY_BUDGET entries each: up to 256 consecutive short rows, whose
// products are staged in LDS by coalesced loads and then summed one row per
// thread, or a row of more than GPK_PDHG_LONG_ROW entries or a part of one,
// reduced by the whole workgroup; the workgroup that finishes a row's last
// part combines the parts in their order.  A column of AT with thousands of
// entries therefore runs neither on one lane nor on one workgroup.  Each row's
// sum has a fixed order (given by the blocks, which depend only on the
// matrix), and every sum over a vector goes through per-block partial sums
// reduced in block order by one workgroup, so a solve is deterministic run to
// run.
//
// What bounds them is a chain of memory round trips, a microsecond and more
// each under load: the block's bounds, its entries (with the row pointers and
// the vectors of its rows, which need nothing but the bounds), the gathers
// and, for a split row, the meeting of its parts; on large LPs the gathers
// (a 128-byte line into the CU's cache for 8 bytes).  A reduced LP of 300,000
// rows x 450,000 columns, 2.4 million entries: primal half step 31.5 -> 25.2
// us, dual 18.8 -> 18.1; of 13,000 x 27,000, 33,000 entries: 4.7 -> 3.8 us
// (a row of up to 256 entries on one thread, the block's row pointers and the
// rows' vectors in trips of their own before).  Entries or gathers loaded
// without a place in the caches were 1.2 to 2 times slower: the matrix stays
// there from launch to launch.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "gp_device.hpp"
#include "gp_kernels.h"

using namespace gpdev;

// The parts of a split row meet through relaxed atomics whose order an empty
// asm statement gives (k_rows): that the exchange's answer comes back only once
// the sum is where every XCD's atomic loads see it is a property of this chip's
// device-scope atomics, not of the memory model.  Another target needs
// a release and an acquire there.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "k_pdhg.hip orders the parts of a row as gfx950 does"
#endif

namespace {

constexpr int kEntryBudget = GPK_PDHG_ENTRY_BUDGET;
constexpr int kStage = kEntryBudget / kBlock;  // staged entries per thread
constexpr int kPartials = 4;
// A thread sums a row by itself (about 15 ns an entry, one after the other), or
// a wave does, at about 200 ns a row.  A block's rows of more than kThreadRow
// entries go to its waves in turn where those are done first, which the plan says
// (GPK_ROWS_BY_WAVE).  (With every such row left to the wave of its thread, a
// block's rows were all one wave's: 128 iterations with rows of 40 entries
// 10.4 ms, 7.4 with a thread a row and 7.2 this way; of 100 entries 9.0, 7.7 and
// 7.1; columns of 200 entries 9.2, 9.8 and 7.7.)
constexpr int kThreadRow = 32;
bool rows_by_wave(int32_t rows, int32_t longest) { return rows > 0 && 200 * rows < kWaves * 15 * longest; }
static_assert(kEntryBudget % kBlock == 0, "entry budget in whole strides");

__device__ inline double clampd(double v, double lo, double hi) { return fmin(fmax(v, lo), hi); }

struct SumOp {
  static __device__ double identity() { return 0.0; }
  static __device__ double combine(double a, double b) { return a + b; }
};
struct MaxOp {
  static __device__ double identity() { return 0.0; }
  static __device__ double combine(double a, double b) { return fmax(a, b); }
};

// Combination of kN values over the block in a fixed order (lanes by shuffle
// tree, waves in index order); every thread gets the results.
template <class C, int kN>
__device__ inline void block_combine(double (&v)[kN], double (*s_w)[kBlock / 64]) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1)
#pragma unroll
    for (int k = 0; k < kN; ++k) v[k] = C::combine(v[k], __shfl_down(v[k], d, 64));
  if (lane_id() == 0)
#pragma unroll
    for (int k = 0; k < kN; ++k) s_w[k][threadIdx.x >> 6] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kN; ++k) {
    v[k] = s_w[k][0];
#pragma unroll
    for (int w = 1; w < kBlock / 64; ++w) v[k] = C::combine(v[k], s_w[k][w]);
  }
  __syncthreads();
}
template <class C>
__device__ inline double block_combine(double v, double (*s_w)[kBlock / 64]) {
  double t[1] = {v};
  block_combine<C>(t, s_w);
  return t[0];
}

// ---- row operations --------------------------------------------------------
// elem(col, val, f): the term of an entry, f = factor() the same for all; load(r): the row's own vector entries,
// loaded before its terms are known; row(r, acc, own, t): consumes the row's
// combined terms (and, with kTerms, adds its KKT terms to t).
struct NoOwn {};

// y = M v, v scaled by 1 / sqrt(sumsq[0]) where that is given and positive
// (the power iteration's normalisation, read from device memory so the host
// need not wait).
struct OpSpmv {
  using Comb = SumOp;
  using Own = NoOwn;
  static constexpr bool kTerms = false;
  const double* v;
  const double* sumsq;
  double* out;
  __device__ double factor() const {
    const double s = sumsq ? sumsq[0] : 0.0;
    return s > 0.0 ? 1.0 / sqrt(s) : 1.0;
  }
  __device__ double elem(int32_t col, double val, double f) const { return val * (v[col] * f); }
  __device__ Own load(int32_t) const { return {}; }
  __device__ void row(int32_t r, double acc, Own, double*) const { out[r] = acc; }
};

// y = M v and, term [0], the sum of y^2.
struct OpSpmvSq {
  using Comb = SumOp;
  using Own = NoOwn;
  static constexpr bool kTerms = true;
  const double* v;
  double* out;
  __device__ double factor() const { return 1.0; }
  __device__ double elem(int32_t col, double val, double) const { return val * v[col]; }
  __device__ Own load(int32_t) const { return {}; }
  __device__ void row(int32_t r, double acc, Own, double* t) const {
    out[r] = acc;
    t[0] += acc * acc;
  }
};

// Ruiz: d[r] /= sqrt(max |entry| of row r) (rows without a nonzero keep d).
struct OpRuiz {
  using Comb = MaxOp;
  using Own = double;
  static constexpr bool kTerms = false;
  double* d;
  __device__ double factor() const { return 1.0; }
  __device__ double elem(int32_t, double val, double) const { return fabs(val); }
  __device__ Own load(int32_t r) const { return d[r]; }
  __device__ void row(int32_t r, double acc, Own o, double*) const {
    if (acc > 0.0) d[r] = o / sqrt(acc);
  }
};

// Halpern weight of iteration k since the restart: (k + 1) / (k + 2), with
// k = step[2] (the count at the start of the launch) + j.
__device__ inline double halpern_weight(const double* step, int32_t j) {
  const double k = step[2] + static_cast<double>(j);
  return (k + 1.0) / (k + 2.0);
}

// Primal half step over the rows of AT: xn = proj_[l,u](x - tau (c - A^T y))
// and xbar = 2 xn - x (the extrapolated point the dual step reads).
// Averaged PDHG: x <- xn, x_acc += xn (the running sum).  Reflected Halpern
// PDHG: x_acc <- xn (the PDHG point T(z)), x <- w xbar + (1 - w) x0, since
// xbar is also the reflected point 2 T(z) - z.
template <bool kHalpern>
struct OpPrimal {
  using Comb = SumOp;
  static constexpr bool kTerms = false;
  const double* y;
  const double* c;
  const double* l;
  const double* u;
  const double* step;
  double* x;
  double* xbar;
  double* x_acc;
  const double* x0;
  int32_t j;
  struct Own {
    double c, l, u, x, acc;  // acc: x0 (Halpern) or the running sum
  };
  __device__ double factor() const { return 1.0; }
  __device__ double elem(int32_t col, double val, double) const { return val * y[col]; }
  __device__ Own load(int32_t r) const { return {c[r], l[r], u[r], x[r], kHalpern ? x0[r] : x_acc[r]}; }
  __device__ void row(int32_t r, double aty, const Own& o, double*) const {
    const double g = o.c - aty;
    const double xo = o.x;
    const double xn = clampd(xo - step[0] * g, o.l, o.u);
    const double xb = 2.0 * xn - xo;
    xbar[r] = xb;
    if (kHalpern) {
      const double w = halpern_weight(step, j);
      x_acc[r] = xn;
      x[r] = w * xb + (1.0 - w) * o.acc;
    } else {
      x[r] = xn;
      x_acc[r] = o.acc + xn;
    }
  }
};

// Dual half step over the rows of A: yn = yt + sigma proj_[AL,AU](-yt / sigma)
// with yt = y - sigma A xbar (the Moreau form of the projected dual ascent).
// Averaged: y <- yn, y_acc += yn.  Reflected Halpern: y_acc <- yn,
// y <- w (2 yn - y) + (1 - w) y0.
template <bool kHalpern>
struct OpDual {
  using Comb = SumOp;
  static constexpr bool kTerms = false;
  const double* xbar;
  const double* AL;
  const double* AU;
  const double* step;
  double* y;
  double* y_acc;
  const double* y0;
  int32_t j;
  struct Own {
    double AL, AU, y, acc;
  };
  __device__ double factor() const { return 1.0; }
  __device__ double elem(int32_t col, double val, double) const { return val * xbar[col]; }
  __device__ Own load(int32_t i) const { return {AL[i], AU[i], y[i], kHalpern ? y0[i] : y_acc[i]}; }
  __device__ void row(int32_t i, double ax, const Own& o, double*) const {
    const double sigma = step[1];
    const double yo = o.y;
    const double yt = yo - sigma * ax;
    const double yn = yt + sigma * clampd(-yt / sigma, o.AL, o.AU);
    if (kHalpern) {
      const double w = halpern_weight(step, j);
      y_acc[i] = yn;
      y[i] = w * (2.0 * yn - yo) + (1.0 - w) * o.acc;
    } else {
      y[i] = yn;
      y_acc[i] = o.acc + yn;
    }
  }
};

// KKT terms of the rows (A, v = x): [0] squared violation of Ax against
// [AL, AU], [1] the rows' dual-objective terms of y, [2] squared bound
// magnitude (the larger finite |AL|, |AU|), [3] y^2 where the bound of y's
// sign is infinite (a dual infeasibility).
struct OpRowTerms {
  using Comb = SumOp;
  static constexpr bool kTerms = true;
  const double* x;
  const double* AL;
  const double* AU;
  const double* y;
  struct Own {
    double AL, AU, y;
  };
  __device__ double factor() const { return 1.0; }
  __device__ double elem(int32_t col, double val, double) const { return val * x[col]; }
  __device__ Own load(int32_t i) const { return {AL[i], AU[i], y[i]}; }
  __device__ void row(int32_t, double ax, const Own& o, double* t) const {
    const double lo = o.AL, hi = o.AU;
    const double viol = ax - clampd(ax, lo, hi);
    t[0] += viol * viol;
    const double yi = o.y;
    if (yi > 0.0) {
      if (isfinite(lo)) t[1] += yi * lo;
      else t[3] += yi * yi;
    } else if (yi < 0.0) {
      if (isfinite(hi)) t[1] += yi * hi;
      else t[3] += yi * yi;
    }
    const double b = fmax(isfinite(lo) ? fabs(lo) : 0.0, isfinite(hi) ? fabs(hi) : 0.0);
    t[2] += b * b;
  }
};

// KKT terms of the columns (AT, v = y): g = c - A^T y and lambda its
// projection on the reduced-cost cone of the column's bounds (lambda >= 0
// needs a finite lower bound, lambda <= 0 a finite upper one); [0] squared
// dual residual (g - lambda), [1] the columns' dual-objective terms, [2] c^2,
// [3] c x; z = lambda when z is given.
struct OpColTerms {
  using Comb = SumOp;
  static constexpr bool kTerms = true;
  const double* y;
  const double* c;
  const double* l;
  const double* u;
  const double* x;
  double* z;
  struct Own {
    double c, l, u, x;
  };
  __device__ double factor() const { return 1.0; }
  __device__ double elem(int32_t col, double val, double) const { return val * y[col]; }
  __device__ Own load(int32_t j) const { return {c[j], l[j], u[j], x[j]}; }
  __device__ void row(int32_t j, double aty, const Own& o, double* t) const {
    const double g = o.c - aty;
    const bool lo_fin = isfinite(o.l), hi_fin = isfinite(o.u);
    const double lam = clampd(g, hi_fin ? -INFINITY : 0.0, lo_fin ? INFINITY : 0.0);
    if (z) z[j] = lam;
    t[0] += (g - lam) * (g - lam);
    if (lam > 0.0) t[1] += lam * o.l;
    else if (lam < 0.0) t[1] += lam * o.u;
    t[2] += o.c * o.c;
    t[3] += o.c * o.x;
  }
};

// acc with s[b .. e) combined one after the other, four at a time on their way.
template <class C>
__device__ inline double combine_in_order(const double* s, int32_t b, int32_t e) {
  double acc = C::identity();
  for (int32_t q = b; q < e; q += 4) {
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = s[min(q + k, e - 1)];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (q + k < e) acc = C::combine(acc, v[k]);
  }
  return acc;
}

template <class Op>
__global__ __launch_bounds__(kBlock) void k_rows(const int32_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                 const double* __restrict__ val,
                                                 const gpk_row_block* __restrict__ blk, double* part_sum,
                                                 int32_t* part_count, double* __restrict__ partial, Op op) {
  using C = typename Op::Comb;
  __shared__ double s_val[kEntryBudget];
  __shared__ double s_w[kPartials][kBlock / 64];
  __shared__ int32_t s_last;
  const int32_t bid = static_cast<int32_t>(blockIdx.x);
  const gpk_row_block b = blk[bid], next = blk[bid + 1];
  const int32_t nr = next.row - b.row, cnt = next.entry - b.entry;
  const int tid = static_cast<int>(threadIdx.x);
  const double factor = op.factor();
  double t[kPartials] = {0.0, 0.0, 0.0, 0.0};
  int32_t ci[kStage];
  double cv[kStage];
  const int32_t* __restrict__ bi = idx + b.entry;
  const double* __restrict__ bv = val + b.entry;
#pragma unroll
  for (int k = 0; k < kStage; ++k) {
    const int32_t q = tid + k * kBlock;
    if (q < cnt) {
      ci[k] = bi[q];
      cv[k] = bv[q];
    }
  }
  // A block's few rows go to its waves in turn where those sum the longer ones
  // (more rows are spread as they stand, and load their own vectors in order: 150
  // entries in each twentieth of rows of 8 are 4.7 ms that way, 4.95 in turn).
  const bool waves = b.parts == GPK_ROWS_BY_WAVE;
  const int at = waves && nr <= 64 ? lane_id() * kWaves + (tid >> 6) : tid;
  const bool mine = at < (b.parts > 0 ? 1 : nr);
  const int32_t r = b.row + (mine ? at : 0);
  typename Op::Own own{};
  int32_t pb = 0, pe = 0;
  if (mine) {
    own = op.load(r);
    if (b.parts <= 0) {
      pb = ptr[r] - b.entry;
      pe = ptr[r + 1] - b.entry;
    }
  }
#pragma unroll
  for (int k = 0; k < kStage; ++k)
    if (tid + k * kBlock < cnt) cv[k] = op.elem(ci[k], cv[k], factor);
  if (b.parts <= 0) {
#pragma unroll
    for (int k = 0; k < kStage; ++k)
      if (tid + k * kBlock < cnt) s_val[tid + k * kBlock] = cv[k];
    __syncthreads();
    double acc = C::identity();
    const bool by_wave = waves && pe - pb > kThreadRow;
    if (!by_wave) acc = combine_in_order<C>(s_val, pb, pe);
    for (uint64_t todo = __ballot(by_wave); todo != 0; todo &= todo - 1) {
      const int q = __ffsll(static_cast<unsigned long long>(todo)) - 1;
      const int32_t rb = __shfl(pb, q, 64), re = __shfl(pe, q, 64);
      double a = C::identity();
      for (int32_t p = rb + lane_id(); p < re; p += 64) a = C::combine(a, s_val[p]);
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) a = C::combine(a, __shfl_xor(a, d, 64));
      if (lane_id() == q) acc = a;
    }
    if (mine) op.row(r, acc, own, t);
  } else {
    // one row or a part of one: each thread its entries, then the tree
    double a = C::identity();
#pragma unroll
    for (int k = 0; k < kStage; ++k)
      if (tid + k * kBlock < cnt) a = C::combine(a, cv[k]);
    a = block_combine<C>(a, s_w);
    bool whole = b.parts == 1;
    if (!whole) {
      // The sum is exchanged, and counted once the exchange has answered (the
      // count's increment is made to depend on it): it is then where every
      // XCD's atomic loads see it, and the sums are all that the last part
      // reads of the others.  A release instead writes back the L2's dirty lines
      // at every part: 57 us for a primal half step that takes 27 this way.
      if (tid == 0) {
        const long long old = __hip_atomic_exchange(reinterpret_cast<long long*>(part_sum) + bid,
                                                    __double_as_longlong(a), __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        int32_t one = 1;
        asm volatile("" : "+v"(one) : "v"(old) : "memory");
        s_last = __hip_atomic_fetch_add(part_count + (bid - b.part), one, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT) == b.parts - 1;
      }
      __syncthreads();
      whole = s_last != 0;
      if (whole) {
        a = C::identity();
        for (int32_t k = tid; k < b.parts; k += kBlock)
          a = C::combine(a, __hip_atomic_load(part_sum + (bid - b.part + k), __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT));
        a = block_combine<C>(a, s_w);
        if (tid == 0)  // for the next launch
          __hip_atomic_store(part_count + (bid - b.part), 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (whole && tid == 0) op.row(r, a, own, t);
    if constexpr (Op::kTerms) {
      // A row's terms stand in its first part's place, whichever block was
      // the last; the other places are empty.
      if (tid < kPartials) {
        if (b.part > 0) partial[static_cast<int64_t>(bid) * kPartials + tid] = 0.0;
      }
      if (whole && tid == 0)
#pragma unroll
        for (int k = 0; k < kPartials; ++k) partial[static_cast<int64_t>(bid - b.part) * kPartials + k] = t[k];
      return;
    }
  }
  if constexpr (Op::kTerms) {
    block_combine<SumOp>(t, s_w);
    if (tid == 0)
#pragma unroll
      for (int k = 0; k < kPartials; ++k) partial[static_cast<int64_t>(bid) * kPartials + k] = t[k];
  }
}

// out[p] = M.val[p] * drow[row(p)] * dcol[idx[p]], over the same row blocks
// (the threads of a block's rows write each entry's row into LDS).
__global__ __launch_bounds__(kBlock) void k_rows_scale(const int32_t* __restrict__ ptr,
                                                       const int32_t* __restrict__ idx,
                                                       const double* __restrict__ val,
                                                       const gpk_row_block* __restrict__ blk,
                                                       const double* __restrict__ drow,
                                                       const double* __restrict__ dcol, double* __restrict__ out) {
  __shared__ uint8_t s_row[kEntryBudget];
  __shared__ double s_d[kBlock];
  const gpk_row_block b = blk[blockIdx.x], next = blk[blockIdx.x + 1];
  const int32_t nr = b.parts > 0 ? 1 : next.row - b.row, cnt = next.entry - b.entry;
  const int tid = static_cast<int>(threadIdx.x);
  int32_t ci[kStage];
  double cv[kStage];
#pragma unroll
  for (int k = 0; k < kStage; ++k) {
    const int32_t q = tid + k * kBlock;
    if (q < cnt) {
      ci[k] = idx[b.entry + q];
      cv[k] = val[b.entry + q];
    }
  }
  if (tid < nr) {
    s_d[tid] = drow[b.row + tid];
    if (b.parts <= 0)
      for (int32_t q = ptr[b.row + tid] - b.entry, e = ptr[b.row + tid + 1] - b.entry; q < e; ++q)
        s_row[q] = static_cast<uint8_t>(tid);
  }
  double g[kStage];
#pragma unroll
  for (int k = 0; k < kStage; ++k)
    if (tid + k * kBlock < cnt) g[k] = dcol[ci[k]];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kStage; ++k) {
    const int32_t q = tid + k * kBlock;
    if (q < cnt) out[b.entry + q] = cv[k] * s_d[b.parts > 0 ? 0 : s_row[q]] * g[k];
  }
}

// out = a * x + b * y (any of the inputs may alias the output).
__global__ void k_pdhg_axpby(double a, const double* x, double b, const double* y, double* out, int32_t n) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = a * x[i] + (y ? b * y[i] : 0.0);
}

__global__ void k_pdhg_mul(const double* __restrict__ x, const double* __restrict__ d, double* __restrict__ out,
                           int32_t n) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = x[i] * d[i];
}

// Scaled vectors: multiply (mul) or divide (!mul) by d; infinities stay.
__global__ void k_pdhg_scale_vec(const double* __restrict__ v, const double* __restrict__ d, double* __restrict__ out,
                                 int32_t n, int32_t mul) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = mul ? v[i] * d[i] : v[i] / d[i];
}

// Sum of (a - b)^2 and of a^2 (b may be null) into partials [0], [1].
__global__ __launch_bounds__(kBlock) void k_pdhg_sq_terms(const double* __restrict__ a,
                                                          const double* __restrict__ b, int32_t n,
                                                          double* __restrict__ partial) {
  __shared__ double s_w[2][kBlock / 64];
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  double t[2] = {0.0, 0.0};
  if (i < n) {
    const double d = a[i] - (b ? b[i] : 0.0);
    t[0] = d * d;
    t[1] = a[i] * a[i];
  }
  block_combine<SumOp>(t, s_w);
  if (threadIdx.x == 0) {
    double* o = partial + static_cast<int64_t>(blockIdx.x) * kPartials;
    o[0] = t[0];
    o[1] = t[1];
    o[2] = 0.0;
    o[3] = 0.0;
  }
}

// out[k] = sum over blocks of partial[b * kPartials + k], in block order (one
// workgroup: thread t sums blocks t, t + 256, ..., then the block tree).
__global__ __launch_bounds__(kBlock) void k_pdhg_reduce(const double* __restrict__ partial, int32_t blocks,
                                                        double* __restrict__ out) {
  __shared__ double s_w[kPartials][kBlock / 64];
  constexpr int kLook = 4;
  double t[kPartials] = {};
  for (int32_t b = threadIdx.x; b < blocks; b += kLook * kBlock) {
    double v[kLook][kPartials];
#pragma unroll
    for (int u = 0; u < kLook; ++u)
#pragma unroll
      for (int k = 0; k < kPartials; ++k)
        if (b + u * kBlock < blocks) v[u][k] = partial[static_cast<int64_t>(b + u * kBlock) * kPartials + k];
#pragma unroll
    for (int u = 0; u < kLook; ++u)
#pragma unroll
      for (int k = 0; k < kPartials; ++k)
        if (b + u * kBlock < blocks) t[k] += v[u][k];
  }
  block_combine<SumOp>(t, s_w);
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < kPartials; ++k) out[k] = t[k];
}

// Start vector of the power iteration: 0.5 + frac(i * golden ratio).
__global__ void k_pdhg_seed(double* __restrict__ p, int32_t n) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const double t = static_cast<double>(i) * 0.6180339887498949;
    p[i] = 0.5 + (t - floor(t));
  }
}

// out = proj_[l,u](xs * d): a scaled primal point back in the LP's own
// variables, clamped so the rounding of l / d * d cannot leave a bound.
__global__ void k_pdhg_unscale_x(const double* __restrict__ xs, const double* __restrict__ d,
                                 const double* __restrict__ l, const double* __restrict__ u, double* __restrict__ out,
                                 int32_t n) {
  const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) out[j] = clampd(xs[j] * d[j], l[j], u[j]);
}

// x = projection of 0 on [l, u].
__global__ void k_pdhg_project_zero(const double* __restrict__ l, const double* __restrict__ u,
                                    double* __restrict__ x, int32_t n) {
  const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) x[j] = clampd(0.0, l[j], u[j]);
}

// The row after the last of the block that starts at row r; *by_wave: its rows
// are the waves'.
int32_t block_end(const int32_t* ptr, int32_t rows, int32_t r, bool* by_wave) {
  *by_wave = false;
  if (ptr[r + 1] - ptr[r] > GPK_PDHG_LONG_ROW) return r + 1;
  const int32_t start = r;
  int32_t cnt = 0, longs = 0, longest = 0;
  while (r < rows && r - start < kBlock) {
    const int32_t len = ptr[r + 1] - ptr[r];
    if (len > GPK_PDHG_LONG_ROW || cnt + len > kEntryBudget) break;
    if (__builtin_expect(len > kThreadRow, 0)) {
      ++longs;
      longest = len > longest ? len : longest;
    }
    cnt += len;
    ++r;
  }
  *by_wave = r - start > 1 && rows_by_wave(longs, longest);
  return r;
}

template <class Op>
hipError_t launch_rows(const gpk_rows& R, const Op& op, double* partial, hipStream_t s) {
  if (R.blocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rows<Op>, dim3(static_cast<unsigned>(R.blocks)), dim3(kBlock), 0, s, R.M.ptr, R.M.idx, R.M.val,
                     R.blk, R.part_sum, R.part_count, partial, op);
  return hipGetLastError();
}

hipError_t launch_reduce(const double* partial, int32_t blocks, double* out, hipStream_t s) {
  hipLaunchKernelGGL(k_pdhg_reduce, dim3(1), dim3(kBlock), 0, s, partial, blocks, out);
  return hipGetLastError();
}

}  // namespace

extern "C" {

int64_t gpk_pdhg_row_plan_most(int32_t rows, int32_t nnz) {
  // A block ends at 256 rows, or past the budget less a row, or before a long row
  // or at the end; a long row's parts are its whole budgets and one.
  const int64_t e = nnz, longs = e / (GPK_PDHG_LONG_ROW + 1);
  return rows / kBlock + e / (kEntryBudget - GPK_PDHG_LONG_ROW) + (longs + 1) + (e / kEntryBudget + longs);
}

int32_t gpk_pdhg_row_plan(const int32_t* ptr, int32_t rows, gpk_row_block* out) {
  int32_t nb = 0;
  for (int32_t r = 0; r < rows;) {
    bool by_wave;
    const int32_t end = block_end(ptr, rows, r, &by_wave), entries = ptr[end] - ptr[r];
    const int32_t parts = end - r > 1 ? (by_wave ? GPK_ROWS_BY_WAVE : 0)
                                      : entries > kEntryBudget ? (entries - 1) / kEntryBudget + 1 : 1;
    for (int32_t k = 0; k < (parts > 0 ? parts : 1); ++k, ++nb)
      if (out) out[nb] = gpk_row_block{r, ptr[r] + k * kEntryBudget, k, parts};
    r = end;
  }
  if (out) out[nb] = gpk_row_block{rows, rows > 0 ? ptr[rows] : 0, 0, 0};
  return nb;
}

hipError_t gpk_pdhg_iterations(gpk_rows A, gpk_rows AT, const double* c, const double* l, const double* u,
                               const double* AL, const double* AU, double* x, double* xbar, double* x_acc, double* y,
                               double* y_acc, const double* x0, const double* y0, const double* step,
                               int32_t halpern, int32_t iterations, hipStream_t s) {
  for (int32_t k = 0; k < iterations; ++k) {
    hipError_t e;
    if (halpern) {
      e = launch_rows(AT, OpPrimal<true>{y, c, l, u, step, x, xbar, x_acc, x0, k}, nullptr, s);
      if (e == hipSuccess) e = launch_rows(A, OpDual<true>{xbar, AL, AU, step, y, y_acc, y0, k}, nullptr, s);
    } else {
      e = launch_rows(AT, OpPrimal<false>{y, c, l, u, step, x, xbar, x_acc, x0, k}, nullptr, s);
      if (e == hipSuccess) e = launch_rows(A, OpDual<false>{xbar, AL, AU, step, y, y_acc, y0, k}, nullptr, s);
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t gpk_pdhg_axpby(double a, const double* x, double b, const double* y, double* out, int32_t n,
                          hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pdhg_axpby, dim3(grid_for(n)), dim3(kBlock), 0, s, a, x, b, y, out, n);
  return hipGetLastError();
}

hipError_t gpk_pdhg_mul(const double* x, const double* d, double* out, int32_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pdhg_mul, dim3(grid_for(n)), dim3(kBlock), 0, s, x, d, out, n);
  return hipGetLastError();
}

hipError_t gpk_pdhg_spmv(gpk_rows M, const double* x, const double* sumsq, double* y, hipStream_t s) {
  return launch_rows(M, OpSpmv{x, sumsq, y}, nullptr, s);
}

hipError_t gpk_pdhg_spmv_sq(gpk_rows M, const double* x, double* y, double* partial, double* out, hipStream_t s) {
  const hipError_t e = launch_rows(M, OpSpmvSq{x, y}, partial, s);
  if (e != hipSuccess) return e;
  return launch_reduce(partial, M.blocks > 0 ? M.blocks : 0, out, s);
}

hipError_t gpk_pdhg_ruiz(gpk_rows M, double* d, hipStream_t s) { return launch_rows(M, OpRuiz{d}, nullptr, s); }

hipError_t gpk_pdhg_scale_csr(gpk_rows M, const double* drow, const double* dcol, double* out, hipStream_t s) {
  if (M.blocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_rows_scale, dim3(static_cast<unsigned>(M.blocks)), dim3(kBlock), 0, s, M.M.ptr, M.M.idx, M.M.val,
                     M.blk, drow, dcol, out);
  return hipGetLastError();
}

hipError_t gpk_pdhg_scale_vec(const double* v, const double* d, double* out, int32_t n, int32_t mul, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pdhg_scale_vec, dim3(grid_for(n)), dim3(kBlock), 0, s, v, d, out, n, mul);
  return hipGetLastError();
}

int32_t gpk_pdhg_partials(int32_t blocks) { return (blocks > 0 ? blocks : 1) * kPartials; }

hipError_t gpk_pdhg_row_terms(gpk_rows A, const double* AL, const double* AU, const double* x, const double* y,
                              double* partial, double* out, hipStream_t s) {
  const hipError_t e = launch_rows(A, OpRowTerms{x, AL, AU, y}, partial, s);
  if (e != hipSuccess) return e;
  return launch_reduce(partial, A.blocks > 0 ? A.blocks : 0, out, s);
}

hipError_t gpk_pdhg_col_terms(gpk_rows AT, const double* c, const double* l, const double* u, const double* x,
                              const double* y, double* z, double* partial, double* out, hipStream_t s) {
  const hipError_t e = launch_rows(AT, OpColTerms{y, c, l, u, x, z}, partial, s);
  if (e != hipSuccess) return e;
  return launch_reduce(partial, AT.blocks > 0 ? AT.blocks : 0, out, s);
}

hipError_t gpk_pdhg_sq_terms(const double* a, const double* b, int32_t n, double* partial, double* out,
                             hipStream_t s) {
  const unsigned blocks = grid_for(n);
  hipLaunchKernelGGL(k_pdhg_sq_terms, dim3(blocks), dim3(kBlock), 0, s, a, b, n, partial);
  return launch_reduce(partial, static_cast<int32_t>(blocks), out, s);
}

hipError_t gpk_pdhg_seed(double* p, int32_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pdhg_seed, dim3(grid_for(n)), dim3(kBlock), 0, s, p, n);
  return hipGetLastError();
}

hipError_t gpk_pdhg_unscale_x(const double* xs, const double* d, const double* l, const double* u, double* out,
                              int32_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pdhg_unscale_x, dim3(grid_for(n)), dim3(kBlock), 0, s, xs, d, l, u, out, n);
  return hipGetLastError();
}

hipError_t gpk_pdhg_project_zero(const double* l, const double* u, double* x, int32_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_pdhg_project_zero, dim3(grid_for(n)), dim3(kBlock), 0, s, l, u, x, n);
  return hipGetLastError();
}

}  // extern "C"
