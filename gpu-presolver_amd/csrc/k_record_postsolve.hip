// Record maintenance (tape index globalization) and postsolve kernels: scatter of the reduced
// solution, fixed-value restore, reverse tape replay and the column-dual
// projection.
#include <hip/hip_runtime.h>

#include <climits>
#include <cmath>
#include <cstdint>

#include "gp_device.hpp"
#include "gp_kernels.h"
#include "gp_record_kernels.h"

using namespace gpdev;

namespace {

// ------------------------------------------------------------ record ----
// kind: 1 = row index, 2 = column index, 0 = not an index.  Out-of-range
// values are left unchanged (gpu_presolve.cu:1347-1361).
__global__ void k_map_tape_indices(int32_t count, int32_t* idx, const uint8_t* kind, const int32_t* row_red2org,
                                   int32_t m, const int32_t* col_red2org, int32_t n) {
  const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= count) return;
  const int32_t v = idx[t];
  if (kind[t] == 1) {
    if (v >= 0 && v < m) idx[t] = row_red2org[v];
  } else if (kind[t] == 2) {
    if (v >= 0 && v < n) idx[t] = col_red2org[v];
  }
}

// --------------------------------------------------------- postsolve ----
__global__ void k_scatter(const double* src, const int32_t* red2org, int32_t n_red, double* dst) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_red) dst[red2org[i]] = src[i];
}

__global__ void k_mark(const int32_t* red2org, int32_t n_red, uint8_t* mask) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_red) mask[red2org[i]] = 1;
}

__global__ void k_restore_fixed(const int32_t* idx, const double* val, int32_t count, double* x) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) x[idx[i]] = val[i];
}

__device__ inline bool pfin(double x) { return x > -INFINITY && x < INFINITY; }
__device__ inline bool at_lower(double x, double l, double tol) { return pfin(l) && x <= l + tol; }
__device__ inline bool at_upper(double x, double u, double tol) { return pfin(u) && x >= u - tol; }
__device__ inline double clamp_inf(double x, double lo, double hi) {
  double y = x;
  if (pfin(lo)) y = fmax(y, lo);
  if (pfin(hi)) y = fmin(y, hi);
  return y;
}

// gpu_postsolve.cu:189-210
__device__ double merged_source_value(double lo, double hi, double tol) {
  if (isfinite(lo) && isfinite(hi)) return 0.5 * (lo + hi);
  if (isfinite(lo)) {
    if (0.0 > lo + tol) return 0.0;
    return lo + fmax(1.0, fabs(lo) * fmax(tol, 1.0e-12));
  }
  if (isfinite(hi)) {
    if (0.0 < hi - tol) return 0.0;
    return hi - fmax(1.0, fabs(hi) * fmax(tol, 1.0e-12));
  }
  return 0.0;
}

// gpu_postsolve.cu:240-282
__device__ void recover_dup_col(double y, double z_to, double r, double sl, double su, double tl, double tu,
                                double tol, double* x_from, double* x_to) {
  double lo = sl, hi = su;
  if (isfinite(tu)) { const double b = (y - tu) / r; if (r > 0.0) lo = fmax(lo, b); else hi = fmin(hi, b); }
  if (isfinite(tl)) { const double b = (y - tl) / r; if (r > 0.0) hi = fmin(hi, b); else lo = fmax(lo, b); }
  double lower = -INFINITY, upper = INFINITY;
  if (r > 0.0) {
    if (isfinite(tl) && isfinite(sl)) lower = tl + r * sl;
    if (isfinite(tu) && isfinite(su)) upper = tu + r * su;
  } else {
    if (isfinite(tl) && isfinite(su)) lower = tl + r * su;
    if (isfinite(tu) && isfinite(sl)) upper = tu + r * sl;
  }
  if (z_to > tol && isfinite(lower) && fabs(y - lower) <= tol) *x_from = r > 0.0 ? sl : su;
  else if (z_to < -tol && isfinite(upper) && fabs(y - upper) <= tol) *x_from = r > 0.0 ? su : sl;
  else *x_from = merged_source_value(lo, hi, tol);
  *x_to = y - r * (*x_from);
}

enum : uint8_t { ST_ZERO = 0, ST_NONNEG = 1, ST_NONPOS = 2, ST_FREE = 3 };
__device__ uint8_t row_state(double act, double lo, double hi, double tol) {
  const bool al = pfin(lo) && act <= lo + tol;
  const bool au = pfin(hi) && act >= hi - tol;
  if (al && au) return ST_FREE;
  if (al) return ST_NONNEG;
  if (au) return ST_NONPOS;
  return ST_ZERO;
}
__device__ void state_interval(uint8_t s, double* lo, double* hi) {
  if (s == ST_FREE) { *lo = -INFINITY; *hi = INFINITY; }
  else if (s == ST_NONNEG) { *lo = 0.0; *hi = INFINITY; }
  else if (s == ST_NONPOS) { *lo = -INFINITY; *hi = 0.0; }
  else { *lo = 0.0; *hi = 0.0; }
}
__device__ void deleted_dual_interval(double yp, double r, uint8_t ks, double* lo, double* hi) {
  const double piv = r * yp;
  if (ks == ST_FREE) { *lo = -INFINITY; *hi = INFINITY; }
  else if (ks == ST_ZERO) { *lo = piv; *hi = piv; }
  else if (ks == ST_NONNEG) { if (r > 0.0) { *lo = -INFINITY; *hi = piv; } else { *lo = piv; *hi = INFINITY; } }
  else { if (r > 0.0) { *lo = piv; *hi = INFINITY; } else { *lo = -INFINITY; *hi = piv; } }
}
// gpu_postsolve.cu:409-469
__device__ bool doc_dual_split(double yp, double r, double kal, double kau, double dsl, double dsu, double tol,
                               double* op, double* od) {
  if (fabs(yp) <= tol) { *op = 0.0; *od = 0.0; return true; }
  const double bl = fmax(kal, dsl), bu = fmin(kau, dsu);
  if (!(bl <= bu + tol)) { *op = yp; *od = 0.0; return false; }
  const bool lt = bl > kal + tol, ut = bu < kau - tol;
  if (lt && ut) { *op = yp; *od = 0.0; return false; }
  if (!lt && !ut) { *op = yp; *od = 0.0; return true; }
  if (yp > 0.0) {
    if (lt) { *op = 0.0; *od = r * yp; } else { *op = yp; *od = 0.0; }
    return true;
  }
  if (lt) { *op = yp; *od = 0.0; } else { *op = 0.0; *od = r * yp; }
  return true;
}
// gpu_postsolve.cu:471-515
__device__ void dbl_recover_z(double xk, double zk_hat, double al, double okl, double oku, double nkl, double nku,
                              double ls, double us, double tol, double* zk, double* ze) {
  if (fabs(al) <= tol) { *zk = zk_hat; *ze = 0.0; return; }
  const bool atl = pfin(nkl) && xk <= nkl + tol;
  const bool atu = pfin(nku) && xk >= nku - tol;
  if (!atl && !atu) { *zk = 0.0; *ze = 0.0; return; }
  double src = atl ? ls : us;
  if (src == 0.0) {
    if (atl) src = (pfin(okl) && fabs(nkl - okl) <= tol) ? 1.0 : 2.0;
    else src = (pfin(oku) && fabs(nku - oku) <= tol) ? 1.0 : 2.0;
  }
  if (src == 2.0) { *zk = 0.0; *ze = zk_hat / al; }
  else { *zk = zk_hat; *ze = 0.0; }
}

// A record goes one of two ways (gpk_record_walks_line), at every turn the same.
//
// A record that walks a line of entries (a row's or column's dual, a
// substituted column's primal) is worked on by sixteen lanes (a DPP row): its
// index words, its values and the entries of its line are one to a lane.  A
// level's time is that of the instructions of one wave and of its round trips
// to memory: with a lane per record the entries of a line are that many loads,
// branches and divides one after the other (9.3 us a level even with all of them
// loaded ahead), so they are side by side instead.
//
// Any other record has one lane: a wave takes 64 of them where sixteen lanes
// each would take 4 (a level of 256 such records 0.8 us, 6.3 with sixteen).
constexpr int kRecLanes = 16;
constexpr int kRecChunks = 2;  // chunks of 16 entries of a line loaded ahead

// Lane k's value of the 16 lanes, k a constant.
template <int k>
__device__ __forceinline__ int32_t row_lane(int32_t v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x150 + k, 0xf, 0xf, true);  // row_newbcast
}
template <int k>
__device__ __forceinline__ double row_lane(double v) {
  const long long b = __double_as_longlong(v);
  return __hiloint2double(row_lane<k>(static_cast<int32_t>(b >> 32)), row_lane<k>(static_cast<int32_t>(b)));
}
// s + (lane 0's term) + (lane 1's term) + ..., added one after the other.  A
// lane without a term holds -0, which leaves any sum as it is.
__device__ __forceinline__ double row_add(double s, double t) {
  s += row_lane<0>(t);
  s += row_lane<1>(t);
  s += row_lane<2>(t);
  s += row_lane<3>(t);
  s += row_lane<4>(t);
  s += row_lane<5>(t);
  s += row_lane<6>(t);
  s += row_lane<7>(t);
  s += row_lane<8>(t);
  s += row_lane<9>(t);
  s += row_lane<10>(t);
  s += row_lane<11>(t);
  s += row_lane<12>(t);
  s += row_lane<13>(t);
  s += row_lane<14>(t);
  s += row_lane<15>(t);
  return s;
}

// s += sum over q in [0, count) with idx[q] != skip of sign * val[q] * vec[idx[q]]
// (sign 1 or -1), accumulated in q order exactly as the plain loop would (every
// product rounded, then added or subtracted one at a time).
__device__ inline double dot_in_order(double s, double sign, const int32_t* __restrict__ idx,
                                      const double* __restrict__ val, const double* vec, int32_t count, int32_t skip) {
  const int t = static_cast<int>(threadIdx.x & (kRecLanes - 1));
#pragma unroll 1
  for (int32_t q = 0; q < count; q += 2 * kRecLanes) {
    double p[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int32_t e = q + c * kRecLanes + t;
      const int32_t j = e < count ? idx[e] : skip;
      const double a = e < count ? val[e] : 0.0;
      p[c] = e < count && j != skip ? sign * (a * vec[j]) : -0.0;
    }
    s = row_add(s, p[0]);
    if (q + kRecLanes < count) s = row_add(s, p[1]);
  }
  return s;
}

// What a record's turn needs of the tape and of the original model, none of
// which the replay writes: it can be loaded before the turn comes, and then
// only the loads of x, y, z and zret are left to it.  Four steps, each one
// memory round trip behind the one before: where the record's indices and
// values sit; its first 16 index words (-1 past its end); the line of entries
// it walks; its first 16 values (0 past its end) and the line's first entries.
struct RecHead {
  int32_t type, i0, i1, v0, v1;  // type -1: an empty slot
};
struct RecLine {
  int32_t qi, qv, n;  // the line's first index and first value, its length
};
struct RecEntries {
  double v;  // the lane's value
  int32_t j[kRecChunks];
  double a[kRecChunks];
};

__device__ inline RecHead load_head(const gp_tape_dev& T, int32_t k) {
  if (k < 0) return RecHead{-1, 0, -1, 0, -1};
  return RecHead{T.types[k], T.index_starts[k], T.index_starts[k + 1] - 1, T.value_starts[k],
                 T.value_starts[k + 1] - 1};
}
__device__ inline int32_t load_word(const gp_tape_dev& T, const RecHead& h, int t) {
  return h.i0 + t <= h.i1 ? T.indices[h.i0 + t] : -1;
}

__device__ inline bool has_payload(const RecHead& h) { return h.i1 >= h.i0 + 3 && h.v1 >= h.v0 + 11; }
// Where the line sits: in the tape, in the columns or in the rows of the model.
enum : int { LINE_TAPE, LINE_COL, LINE_ROW };
__device__ inline int line_kind(const RecHead& h) {
  if (h.type == 12 || h.type == 4) return LINE_ROW;
  return h.type == 5 || (h.type == 13 && !has_payload(h)) ? LINE_COL : LINE_TAPE;
}
// The lines of types 0, 4, 5 and 13 are walked for y, and a line's place is
// checked by the host only where there is a y.
__device__ inline RecLine load_line(const gp_orig_dev& O, const RecHead& h, int32_t word, bool has_y, bool dual) {
  const int32_t type = h.type;
  if (!dual && type == 2) return RecLine{h.i0 + 3, h.v0 + 6, row_lane<2>(word)};
  if (dual && type == 0 && has_y) return RecLine{h.i0 + 1, h.v0 + 2, h.i1 - h.i0};
  if (dual && O.present != 0 && (has_y || type == 12)) {
    const int kind = line_kind(h);
    if (type == 13 && kind == LINE_TAPE) return RecLine{h.i0 + 4, h.v0 + 12, row_lane<3>(word)};
    const int32_t line = type == 13 || type == 4 ? row_lane<0>(word) : row_lane<1>(word);
    if (kind != LINE_TAPE && line >= 0) {
      const int32_t* ptr = kind == LINE_ROW ? O.a_ptr : O.at_ptr;
      const int32_t b = ptr[line];
      return RecLine{b, b, ptr[line + 1] - b};
    }
  }
  return RecLine{0, 0, 0};
}
__device__ inline const int32_t* line_idx(const gp_tape_dev& T, const gp_orig_dev& O, int kind) {
  return kind == LINE_TAPE ? T.indices : kind == LINE_COL ? O.at_idx : O.a_idx;
}
__device__ inline const double* line_val(const gp_tape_dev& T, const gp_orig_dev& O, int kind) {
  return kind == LINE_TAPE ? T.vals : kind == LINE_COL ? O.at_val : O.a_val;
}
__device__ inline RecEntries load_entries(const gp_tape_dev& T, const gp_orig_dev& O, const RecHead& h,
                                          const RecLine& ln, int t) {
  RecEntries r;
  r.v = h.v0 + t <= h.v1 ? T.vals[h.v0 + t] : 0.0;
  const int kind = line_kind(h);
  const int32_t* idx = line_idx(T, O, kind);
  const double* val = line_val(T, O, kind);
#pragma unroll
  for (int c = 0; c < kRecChunks; ++c) {
    const int32_t e = c * kRecLanes + t;
    r.j[c] = e < ln.n ? idx[ln.qi + e] : -1;
    r.a[c] = e < ln.n ? val[ln.qv + e] : 0.0;
  }
  return r;
}

// The column and the row whose values a record reads besides its line's.
__device__ inline int32_t column_read(int32_t type, int32_t w0, int32_t w1) {
  return type == 13 || type == 5 ? w1 : type == 12 ? w0 : -1;
}
__device__ inline int32_t row_read(int32_t type, int32_t w0, int32_t w1) {
  return type == 12 ? w1 : type == 4 ? w0 : -1;
}

// A record's packet: all of its operands that are not values, in the order of a
// schedule, so that a turn is three chained loads (packet, line and values, x and
// y and z) instead of six.  A record without a line has the first eight words.
enum : int { PK_TYPE = 0, PK_I0 = 1, PK_I1 = 2, PK_V0 = 3, PK_V1 = 4, PK_W0 = 5, PK_QI = 9, PK_QV = 10, PK_N = 11 };
static_assert(GPK_PACKET_WORDS == kRecLanes, "a word to a lane");
static_assert(GPK_SIMPLE_WORDS == 8 && PK_W0 + 3 == GPK_SIMPLE_WORDS, "two loads of sixteen bytes");
__device__ __forceinline__ RecHead packet_head(int32_t p) {
  return RecHead{row_lane<PK_TYPE>(p), row_lane<PK_I0>(p), row_lane<PK_I1>(p), row_lane<PK_V0>(p),
                 row_lane<PK_V1>(p)};
}
__device__ __forceinline__ RecLine packet_line(int32_t p) {
  return RecLine{row_lane<PK_QI>(p), row_lane<PK_QV>(p), row_lane<PK_N>(p)};
}
// The word of lane t of an empty slot's packet.
__device__ __forceinline__ int32_t packet_none(int t) {
  return t == PK_TYPE || t == PK_I1 || t == PK_V1 ? -1 : 0;
}

// The record's first index words.
struct RecVars {
  int32_t w0, w1, w2;
};

// A record without a line, a lane to itself.
struct SimpleRec {
  int32_t type, i0, i1, v0, v1, w0, w1, w2;  // type -1: none
};
// Its values [0, 6) and 9 (0 past its end).
struct SimpleVals {
  double v[6], v9;
};
// What its turn reads.
struct SimpleReads {
  double x, z, y;
};
__device__ __forceinline__ SimpleRec simple_none() { return SimpleRec{-1, 0, -1, 0, -1, -1, -1, -1}; }
__device__ __forceinline__ SimpleRec simple_packet(const int32_t* __restrict__ packets, int64_t slot) {
  const int4* p = reinterpret_cast<const int4*>(packets) + slot * (GPK_SIMPLE_WORDS / 4);
  const int4 a = p[0], b = p[1];
  return SimpleRec{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
}
__device__ __forceinline__ SimpleVals simple_values(const gp_tape_dev& T, const SimpleRec& h) {
  SimpleVals r;
#pragma unroll
  for (int q = 0; q < 6; ++q) r.v[q] = h.v0 + q <= h.v1 ? T.vals[h.v0 + q] : 0.0;
  r.v9 = h.v0 + 9 <= h.v1 ? T.vals[h.v0 + 9] : 0.0;
  return r;
}
template <bool kDual>
__device__ __forceinline__ SimpleReads simple_reads(const SimpleRec& h, const double* x, const double* y,
                                                    const double* z) {
  const int32_t col = h.type == 3 || h.type == 13 ? h.w1 : -1;
  const int32_t row = h.type == 2 ? h.w1 : h.type == 10 ? h.w0 : -1;
  SimpleReads v;
  v.x = !kDual && col >= 0 ? x[col] : 0.0;
  v.z = col >= 0 && z ? z[col] : 0.0;
  v.y = kDual && row >= 0 && y ? y[row] : 0.0;
  return v;
}

template <bool kDual>
__device__ __forceinline__ void replay_simple(const gp_tape_dev& T, double* x, double* y, double* z, uint8_t* zret,
                                              const SimpleRec& h, const SimpleVals& r, const SimpleReads& in,
                                              double tol) {
  const int32_t type = h.type, w0 = h.w0, w1 = h.w1;
  if (type < 0) return;
  constexpr bool primal = !kDual, dual = kDual;
  const int32_t* I = T.indices;
  const double* V = T.vals;
  const int32_t i0 = h.i0, v0 = h.v0;
  const double xc = in.x, zc = in.z, yr = in.y;
  if (type == 3) {  // DuplicateColumn
    if (primal) {
      double xf = 0.0, xt = xc;
      recover_dup_col(xc, zc, r.v[0], r.v[1], r.v[2], r.v[3], r.v[4], tol, &xf, &xt);
      x[w0] = xf;
      x[w1] = xt;
    }
    if (dual && z) { z[w0] = r.v[0] * zc; if (zret) zret[w0] = 1; }
  } else if (type == 13) {  // DoubletonEquation; dual: without an original model or y
    const double ecoef = r.v[0], kcoef = r.v[1], rhs = r.v[2], eobj = r.v9;
    const double al = -kcoef / ecoef, be = rhs / ecoef;
    if (primal) x[w0] = be + al * xc;
    if (dual) {
      if (z) { z[w0] = 0.0; if (zret) zret[w0] = 1; }
      if (y && h.w2 >= 0) y[h.w2] = eobj / ecoef;
    }
  } else if (dual && type == 2) {  // SubCol
    const double piv = r.v[0], eobj = r.v[4];
    const bool row_deleted = r.v[5] != 0.0;
    const double y_new = row_deleted ? eobj / piv : yr + eobj / piv;
    if (y && w1 >= 0) y[w1] = y_new;
    if (z) {
      z[w0] = (row_deleted || !y) ? 0.0 : eobj - piv * (w1 >= 0 ? y_new : 0.0);
      if (zret) zret[w0] = 1;
    }
  } else if (type == 0) {  // FixedCol; dual: without rows or y
    if (primal) x[w0] = r.v[0];
    if (dual && z) { z[w0] = r.v[1]; if (zret) zret[w0] = 1; }
  } else if (type == 1) {  // FixedColInf
    const bool pos_inf = w0 > 0;
    const int32_t col = w1;
    if (primal) {
      const int32_t nrows = static_cast<int32_t>(llround(r.v[0]));
      double ext = r.v[1];
      int32_t ip = i0 + 2, vp = v0 + 2;
      for (int32_t q = 0; q < nrows; ++q) {
        const int32_t len = I[ip];
        double side = V[vp], coef = 0.0;
        for (int32_t t = 0; t < len; ++t) {
          const int32_t rc = I[ip + 1 + t];
          const double rv = V[vp + 1 + t];
          if (rc == col) coef = rv; else side -= rv * x[rc];
        }
        const double cand = side / coef;
        ext = pos_inf ? fmax(ext, cand) : fmin(ext, cand);
        ip += len + 1;
        vp += len + 1;
      }
      x[col] = ext;
    }
    if (dual && z) { z[col] = 0.0; if (zret) zret[col] = 1; }
  } else if (type == 14) {  // FmeCol
    const int32_t K = w0, ec = w1;
    if (primal) {
      const int32_t L = static_cast<int32_t>(llround(r.v[0]));
      int32_t cc = i0 + 3 + K, vp = v0 + 1;
      double lo = -INFINITY, hi = INFINITY;
      bool hl = false, hh = false;
      for (int32_t q = 0; q < L; ++q) {
        const double orient = V[vp];
        const int32_t len = static_cast<int32_t>(llround(V[vp + 1]));
        double cand = V[vp + 2];
        for (int32_t t = 0; t < len; ++t) cand += V[vp + 3 + t] * x[I[cc++]];
        if (orient > 0.0) { lo = fmax(lo, cand); hl = true; }
        else { hi = fmin(hi, cand); hh = true; }
        vp += 3 + len;
      }
      x[ec] = hl ? lo : (hh ? hi : 0.0);
    }
    if (dual && z) { z[ec] = 0.0; if (zret) zret[ec] = 1; }
    if (dual && y) for (int32_t t = 0; t < K; ++t) y[I[i0 + 2 + t]] = 0.0;
  } else if (dual && type == 10) {  // EqToIneq
    if (y) y[w0] = yr + r.v[0];
  } else if (dual && type == 4 && w1 >= 0 && h.v1 >= v0 + 4) {  // DuplicateRow without an original model
    const double q = r.v[0], kal = r.v[1], kau = r.v[2];
    if (fabs(q) <= tol || !y) return;
    const double a = r.v[3] * q, b = r.v[4] * q;
    const double dsl = q >= 0.0 ? a : b, dsu = q >= 0.0 ? b : a;
    if (dsl <= kal + tol && kau <= dsu + tol) y[w1] = 0.0;
  }
}

// A record with a line of the reverse replay (_kernel_replay_postsolve_tape,
// gpu_postsolve.cu:605-1046); all sixteen lanes come with the same record.
// kDual picks the pass.  All loads of x, y, z and zret that the record's type
// needs go out together at the top: a wave waits for one round trip, for two
// where a decision comes before a row is read.
template <bool kDual>
__device__ __forceinline__ void replay_line(const gp_tape_dev& T, const gp_orig_dev& O, double* x, double* y, double* z,
                                           uint8_t* zret, const RecHead& h, const RecVars& rv, const RecLine& ln,
                                           RecEntries r, double tol) {
  const bool has_orig = O.present != 0;
  const int32_t type = h.type;
  if (type < 0) return;
  constexpr bool primal = !kDual, dual = kDual;
  const int t = static_cast<int>(threadIdx.x & (kRecLanes - 1));
  const bool first = t == 0;  // the lane that stores what the record has one of
  const int32_t v0 = h.v0;
  // The record's first index words and values.
  const int32_t w0 = rv.w0, w1 = rv.w1, w2 = rv.w2;
  const double W0 = row_lane<0>(r.v), W1 = row_lane<1>(r.v), W2 = row_lane<2>(r.v), W3 = row_lane<3>(r.v),
               W4 = row_lane<4>(r.v), W5 = row_lane<5>(r.v);

  const int32_t col_in = column_read(type, w0, w1), row_in = row_read(type, w0, w1);
  const double xc = col_in >= 0 ? x[col_in] : 0.0;
  const double zc = col_in >= 0 && z ? z[col_in] : 0.0;
  const bool col_set = type == 12 && dual && zret ? zret[col_in] != 0 : true;
  const double yr = dual && row_in >= 0 && y ? y[row_in] : 0.0;
  const int32_t cost = type == 13 ? w0 : type == 5 ? w1 : -1;
  const double cc = dual && has_orig && cost >= 0 ? O.c[cost] : 0.0;

  // A bound change's row: its z and whether each is set.
  bool on[kRecChunks];
  double zk[kRecChunks];
  if (dual && type == 12) {
#pragma unroll
    for (int c = 0; c < kRecChunks; ++c) {
      const bool other = r.j[c] >= 0 && r.j[c] != w0;
      zk[c] = other ? z[r.j[c]] : 0.0;
      on[c] = other && (!zret || zret[r.j[c]]);
    }
  }

  // The sum over the line with x (types 2 and 4) or y, in order.
  const int kind = line_kind(h);
  double sum = type == 0 ? W1 : type == 5 ? cc : 0.0;
  if (ln.n > 0 && type != 12) {
    const double* vec = type == 2 || type == 4 ? x : y;
    const double sign = type == 0 || type == 5 ? -1.0 : 1.0;
    const int32_t skip = type == 5 ? w0 : type == 13 && kind == LINE_COL ? w2 : -1;
    double p[kRecChunks];
#pragma unroll
    for (int c = 0; c < kRecChunks; ++c)
      p[c] = r.j[c] >= 0 && r.j[c] != skip ? sign * (r.a[c] * vec[r.j[c]]) : -0.0;
#pragma unroll
    for (int c = 0; c < kRecChunks; ++c)
      if (ln.n > c * kRecLanes) sum = row_add(sum, p[c]);
    constexpr int kHave = kRecChunks * kRecLanes;
    if (ln.n > kHave)
      sum = dot_in_order(sum, sign, line_idx(T, O, kind) + ln.qi + kHave, line_val(T, O, kind) + ln.qv + kHave, vec,
                         ln.n - kHave, skip);
  }

  if (dual && type == 13) {  // DoubletonEquation
    const int32_t ec = w0, kc = w1, row = w2;
    const double ecoef = W0, al = -W1 / ecoef, eobj = row_lane<9>(r.v);
    double zk = 0.0, ze = 0.0;
    dbl_recover_z(xc, zc, al, W5, row_lane<6>(r.v), row_lane<7>(r.v), row_lane<8>(r.v), row_lane<10>(r.v),
                  row_lane<11>(r.v), tol, &zk, &ze);
    const double yrow = ((kind == LINE_TAPE ? eobj : cc) - sum - ze) / ecoef;
    if (first) {
      y[row] = yrow;
      z[kc] = zk;
      z[ec] = ze;
      if (zret) { zret[kc] = 1; zret[ec] = 1; }
    }
  } else if (primal && type == 2) {  // SubCol
    if (first) x[w0] = (W1 - sum) / W0;
  } else if (dual && type == 0) {  // FixedCol
    if (z && first) {
      z[w0] = sum;
      if (zret) zret[w0] = 1;
    }
  } else if (dual && type == 4 && w1 >= 0 && h.v1 >= v0 + 4) {  // DuplicateRow
    const int32_t kr = w0, dr = w1;
    const double q = W0, kal = W1, kau = W2, dal = W3, dau = W4;
    if (fabs(q) <= tol || !y) return;
    const double a = dal * q, b = dau * q;
    const double dsl = q >= 0.0 ? a : b, dsu = q >= 0.0 ? b : a;
    if (dsl <= kal + tol && kau <= dsu + tol) {
      if (first) y[dr] = 0.0;
      return;
    }
    if (has_orig) {
      const int32_t db = O.a_ptr[dr], de = O.a_ptr[dr + 1];
      const double ap = sum;
      const double ad = dot_in_order(0.0, 1.0, O.a_idx + db, O.a_val + db, x, de - db, -1);
      const uint8_t ks = row_state(ap, kal, kau, tol), ds = row_state(ad, dal, dau, tol);
      double ydl, ydh, ypl, yph;
      state_interval(ds, &ydl, &ydh);
      deleted_dual_interval(yr, q, ks, &ypl, &yph);
      const double sl = fmax(ydl, ypl), sh = fmin(ydh, yph);
      if (sl <= sh + tol) {
        const double ydn = clamp_inf(0.0, sl, sh);
        if (first) { y[kr] = yr - ydn / q; y[dr] = ydn; }
        return;
      }
      double ypd = yr, ydd = 0.0;
      if (doc_dual_split(yr, q, kal, kau, dsl, dsu, tol, &ypd, &ydd) && first) { y[kr] = ypd; y[dr] = ydd; }
    }
  } else if (dual && type == 5 && has_orig && w1 >= 0 && h.v1 >= v0 + 2) {  // DeletedRow
    const int32_t row = w0, col = w1;
    const double oal = W0, oau = W1, aij = W2;
    if (fabs(aij) <= tol) return;
    const double gamma = sum;
    const double xj = xc, zbar = zc;
    const double act = aij * xj;
    const bool ral = pfin(oal) && act <= oal + tol;
    const bool rau = pfin(oau) && act >= oau - tol;
    double izl = -INFINITY, izh = INFINITY;
    if (!(ral && rau)) {
      if (ral) { if (aij > 0.0) izh = gamma; else izl = gamma; }
      else if (rau) { if (aij > 0.0) izl = gamma; else izh = gamma; }
      else { izl = gamma; izh = gamma; }
    }
    const bool atl = at_lower(xj, O.l[col], tol), atu = at_upper(xj, O.u[col], tol);
    double zl = izl, zh = izh;
    if (!atl && !atu) {
      if ((pfin(izl) && izl > tol) || (pfin(izh) && izh < -tol)) { zl = gamma; zh = gamma; }
      else { zl = 0.0; zh = 0.0; }
    } else if (atl && !atu) {
      zl = fmax(zl, 0.0);
    } else if (!atl && atu) {
      zh = fmin(zh, 0.0);
    }
    if (pfin(zl) && pfin(zh) && zl > zh + tol) return;
    const double zn = clamp_inf(zbar, zl, zh);
    if (!first) return;
    z[col] = zn;
    if (y) y[row] = (gamma - zn) / aij;
    if (zret) zret[col] = 1;
  } else if (dual && type == 12 && has_orig && w1 >= 0) {  // BoundChangeTheRow
    const int32_t col = w0, row = w1;
    const double ol = W0, ou = W1, nl = W2, nu = W3;
    const double xj = xc, zj = zc;
    if (!col_set) return;
    const bool lc = nl > ol + tol, uc = nu < ou - tol;
    if (lc == uc) return;
    const double implied = lc ? nl : nu;
    const double other = lc ? ou : ol;
    const bool other_is_lower = !lc;
    if (pfin(other) && fabs(xj - other) <= tol) {
      const bool ok = other_is_lower ? (zj >= -tol) : (zj <= tol);
      if (ok) return;
    }
    if (fabs(xj - implied) > tol) return;
    if (ln.n <= 0) return;  // an empty row holds no a_ij
    // a_ij is the row's first entry in the column.
    double aij = 0.0;
    const int g0 = lane_id() & ~(kRecLanes - 1);
    for (int32_t q = 0; q < ln.n; q += kRecLanes) {
      const int32_t e = ln.qi + min(q + t, ln.n - 1);
      const int32_t j = q == 0 ? r.j[0] : q == kRecLanes ? r.j[1] : O.a_idx[e];
      const uint32_t hit = static_cast<uint32_t>(__ballot(j == col) >> g0) & 0xffffu;
      if (hit == 0) continue;
      const double a = q == 0 ? r.a[0] : q == kRecLanes ? r.a[1] : O.a_val[e];
      aij = __shfl(a, __ffs(hit) - 1, kRecLanes);
      break;
    }
    if (fabs(aij) <= tol) return;
    if (y && first) y[row] = yr + zj / aij;
    // The row's columns are distinct, so its updates are independent: the
    // results are those of the entry-by-entry loop.
    for (int32_t q = 0;;) {
#pragma unroll
      for (int c = 0; c < kRecChunks; ++c)
        if (on[c]) z[r.j[c]] = zk[c] - (r.a[c] / aij) * zj;
      q += kRecChunks * kRecLanes;
      if (q >= ln.n) break;
#pragma unroll
      for (int c = 0; c < kRecChunks; ++c) {
        const int32_t e = q + c * kRecLanes + t;
        r.j[c] = e < ln.n ? O.a_idx[ln.qi + e] : -1;
        r.a[c] = e < ln.n ? O.a_val[ln.qi + e] : 0.0;
        const bool other = r.j[c] >= 0 && r.j[c] != col;
        zk[c] = other ? z[r.j[c]] : 0.0;
        on[c] = other && (!zret || zret[r.j[c]]);
      }
    }
    if (!first) return;
    z[col] = 0.0;
    if (zret) zret[col] = 1;
  }
}

// The packets of a plan's schedules, primal first: line slots from dual_line on
// are of the dual pass (the others' packets are the same in both).  Blocks: the records with a line, sixteen
// lanes each, then the others.
__global__ void __launch_bounds__(kBlock) k_pack_records(gp_tape_dev T, gp_orig_dev O, gpk_replay_slots s,
                                                         int32_t dual_line, int32_t has_y, int32_t line_blocks) {
  const int32_t block = static_cast<int32_t>(blockIdx.x);
  if (block >= line_blocks) {
    const int32_t i = (block - line_blocks) * kBlock + static_cast<int32_t>(threadIdx.x);
    if (i >= s.simple_slots) return;
    const RecHead h = load_head(T, s.simple_records[i]);
    int4* p = reinterpret_cast<int4*>(s.simple) + static_cast<int64_t>(i) * (GPK_SIMPLE_WORDS / 4);
    p[0] = make_int4(h.type, h.i0, h.i1, h.v0);
    p[1] = make_int4(h.v1, load_word(T, h, 0), load_word(T, h, 1), load_word(T, h, 2));
    return;
  }
  const int32_t i = block * (kBlock / kRecLanes) + static_cast<int32_t>(threadIdx.x) / kRecLanes;
  if (i >= s.line_slots) return;
  const int t = static_cast<int>(threadIdx.x & (kRecLanes - 1));
  const RecHead h = load_head(T, s.line_records[i]);
  const int32_t word = load_word(T, h, t);
  const RecLine ln = load_line(O, h, word, has_y != 0, i >= dual_line);
  const int32_t w = __shfl(word, t >= PK_W0 && t < PK_QI ? t - PK_W0 : 0, kRecLanes);
  const int32_t p = t == PK_TYPE ? h.type : t == PK_I0 ? h.i0 : t == PK_I1 ? h.i1 : t == PK_V0 ? h.v0
                    : t == PK_V1 ? h.v1 : t < PK_QI ? w : t == PK_QI ? ln.qi : t == PK_QV ? ln.qv
                    : t == PK_N ? ln.n : 0;
  s.line[static_cast<int64_t>(i) * GPK_PACKET_WORDS + t] = p;
}

// One level of a dependency-level schedule: its records touch disjoint
// variables.  Blocks: line records, sixteen lanes each, then the others, a lane
// each.  Three chains of loads and little else: 5.6 us for 1,000 to 30,000 line
// records (16 us with a lane per record, 6.5 with six chains).
template <bool kDual>
__global__ void __launch_bounds__(kBlock)
    k_replay_list(gp_tape_dev T, gp_orig_dev O, double* x, double* y, double* z, uint8_t* zret,
                  const int32_t* __restrict__ line, int32_t lines, const int32_t* __restrict__ simple, int32_t simples,
                  int32_t line_blocks, double tol) {
  const int32_t block = static_cast<int32_t>(blockIdx.x);
  if (block >= line_blocks) {
    const int32_t i = (block - line_blocks) * kBlock + static_cast<int32_t>(threadIdx.x);
    if (i >= simples) return;
    const SimpleRec h = simple_packet(simple, i);
    replay_simple<kDual>(T, x, y, z, zret, h, simple_values(T, h), simple_reads<kDual>(h, x, y, z), tol);
    return;
  }
  const int32_t i = block * (kBlock / kRecLanes) + static_cast<int32_t>(threadIdx.x) / kRecLanes;
  if (i >= lines) return;
  const int t = static_cast<int>(threadIdx.x & (kRecLanes - 1));
  const int32_t p = line[static_cast<int64_t>(i) * GPK_PACKET_WORDS + t];
  const RecHead h = packet_head(p);
  const RecLine ln = packet_line(p);
  const RecEntries r = load_entries(T, O, h, ln, t);
  const RecVars rv{row_lane<PK_W0>(p), row_lane<PK_W0 + 1>(p), row_lane<PK_W0 + 2>(p)};
  replay_line<kDual>(T, O, x, y, z, zret, h, rv, ln, r, tol);
}

constexpr int kLevelBlock = 64 * GPK_REPLAY_WAVES;
constexpr int kWaveLines = 64 / kRecLanes;
static_assert(GPK_WAVE_LINES == kWaveLines, "a wave's line records");

// The line records of a run of levels, by the workgroup's first waves: those of a
// level, then the barrier.  A wave has the packets of its records two levels
// ahead and their lines and values one level ahead on their way, so that a level
// waits only for its x, y, z and zret, and for its stores at the barrier.  Bound
// by that chain: 1,106 dual levels, most of about 31 records, take 2.7 ms (2.5 us
// each; 11.4 ms for 1,207 with a lane per record and each chain in its turn, 4.2
// with a record's six chains five levels ahead in place of packets).  Reading x,
// y, z and zret once a level ahead, to have them in the CU's cache, cost 0.4 ms
// more.  The levels' slots come by vector loads: a scalar one would be waited
// for together with the newest of its kind (2.28 us a level against 2.35).
template <bool kDual>
__device__ __forceinline__ void replay_level_lines(const gp_tape_dev& T, const gp_orig_dev& O, double* x, double* y,
                                                   double* z, uint8_t* zret, const int32_t* __restrict__ line,
                                                   const gpk_replay_level* __restrict__ levels, int32_t nlevels,
                                                   double tol) {
  const int32_t slot = static_cast<int32_t>(threadIdx.x) / kRecLanes;
  const int t = static_cast<int>(threadIdx.x & (kRecLanes - 1));
  int32_t zero = 0;
  asm("" : "+v"(zero));
  const auto level = [&](int32_t l) {
    return l < nlevels ? reinterpret_cast<const int2*>(levels)[2 * (l + zero)] : make_int2(0, 0);
  };
  const auto packet = [&](int2 d) {
    return slot < d.y ? line[(static_cast<int64_t>(d.x) + slot) * GPK_PACKET_WORDS + t] : packet_none(t);
  };
  int2 d2 = level(2);
  int32_t p0 = packet(level(0)), p1 = packet(level(1));
  RecEntries r0 = load_entries(T, O, packet_head(p0), packet_line(p0), t);
#pragma unroll 1
  for (int32_t l = 0; l < nlevels; ++l) {
    const int2 d3 = level(l + 3);
    const int32_t p2 = packet(d2);
    const RecEntries r1 = load_entries(T, O, packet_head(p1), packet_line(p1), t);
    const RecVars rv{row_lane<PK_W0>(p0), row_lane<PK_W0 + 1>(p0), row_lane<PK_W0 + 2>(p0)};
    replay_line<kDual>(T, O, x, y, z, zret, packet_head(p0), rv, packet_line(p0), r0, tol);
    __syncthreads();
    p0 = p1;
    p1 = p2;
    r0 = r1;
    d2 = d3;
  }
}

// The other records, by the waves from `first` on, in the same way.
template <bool kDual>
__device__ __forceinline__ void replay_level_simples(const gp_tape_dev& T, double* x, double* y, double* z,
                                                     uint8_t* zret, const int32_t* __restrict__ simple,
                                                     const gpk_replay_level* __restrict__ levels, int32_t nlevels,
                                                     int32_t first, double tol) {
  const int32_t slot = static_cast<int32_t>(threadIdx.x) - 64 * first;
  const auto level = [&](int32_t l) {
    return l < nlevels ? reinterpret_cast<const int2*>(levels)[2 * l + 1] : make_int2(0, 0);
  };
  const auto packet = [&](int2 d) {
    return slot < d.y ? simple_packet(simple, static_cast<int64_t>(d.x) + slot) : simple_none();
  };
  int2 d2 = level(2);
  SimpleRec h0 = packet(level(0)), h1 = packet(level(1));
  SimpleVals v0 = simple_values(T, h0);
#pragma unroll 1
  for (int32_t l = 0; l < nlevels; ++l) {
    const int2 d3 = level(l + 3);
    const SimpleReads in = simple_reads<kDual>(h0, x, y, z);  // on their way before the loads ahead
    const SimpleRec h2 = packet(d2);
    const SimpleVals v1 = simple_values(T, h1);
    replay_simple<kDual>(T, x, y, z, zret, h0, v0, in, tol);
    __syncthreads();
    h0 = h1;
    h1 = h2;
    v0 = v1;
    d2 = d3;
  }
}

// A run of small levels in one workgroup, which meets at a barrier after each.
// Its first waves replay the line records, the others the rest, as many of each
// as the run's largest level fills (a chain of single records: one wave, 0.7 us a
// level against 1.1 with sixteen).  All waves run on one CU, so the barrier's
// workgroup-scope fence makes one level's global stores visible to the next
// level's loads.  Both kinds of wave come to the barrier once a level.
template <bool kDual>
__global__ void __launch_bounds__(kLevelBlock)
    k_replay_levels(gp_tape_dev T, gp_orig_dev O, double* x, double* y, double* z, uint8_t* zret,
                    const int32_t* __restrict__ line, const int32_t* __restrict__ simple,
                    const gpk_replay_level* __restrict__ levels, int32_t nlevels, int32_t line_waves, double tol) {
  const int32_t wave = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(threadIdx.x) >> 6);
  if (wave < line_waves) replay_level_lines<kDual>(T, O, x, y, z, zret, line, levels, nlevels, tol);
  else replay_level_simples<kDual>(T, x, y, z, zret, simple, levels, nlevels, line_waves, tol);
}

// gpu_postsolve.cu:162-180, 568-603: z_j from r = c_j - (A^T y)_j and the
// bound state of x_j.  (A^T y)_j is summed in AT order; columns longer than
// kLongCol are left to k_project_duals_long, which loads a column 64 entries
// at a time across a wave and adds the products in the same order.
constexpr int32_t kLongCol = 64;

__device__ inline double project_dual(const gp_orig_dev& O, int32_t col, double aty, const double* x, double tol) {
  const double r = O.c[col] - aty;
  const double xj = x[col], lj = O.l[col], uj = O.u[col];
  const bool atl = at_lower(xj, lj, tol), atu = at_upper(xj, uj, tol);
  double zj;
  if (atl && atu) zj = r;
  else if (!atl && !atu) zj = 0.0;
  else if (atl) zj = fmax(r, 0.0);
  else zj = fmin(r, 0.0);
  const double eps = fmin(tol, 1.0e-12);
  if (zj > eps && !isfinite(lj)) zj = 0.0;
  else if (zj < -eps && !isfinite(uj)) zj = 0.0;
  return zj;
}

// The sum over q in [0, count) of val[q] * vec[idx[q]] in q order.  The loads of
// eight terms go out together, past the end the last term again.
__device__ inline double column_dot(const int32_t* __restrict__ idx, const double* __restrict__ val,
                                    const double* __restrict__ vec, int32_t count) {
  constexpr int U = 8;
  double s = 0.0;
#pragma unroll 1
  for (int32_t q = 0; q < count; q += U) {
    int32_t j[U];
    double a[U], v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int32_t p = min(q + k, count - 1);
      j[k] = idx[p];
      a[k] = val[p];
    }
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = vec[j[k]];
#pragma unroll
    for (int k = 0; k < U; ++k)
      if (q + k < count) s += a[k] * v[k];
  }
  return s;
}

__global__ void k_project_duals(gp_orig_dev O, const uint8_t* prot, const double* x, const double* y, double* z,
                                int32_t n, double tol, int32_t* long_count, int32_t* long_cols) {
  const int32_t col = blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= n || (prot && prot[col])) return;
  const int32_t b = O.at_ptr[col], e = O.at_ptr[col + 1];
  if (e - b > kLongCol) {
    long_cols[atomicAdd(long_count, 1)] = col;
    return;
  }
  const double aty = column_dot(O.at_idx + b, O.at_val + b, y, e - b);
  z[col] = project_dual(O, col, aty, x, tol);
}

// Lane t's double, in every lane (t the same in all lanes).
__device__ inline double lane_f64(double v, int t) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), t);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), t);
  return __hiloint2double(hi, lo);
}

// One wave per listed column; a fixed grid whose waves stride over the list.
// The column's products are formed kLongSlices x 64 at a time (all loads of
// the batch in flight together) and added to the running sum one by one in
// AT order, each read from its lane into scalar registers, so the serial
// chain costs one add per entry.
constexpr int kLongSlices = 4;
constexpr int kLongGrid = 2048;
__global__ void k_project_duals_long(gp_orig_dev O, const double* x, const double* y, double* z, double tol,
                                     const int32_t* long_count, const int32_t* long_cols) {
  const int lane = lane_id();
  const int32_t waves = gridDim.x * (blockDim.x / 64);
  const int32_t count = *long_count;
  for (int32_t w = blockIdx.x * (blockDim.x / 64) + static_cast<int32_t>(threadIdx.x / 64); w < count; w += waves) {
    const int32_t col = long_cols[w];
    const int32_t b = O.at_ptr[col], e = O.at_ptr[col + 1];
    double aty = 0.0;
    for (uint32_t base = 0, n = row_length(b, e); base < n; base += 64 * kLongSlices) {
      int32_t j[kLongSlices];
      double a[kLongSlices], p[kLongSlices];
#pragma unroll
      for (int u = 0; u < kLongSlices; ++u) {
        const uint32_t o = base + 64 * u + lane;
        const int32_t q = row_entry(b, e, o);
        j[u] = o < n ? O.at_idx[q] : -1;
        a[u] = o < n ? O.at_val[q] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < kLongSlices; ++u) p[u] = j[u] >= 0 ? a[u] * y[j[u]] : 0.0;
#pragma unroll
      for (int u = 0; u < kLongSlices; ++u) {
        const uint32_t s0 = base + 64 * u;
        if (s0 + 64 <= n) {
#pragma unroll
          for (int t = 0; t < 64; ++t) aty += lane_f64(p[u], t);
        } else {
          for (uint32_t t = s0; t < n; ++t) aty += lane_f64(p[u], static_cast<int>(t - s0));
        }
      }
    }
    if (lane == 0) z[col] = project_dual(O, col, aty, x, tol);
  }
}

// Lengths and packed copies of selected CSR lines (the original rows and
// columns that the host schedules the dual replay by).
__global__ void k_seg_lengths(const int32_t* ptr, const int32_t* list, int32_t count, int32_t* len) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) len[i] = ptr[list[i] + 1] - ptr[list[i]];
}

__global__ void k_seg_copy(const int32_t* ptr, const int32_t* idx, const int32_t* list, int32_t count,
                           const int32_t* off, int32_t* out) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const int32_t b = ptr[list[i]], e = ptr[list[i] + 1];
  int32_t o = off[i];
  for (int32_t q = b; q < e; ++q) out[o++] = idx[q];
}

// Columns whose dual the replay determines exactly (gpu_postsolve.cu:1370-1402).
__global__ void k_protect(gp_tape_dev T, int32_t n, uint8_t* prot) {
  const int32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= T.count) return;
  const int32_t i0 = T.index_starts[k];
  const int32_t t = T.types[k];
  int32_t a = -1, b = -1;
  if (t == 2) a = T.indices[i0];
  else if (t == 13) { a = T.indices[i0]; b = T.indices[i0 + 1]; }
  else if (t == 1) a = T.indices[i0 + 1];
  else if (t == 3) a = T.indices[i0];
  if (a >= 0 && a < n) prot[a] = 1;
  if (b >= 0 && b < n) prot[b] = 1;
}

}  // namespace

#define GPK_LAUNCH(kernel, n, ...)                                                      \
  do {                                                                                  \
    if ((n) > 0) hipLaunchKernelGGL(kernel, dim3(grid_for(n)), dim3(kBlock), 0, stream, __VA_ARGS__); \
    return hipGetLastError();                                                           \
  } while (0)

extern "C" {

hipError_t gpk_map_tape_indices(int32_t count, int32_t* idx, const uint8_t* kind, const int32_t* row_red2org,
                                int32_t m, const int32_t* col_red2org, int32_t n, hipStream_t stream) {
  GPK_LAUNCH(k_map_tape_indices, count, count, idx, kind, row_red2org, m, col_red2org, n);
}
hipError_t gpk_scatter(const double* src, const int32_t* red2org, int32_t n_red, double* dst, hipStream_t stream) {
  GPK_LAUNCH(k_scatter, n_red, src, red2org, n_red, dst);
}
hipError_t gpk_mark(const int32_t* red2org, int32_t n_red, uint8_t* mask, hipStream_t stream) {
  GPK_LAUNCH(k_mark, n_red, red2org, n_red, mask);
}
hipError_t gpk_restore_fixed(const int32_t* idx, const double* val, int32_t count, double* x, hipStream_t stream) {
  GPK_LAUNCH(k_restore_fixed, count, idx, val, count, x);
}
hipError_t gpk_pack_records(gp_tape_dev tape, gp_orig_dev orig, gpk_replay_slots slots, int32_t dual_line,
                            int32_t has_y, hipStream_t stream) {
  const int32_t lb = slots.line_slots > 0 ? static_cast<int32_t>(grid_for(slots.line_slots, kBlock / kRecLanes)) : 0;
  const int32_t sb = slots.simple_slots > 0 ? static_cast<int32_t>(grid_for(slots.simple_slots)) : 0;
  if (lb + sb == 0) return hipSuccess;
  hipLaunchKernelGGL(k_pack_records, dim3(lb + sb), dim3(kBlock), 0, stream, tape, orig, slots, dual_line, has_y, lb);
  return hipGetLastError();
}
hipError_t gpk_replay_list(gp_tape_dev tape, gp_orig_dev orig, double* x, double* y, double* z, uint8_t* zret,
                           const int32_t* line, int32_t lines, const int32_t* simple, int32_t simples, int32_t dual,
                           double tol, hipStream_t stream) {
  const int32_t lb = lines > 0 ? static_cast<int32_t>(grid_for(lines, kBlock / kRecLanes)) : 0;
  const int32_t sb = simples > 0 ? static_cast<int32_t>(grid_for(simples)) : 0;
  if (lb + sb == 0) return hipSuccess;
  if (dual)
    hipLaunchKernelGGL(k_replay_list<true>, dim3(lb + sb), dim3(kBlock), 0, stream, tape, orig, x, y, z, zret, line,
                       lines, simple, simples, lb, tol);
  else
    hipLaunchKernelGGL(k_replay_list<false>, dim3(lb + sb), dim3(kBlock), 0, stream, tape, orig, x, y, z, zret, line,
                       lines, simple, simples, lb, tol);
  return hipGetLastError();
}
hipError_t gpk_replay_levels(gp_tape_dev tape, gp_orig_dev orig, double* x, double* y, double* z, uint8_t* zret,
                             const int32_t* line, const int32_t* simple, const gpk_replay_level* levels,
                             int32_t nlevels, int32_t line_waves, int32_t simple_waves, int32_t dual, double tol,
                             hipStream_t stream) {
  if (nlevels <= 0) return hipSuccess;
  const int32_t waves = line_waves + simple_waves;
  if (line_waves < 0 || simple_waves < 0 || waves < 1 || waves > GPK_REPLAY_WAVES) return hipErrorInvalidValue;
  const auto run = dual ? k_replay_levels<true> : k_replay_levels<false>;
  hipLaunchKernelGGL(run, dim3(1), dim3(64 * waves), 0, stream, tape, orig, x, y, z, zret, line, simple, levels,
                     nlevels, line_waves, tol);
  return hipGetLastError();
}
hipError_t gpk_seg_lengths(const int32_t* ptr, const int32_t* list, int32_t count, int32_t* len, hipStream_t stream) {
  GPK_LAUNCH(k_seg_lengths, count, ptr, list, count, len);
}
hipError_t gpk_seg_copy(const int32_t* ptr, const int32_t* idx, const int32_t* list, int32_t count,
                        const int32_t* off, int32_t* out, hipStream_t stream) {
  GPK_LAUNCH(k_seg_copy, count, ptr, idx, list, count, off, out);
}
hipError_t gpk_protect_columns(gp_tape_dev tape, int32_t n, uint8_t* prot, hipStream_t stream) {
  GPK_LAUNCH(k_protect, tape.count, tape, n, prot);
}
hipError_t gpk_project_duals(gp_orig_dev orig, const uint8_t* prot, const double* x, const double* y, double* z,
                             int32_t n, double tol, int32_t* long_count, int32_t* long_cols, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_project_duals, dim3(grid_for(n)), dim3(kBlock), 0, stream, orig, prot, x, y, z, n, tol,
                     long_count, long_cols);
  hipLaunchKernelGGL(k_project_duals_long, dim3(kLongGrid), dim3(kBlock), 0, stream, orig, x, y, z, tol, long_count,
                     long_cols);
  return hipGetLastError();
}

}  // extern "C"
