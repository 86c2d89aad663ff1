// Host-side infrastructure: context, device memory, scans, compaction,
// transpose and the FixedCol tape packer.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <shared_mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "gp_host.hpp"

namespace gpu_presolver::amd {

using presolve::DeviceCsrMatrix;
using presolve::PostsolveDualMode;
using presolve::PostsolveReductionType;
using presolve::PostsolveTape;

namespace {

// Keep freed blocks of the device's default pool cached for reuse: rules
// allocate and release their scratch once per call.
void configure_pool_once() {
  static std::once_flag once;
  std::call_once(once, []() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    hipMemPool_t pool = nullptr;
    if (hipDeviceGetDefaultMemPool(&pool, dev) != hipSuccess || pool == nullptr) return;
    uint64_t threshold = std::numeric_limits<uint64_t>::max();
    (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &threshold);
  });
}

thread_local Ctx* t_current = nullptr;
thread_local Ctx* t_own = nullptr;  // the thread's own context (created on first use)

}  // namespace

Ctx::Ctx(hipStream_t stream, bool own_stream) {
  configure_pool_once();
  if (stream == nullptr && own_stream) {
    check(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate");
    own_stream_ = true;
  } else {
    stream_ = stream;
    own_stream_ = false;
  }
  check(hipMalloc(&d_flags_, sizeof(int32_t) * kFlags * kFlagSlots), "hipMalloc flags");
  check(hipMemsetAsync(d_flags_, 0, sizeof(int32_t) * kFlags * kFlagSlots, stream_), "hipMemset flags");
  check(hipMalloc(&d_tickets_, sizeof(int32_t) * kTickets), "hipMalloc tickets");
  check(hipMemsetAsync(d_tickets_, 0, sizeof(int32_t) * kTickets, stream_), "hipMemset tickets");
  check(hipHostMalloc(&h_error_, sizeof(int32_t), hipHostMallocMapped), "hipHostMalloc error flag");
  *h_error_ = 0;
  check(hipHostGetDevicePointer(reinterpret_cast<void**>(&d_error_), h_error_, 0), "hipHostGetDevicePointer");
  check(hipHostMalloc(&h_mail_, sizeof(uint32_t) * (4 + kMailWords), hipHostMallocMapped | hipHostMallocCoherent),
        "hipHostMalloc mail");
  std::memset(h_mail_, 0, sizeof(uint32_t) * (4 + kMailWords));
  check(hipHostGetDevicePointer(reinterpret_cast<void**>(&d_mail_), h_mail_, 0), "hipHostGetDevicePointer mail");
}

gpk_lookback Ctx::lookback(int64_t tiles) {
  if (tiles > status_cap_) {
    int64_t cap = 1024;
    while (cap < tiles) cap <<= 1;
    sync("look-back status growth");
    if (d_status_) check(hipFree(d_status_), "hipFree look-back status");
    d_status_ = nullptr;
    check(hipMalloc(&d_status_, sizeof(uint64_t) * static_cast<size_t>(cap)), "hipMalloc look-back status");
    check(hipMemsetAsync(d_status_, 0, sizeof(uint64_t) * static_cast<size_t>(cap), stream_),
          "hipMemset look-back status");
    status_cap_ = cap;
  }
  if (ticket_ == kTickets) {
    check(hipMemsetAsync(d_tickets_, 0, sizeof(int32_t) * kTickets, stream_), "hipMemset tickets");
    ticket_ = 0;
  }
  epoch_ = epoch_ + 1 >= (1u << 30) ? 1u : epoch_ + 1;
  return gpk_lookback{d_status_, d_tickets_ + ticket_++, d_error_, epoch_};
}

Ctx::~Ctx() {
  if (stream_) (void)hipStreamSynchronize(stream_);
  release_cached_blocks(stream_);
  if (stream_) (void)hipStreamSynchronize(stream_);
  (void)hipFree(d_flags_);
  (void)hipFree(d_tickets_);
  if (d_status_) (void)hipFree(d_status_);
  (void)hipHostFree(h_error_);
  (void)hipHostFree(h_mail_);
  if (h_stage_) (void)hipHostFree(h_stage_);
  if (own_stream_) (void)hipStreamDestroy(stream_);
}

// Flag words come from a ring of zeroed slots; the whole ring is cleared
// (stream-ordered, after every earlier use) once per kFlagSlots handouts.
int32_t* Ctx::flags() {
  if (slot_ == kFlagSlots) {
    check(hipMemsetAsync(d_flags_, 0, sizeof(int32_t) * kFlags * kFlagSlots, stream_), "hipMemset flags");
    slot_ = 0;
  }
  cur_ = d_flags_ + static_cast<size_t>(slot_++) * kFlags;
  return cur_;
}

const int32_t* Ctx::read_flags(int count) {
  static_assert(kFlags <= kMailWords, "a flag slot fits the mailbox");
  if (count < 0 || count > kFlags) throw std::invalid_argument("read_flags: count out of range");
  return reinterpret_cast<const int32_t*>(mail(cur_ ? cur_ : d_flags_, count, "read flags"));
}

void Ctx::check_error_flag(const char* context) {
  if (*h_error_ != 0) {
    *h_error_ = 0;
    throw std::runtime_error(std::string(context) + ": a single-pass scan exceeded its spin limit");
  }
}

void Ctx::sync(const char* context) { (void)mail(nullptr, 0, context); }

size_t Ctx::stage_reserve(size_t bytes, const char* context) {
  size_t off = (stage_used_ + 255) & ~static_cast<size_t>(255);
  if (off + bytes > stage_cap_) {
    if (stage_used_ > 0) sync(context);  // staged copies in flight complete (and the area is released)
    off = 0;
    if (bytes > stage_cap_) {
      if (h_stage_) check(hipHostFree(h_stage_), "hipHostFree staging");
      h_stage_ = d_stage_ = nullptr;
      stage_cap_ = 0;
      size_t cap = size_t{1} << 20;
      while (cap < bytes) cap <<= 1;
      check(hipHostMalloc(reinterpret_cast<void**>(&h_stage_), cap, hipHostMallocMapped | hipHostMallocCoherent),
            "hipHostMalloc staging");
      check(hipHostGetDevicePointer(reinterpret_cast<void**>(&d_stage_), h_stage_, 0), "staging device pointer");
      stage_cap_ = cap;
    }
  }
  stage_used_ = off + bytes;
  return off;
}

// Copies larger than this bypass the staging area (a direct copy and a
// stream synchronization), so the pinned area stays modest.
constexpr size_t kStageMaxBytes = size_t{64} << 20;

void Ctx::download(void* dst, const void* dev, size_t bytes, const char* context) {
  if (bytes == 0) return;
  if (bytes > kStageMaxBytes) {
    check(hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, stream_), context);
    check(hipStreamSynchronize(stream_), context);
    return;
  }
  const size_t off = stage_reserve(bytes, context);
  enqueue_copy(gpk_copy_seg{d_stage_ + off, dev, static_cast<int64_t>(bytes)}, context);
  downloads_.push_back(Download{dst, off, bytes});
}

void Ctx::enqueue_copy(const gpk_copy_seg& seg, const char* context) {
  if (!grouping_) {
    check(gpk_copy_many(&seg, 1, stream_), context);
    return;
  }
  pending_.push_back(seg);
  if (pending_.size() == GPK_COPY_MAX) flush_pending(context);
}

void Ctx::flush_pending(const char* context) {
  if (pending_.empty()) return;
  const hipError_t e = gpk_copy_many(pending_.data(), static_cast<int32_t>(pending_.size()), stream_);
  pending_.clear();
  check(e, context);
}

void Ctx::end_copy_group(const char* context) {
  grouping_ = false;
  flush_pending(context);
}

void* Ctx::stage(const void* host, size_t bytes, void* dst_after, size_t dst_bytes, const char* context) {
  if (bytes == 0) return nullptr;
  if (dst_bytes > bytes) throw std::invalid_argument("Ctx::stage: dst_bytes exceeds the staged bytes");
  if (bytes > kStageMaxBytes) throw std::length_error("Ctx::stage: more than 64 MB to stage");
  const size_t off = stage_reserve(bytes, context);
  std::memcpy(h_stage_ + off, host, bytes);
  if (dst_after && dst_bytes > 0) downloads_.push_back(Download{dst_after, off, dst_bytes});
  return d_stage_ + off;
}

void Ctx::upload(void* dev, const void* host, size_t bytes, const char* context) {
  if (bytes == 0) return;
  if (bytes > kStageMaxBytes) {
    check(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream_), context);
    check(hipStreamSynchronize(stream_), context);
    return;
  }
  const size_t off = stage_reserve(bytes, context);
  std::memcpy(h_stage_ + off, host, bytes);
  enqueue_copy(gpk_copy_seg{dev, d_stage_ + off, static_cast<int64_t>(bytes)}, context);
}

void Ctx::finish_downloads() {
  for (const Download& d : downloads_) std::memcpy(d.dst, h_stage_ + d.offset, d.bytes);
  downloads_.clear();
  stage_used_ = 0;
  if (after_.empty()) return;
  std::vector<std::function<void()>> run;
  run.swap(after_);
  for (auto& fn : run) fn();
}

const uint32_t* Ctx::mail(const void* dev, int words, const char* context) {
  grouping_ = false;  // a wait closes the group; its copies precede the wait
  flush_pending(context);
  ++syncs_;
  if (++mail_seq_ == 0) mail_seq_ = 1;
  const uint32_t seq = mail_seq_;
  check(gpk_mail(static_cast<const uint32_t*>(dev), words, d_mail_, seq, stream_), context);
  volatile uint32_t* word = h_mail_;
  const auto t0 = std::chrono::steady_clock::now();
  // Spin briefly (most decisions wait a few microseconds), then yield; every
  // few thousand polls the stream is asked for an error so a failed launch
  // does not leave the host waiting.
  for (int64_t polls = 0; word[0] != seq; ++polls) {
    if (polls < 2048) {
      __builtin_ia32_pause();
      continue;
    }
    if ((polls & 4095) == 0) {
      const hipError_t e = hipStreamQuery(stream_);
      if (e != hipSuccess && e != hipErrorNotReady) throw HipError(context, e);
    }
    std::this_thread::yield();
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  wait_s_ += std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  finish_downloads();
  check_error_flag(context);
  return const_cast<const uint32_t*>(h_mail_ + 4);
}

Ctx& ctx() {
  if (t_current) return *t_current;
  if (!t_own) t_own = new Ctx();  // lives for the thread
  return *t_own;
}

void Ctx::abandon() noexcept {
  if (stream_) (void)hipStreamSynchronize(stream_);
  grouping_ = false;
  pending_.clear();
  downloads_.clear();
  after_.clear();
  stage_used_ = 0;
  if (h_error_) *h_error_ = 0;
}

void abandon_pending_copies() noexcept {
  Ctx* c = t_current ? t_current : t_own;
  if (c) c->abandon();
}

JobMode& job_mode() {
  thread_local JobMode mode;
  return mode;
}

namespace {

// Device-wide waits go on beside each other and captures beside each other, but
// not the one beside the other; who comes first goes first, so neither kind is
// kept out for good.
class CaptureGate {
 public:
  void enter(int kind) {
    std::unique_lock<std::mutex> lk(mu_);
    const uint64_t ticket = next_++;
    cv_.wait(lk, [&] { return ticket == turn_ && inside_[1 - kind] == 0; });
    ++turn_;
    ++inside_[kind];
    cv_.notify_all();
  }
  void leave(int kind) {
    std::lock_guard<std::mutex> lk(mu_);
    --inside_[kind];
    cv_.notify_all();
  }

 private:
  std::mutex mu_;
  std::condition_variable cv_;
  uint64_t next_ = 0, turn_ = 0;
  int inside_[2] = {0, 0};
};

constexpr int kWait = 0, kCapture = 1;

// Never destroyed: a thread may still be inside when the process ends.
CaptureGate& capture_gate() {
  static CaptureGate* g = new CaptureGate;
  return *g;
}

}  // namespace

void device_sync(const char* what) {
  capture_gate().enter(kWait);
  const hipError_t st = hipDeviceSynchronize();
  capture_gate().leave(kWait);
  check(st, what);
}

CaptureSection::CaptureSection() { capture_gate().enter(kCapture); }
CaptureSection::~CaptureSection() { capture_gate().leave(kCapture); }

ScopedCtx::ScopedCtx(Ctx& c) : prev_(t_current) { t_current = &c; }
ScopedCtx::~ScopedCtx() { t_current = prev_; }

// ---- caching device allocator ----------------------------------------------
// Blocks are rounded up to a power of two (>= 512 B) and, when released, kept
// on a free list of the stream they were allocated on.  Work on one stream
// runs in order, so a block released after its last use can be handed to the
// next allocation on that stream without any synchronization; the device is
// only asked for memory (hipMallocAsync) on a miss.  This replaces one
// hipMallocAsync/hipFreeAsync pair per temporary buffer of every rule call.
// Each stream has its own arena and lock, so the serving workers (one stream
// each) never wait for one another here.
namespace {
struct StreamArena {
  std::mutex mu;
  std::unordered_map<size_t, std::vector<void*>> free_lists;  // size class -> blocks
  std::unordered_map<void*, size_t> live;                     // block -> size class
};
struct Arena {
  std::shared_mutex mu;  // guards the map (arenas are never removed)
  std::unordered_map<hipStream_t, std::unique_ptr<StreamArena>> streams;
};
Arena& arena() {
  static auto* a = new Arena();  // never destroyed: blocks may be released at exit
  return *a;
}
StreamArena& stream_arena(hipStream_t stream) {
  thread_local hipStream_t last_stream = nullptr;
  thread_local StreamArena* last = nullptr;
  if (last && last_stream == stream) return *last;
  Arena& a = arena();
  {
    std::shared_lock<std::shared_mutex> lock(a.mu);
    auto it = a.streams.find(stream);
    if (it != a.streams.end()) {
      last_stream = stream;
      last = it->second.get();
      return *last;
    }
  }
  std::unique_lock<std::shared_mutex> lock(a.mu);
  auto& slot = a.streams[stream];
  if (!slot) {
    slot = std::make_unique<StreamArena>();
    slot->live.reserve(1024);
  }
  last_stream = stream;
  last = slot.get();
  return *last;
}
size_t size_class(size_t bytes) {
  size_t c = 512;
  while (c < bytes) c <<= 1;
  return c;
}
// Returns a live block to the free list of the arena that allocated it.
bool recycle(StreamArena& sa, void* p) {
  std::lock_guard<std::mutex> lock(sa.mu);
  auto it = sa.live.find(p);
  if (it == sa.live.end()) return false;
  sa.free_lists[it->second].push_back(p);
  sa.live.erase(it);
  return true;
}
}  // namespace

void release_cached_blocks(hipStream_t stream) noexcept {
  StreamArena& sa = stream_arena(stream);
  std::vector<void*> blocks;
  {
    std::lock_guard<std::mutex> lock(sa.mu);
    for (auto& kv : sa.free_lists) blocks.insert(blocks.end(), kv.second.begin(), kv.second.end());
    sa.free_lists.clear();
  }
  for (void* p : blocks) (void)hipFreeAsync(p, stream);
}

void* dev_alloc(size_t bytes, hipStream_t stream, const char* context) {
  StreamArena& sa = stream_arena(stream);
  const size_t cls = size_class(bytes);
  {
    std::lock_guard<std::mutex> lock(sa.mu);
    auto f = sa.free_lists.find(cls);
    if (f != sa.free_lists.end() && !f->second.empty()) {
      void* p = f->second.back();
      f->second.pop_back();
      sa.live.emplace(p, cls);
      return p;
    }
  }
  void* p = nullptr;
  hipError_t st = hipMallocAsync(&p, cls, stream);
  if (st == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    release_cached_blocks(stream);
    st = hipMallocAsync(&p, cls, stream);
  }
  check(st, context);
  std::lock_guard<std::mutex> lock(sa.mu);
  sa.live.emplace(p, cls);
  return p;
}

void dev_free(void* p, hipStream_t stream) noexcept {
  if (!p) return;
  if (recycle(stream_arena(stream), p)) return;
  {  // allocated on another stream
    Arena& a = arena();
    StreamArena* owner = nullptr;
    {
      std::shared_lock<std::shared_mutex> lock(a.mu);
      for (auto& kv : a.streams) {
        std::lock_guard<std::mutex> l2(kv.second->mu);
        if (kv.second->live.count(p)) {
          owner = kv.second.get();
          break;
        }
      }
    }
    if (owner) {
      // The owning stream's next allocation may hand this block out with no
      // ordering against work still queued on the freeing stream: that work
      // finishes first.
      (void)hipStreamSynchronize(stream);
      if (recycle(*owner, p)) return;
    }
  }
  // Memory the caller allocated with hipMalloc (e.g. a plan's new_A).
  (void)hipStreamSynchronize(stream);
  (void)hipFree(p);
}

void row_activity(const int32_t* ptr, const int32_t* idx, const double* val, int32_t m, int32_t n, int32_t nnz, const double* l,
                  const double* u, double ztol, double* min_fin, double* max_fin, int32_t* neg_inf, int32_t* pos_inf,
                  hipStream_t stream) {
  if (m <= 0) return;
  void* lu = dev_alloc(sizeof(double) * 2 * static_cast<size_t>(n > 0 ? n : 1), stream, "packed bounds");
  hipError_t st = gpk_pack_lu(l, u, n, static_cast<double*>(lu), stream);
  if (st == hipSuccess)
    st = gpk_row_activity_lu(ptr, idx, val, m, nnz, static_cast<const double*>(lu), ztol, min_fin, max_fin, neg_inf,
                             pos_inf, stream);
  dev_free(lu, stream);  // stream-ordered reuse: later work on `stream` runs after the kernels
  check(st, "row activity");
}

void scan_mask_launch(const uint8_t* mask, int32_t n, int32_t* out) {
  Ctx& c = ctx();
  if (n <= 0) check(gpk_fill_i32(out, 0, 1, c.stream()), "scan empty");
  else check(gpk_scan_lb_mask(mask, out, n, c.lookback(gpk_lookback_tiles(n)), c.stream()), "scan mask");
}

int32_t scan_mask_count(const uint8_t* mask, int32_t n, int32_t* out) {
  scan_mask_launch(mask, n, out);
  return n <= 0 ? 0 : ctx().scalar_to_host(out + n, "scan total");
}

void scan_counts_launch(const int32_t* in, int32_t n, int32_t* out) {
  Ctx& c = ctx();
  if (n <= 0) check(gpk_fill_i32(out, 0, 1, c.stream()), "scan empty");
  else check(gpk_scan_lb_i32(in, out, n, c.lookback(gpk_lookback_tiles(n)), c.stream()), "scan counts");
}

int32_t scan_counts(const int32_t* in, int32_t n, int32_t* out) {
  scan_counts_launch(in, n, out);
  return n <= 0 ? 0 : ctx().scalar_to_host(out + n, "scan total");
}

// Terms fetched together with their count (32 KB).
constexpr int32_t kSpeculativeTerms = 4096;

double ordered_masked_sum(const uint8_t* mask, const double* vals, int32_t n) {
  if (n <= 0) return 0.0;
  Ctx& c = ctx();
  hipStream_t s = c.stream();
  DBuf<int32_t> prefix(static_cast<int64_t>(n) + 1);
  DBuf<double> packed(n);
  check(gpk_scan_lb_mask(mask, prefix, n, c.lookback(gpk_lookback_tiles(n)), s), "scan objective mask");
  check(gpk_pack_f64(mask, vals, prefix, n, packed, s), "pack objective terms");
  // The first kSpeculativeTerms packed terms travel with the count, so the
  // usual case (few terms) costs one wait.
  const int32_t head = std::min<int32_t>(n, kSpeculativeTerms);
  std::vector<double> h(static_cast<size_t>(head));
  c.download(h.data(), packed.get(), sizeof(double) * static_cast<size_t>(head), "objective terms");
  const int32_t k = c.scalar_to_host(prefix.get() + n, "objective term count");
  if (k > head) {
    h.resize(static_cast<size_t>(k));
    c.download(h.data() + head, packed.get() + head, sizeof(double) * static_cast<size_t>(k - head),
               "objective terms");
    c.sync("objective terms");
  }
  double sum = 0.0;
  for (int32_t t = 0; t < k; ++t) sum += h[static_cast<size_t>(t)];
  return sum;
}

void add_ordered_masked_sum(double* target, const uint8_t* mask, const double* vals, int32_t n) {
  Ctx& c = ctx();
  if (!c.defer_objective_sums || n <= 0) {
    *target += ordered_masked_sum(mask, vals, n);
    return;
  }
  hipStream_t s = c.stream();
  // The packed terms and the count stay allocated until the addition has run.
  struct Terms {
    DBuf<int32_t> prefix;
    DBuf<double> packed;
    std::vector<double> h;
    int32_t k = 0;
  };
  auto t = std::make_shared<Terms>();
  t->prefix.alloc(static_cast<int64_t>(n) + 1);
  t->packed.alloc(n);
  check(gpk_scan_lb_mask(mask, t->prefix, n, c.lookback(gpk_lookback_tiles(n)), s), "scan objective mask");
  check(gpk_pack_f64(mask, vals, t->prefix, n, t->packed, s), "pack objective terms");
  const int32_t head = std::min<int32_t>(n, kSpeculativeTerms);
  t->h.resize(static_cast<size_t>(head));
  c.begin_copy_group();
  c.download(t->h.data(), t->packed.get(), sizeof(double) * static_cast<size_t>(head), "objective terms");
  c.download(&t->k, t->prefix.get() + n, sizeof(int32_t), "objective term count");
  c.end_copy_group("objective terms");
  c.after_wait([t, target, head, s] {
    const int32_t k = t->k;
    if (k > head) {  // the stream is idle: the rest comes over directly
      t->h.resize(static_cast<size_t>(k));
      check(hipMemcpyAsync(t->h.data() + head, t->packed.get() + head, sizeof(double) * static_cast<size_t>(k - head),
                           hipMemcpyDeviceToHost, s),
            "objective terms");
      check(hipStreamSynchronize(s), "objective terms");
    }
    double sum = 0.0;
    for (int32_t q = 0; q < k; ++q) sum += t->h[static_cast<size_t>(q)];
    *target += sum;
  });
}

void free_csr(DeviceCsrMatrix& A) noexcept {
  hipStream_t s = ctx().stream();
  dev_free(A.rowPtr, s);
  dev_free(A.colVal, s);
  dev_free(A.nzVal, s);
  A.rowPtr = nullptr;
  A.colVal = nullptr;
  A.nzVal = nullptr;
}

// ---- compaction (compact_csr_by_masks_gpu, gpu_presolve.cu:1881-1978) -------
namespace {
size_t align256(size_t b) { return (b + 255) & ~size_t{255}; }
size_t compact_words(int32_t nnz) {
  return (static_cast<size_t>(gpk_compact_chunks(nnz)) << gpk_compact_shift(nnz)) / 64;
}
// A side's entry map, kept-entry words and their prefix sums.
size_t compact_work_bytes(int32_t nnz) {
  const size_t words = compact_words(nnz);
  return align256(sizeof(int32_t) * static_cast<size_t>(nnz)) + align256(sizeof(uint64_t) * words) +
         align256(sizeof(int32_t) * words);
}
gpk_compact_side compact_side(const DeviceCsrMatrix& M, const int32_t* row_map, const gpk_rank_word* col_rank,
                              const int32_t* chunk_row, char* work) {
  const size_t words = compact_words(M.nnz);
  gpk_compact_side s{};
  s.ptr = M.rowPtr;
  s.idx = M.colVal;
  s.val = M.nzVal;
  s.m_old = M.rows;
  s.nnz = M.nnz;
  s.row_map = row_map;
  s.col_rank = col_rank;
  s.chunk_row = chunk_row;
  s.jn = reinterpret_cast<int32_t*>(work);
  work += align256(sizeof(int32_t) * static_cast<size_t>(M.nnz));
  s.mask = reinterpret_cast<uint64_t*>(work);
  work += align256(sizeof(uint64_t) * words);
  s.word_pre = reinterpret_cast<int32_t*>(work);
  return s;
}
}  // namespace

CompactStart compact_start(const DeviceCsrMatrix& A, const int32_t* row_map, const gpk_rank_word* col_rank,
                           const int32_t* chunk_row, int32_t* kept, const DeviceCsrMatrix* AT, const int32_t* col_map,
                           const gpk_rank_word* row_rank, const int32_t* t_chunk_row) {
  if (AT != nullptr && (AT->rows != A.cols || AT->cols != A.rows || AT->nnz != A.nnz))
    throw std::logic_error("compact_start: AT is not the transpose shape of A");
  CompactStart st;
  st.A = &A;
  st.AT = AT;
  if (A.rows == 0 || A.cols == 0 || A.nnz == 0) return st;  // *kept stays as the caller zeroed it
  const int32_t chunks = gpk_compact_chunks(A.nnz);
  const size_t side = compact_work_bytes(A.nnz);
  // Room for the transpose as well: it may be added after the sizes are read.
  st.work.alloc(static_cast<int64_t>(2 * side + sizeof(int32_t) * (2 * static_cast<size_t>(chunks) + 1)),
                "compact work");
  st.cnt = reinterpret_cast<int32_t*>(st.work.get() + 2 * side);
  st.a = compact_side(A, row_map, col_rank, chunk_row, st.work.get());
  if (AT != nullptr) st.t = compact_side(*AT, col_map, row_rank, t_chunk_row, st.work.get() + side);
  check(gpk_compact_map(st.a, st.t, st.cnt, kept, ctx().stream()), "compact map");
  return st;
}

void compact_add_transpose(CompactStart& st, const DeviceCsrMatrix& AT, const int32_t* col_map,
                           const gpk_rank_word* row_rank, const int32_t* t_chunk_row) {
  if (AT.rows != st.A->cols || AT.cols != st.A->rows || AT.nnz != st.A->nnz)
    throw std::logic_error("compact_add_transpose: AT is not the transpose shape of A");
  st.AT = &AT;
  if (st.cnt == nullptr) return;
  st.t = compact_side(AT, col_map, row_rank, t_chunk_row, st.work.get() + compact_work_bytes(AT.nnz));
  check(gpk_compact_map(gpk_compact_side{}, st.t, st.cnt + gpk_compact_chunks(AT.nnz), nullptr, ctx().stream()),
        "compact map of the transpose");
}

CompactOut compact_finish(CompactStart& st, int32_t m_new, int32_t n_new, int32_t nnz_new,
                          const gpk_apply_gathers_args* gathers) {
  Ctx& c = ctx();
  hipStream_t s = c.stream();
  CompactOut out;
  out.A.rows = out.AT.cols = m_new;
  out.A.cols = out.AT.rows = n_new;
  DBuf<int32_t> ptr(static_cast<int64_t>(m_new) + 1, "compact rowPtr"), t_ptr;
  if (st.AT != nullptr) t_ptr.alloc(static_cast<int64_t>(n_new) + 1, "compact AT rowPtr");
  if (m_new == 0 || n_new == 0 || st.cnt == nullptr) {
    CopyBatch zeros;
    zeros.zero(ptr.get(), static_cast<int64_t>(m_new) + 1);
    if (st.AT != nullptr) zeros.zero(t_ptr.get(), static_cast<int64_t>(n_new) + 1);
    zeros.run("compact empty rowPtr");
    out.A.rowPtr = ptr.release();
    out.AT.rowPtr = t_ptr.release();
    return out;
  }
  const int32_t nnz = st.A->nnz, chunks = gpk_compact_chunks(nnz);
  const int32_t scanned = chunks * (st.AT != nullptr ? 2 : 1);
  const bool from_counts = chunks <= GPK_COMPACT_COUNT_CHUNKS;
  if (!from_counts)
    check(gpk_scan_lb_i32(st.cnt, st.cnt, scanned, c.lookback(gpk_lookback_tiles(scanned)), s),
          "compact chunk offsets");
  DBuf<int32_t> idx(nnz, "compact colVal"), t_idx;
  DBuf<double> val(nnz, "compact nzVal"), t_val;
  gpk_apply_gathers_args g{};
  st.a.m_new = m_new;
  st.a.out_ptr = ptr;
  st.a.out_idx = idx;
  st.a.out_val = val;
  if (st.AT != nullptr) {
    t_idx.alloc(nnz, "compact AT colVal");
    t_val.alloc(nnz, "compact AT nzVal");
    st.t.m_new = n_new;
    st.t.out_ptr = t_ptr;
    st.t.out_idx = t_idx;
    st.t.out_val = t_val;
    if (gathers != nullptr) {
      g = *gathers;
      out.gathered = true;
    }
  }
  check(gpk_compact_write(st.a, st.t, st.cnt, from_counts ? 1 : 0, g, s), "compact write");
  out.A.nnz = nnz_new;
  out.A.rowPtr = ptr.release();
  out.A.colVal = idx.release();
  out.A.nzVal = val.release();
  if (st.AT != nullptr) {
    out.AT.nnz = nnz_new;
    out.AT.rowPtr = t_ptr.release();
    out.AT.colVal = t_idx.release();
    out.AT.nzVal = t_val.release();
  }
  return out;
}

DeviceCsrMatrix compact_csr(const DeviceCsrMatrix& A, const uint8_t* keep_row, const uint8_t* keep_col) {
  Ctx& c = ctx();
  DBuf<int32_t> row_map(A.rows, "row map"), col_map(A.cols, "column map");
  DBuf<gpk_rank_word> col_rank((static_cast<int64_t>(A.cols) + 63) / 64, "column rank");
  DBuf<int32_t> chunk_row(static_cast<int64_t>(gpk_compact_chunks(A.nnz)) + 1, "chunk rows");
  const int64_t tiles = gpk_apply_maps_tiles(A.rows, A.cols);
  DBuf<int32_t> tile_counts(tiles, "map tile counts");
  int32_t* counts = c.flags();
  gpk_apply_maps_args maps{};
  maps.m = A.rows;
  maps.n = A.cols;
  maps.keep_row = keep_row;
  maps.keep_col = keep_col;
  maps.row_map = row_map;
  maps.col_map = col_map;
  maps.counts = counts;
  maps.col_rank = col_rank;
  maps.a_ptr = A.rowPtr;
  maps.a_chunk = chunk_row;
  maps.tile_counts = tile_counts;
  maps.chunk_shift = gpk_compact_shift(A.nnz);
  maps.chunks = gpk_compact_chunks(A.nnz);
  check(gpk_apply_maps(maps, c.lookback(tiles), c.stream()), "keep maps");
  CompactStart st = compact_start(A, row_map, col_rank, chunk_row, counts + 4, nullptr, nullptr, nullptr, nullptr);
  int32_t h[5];
  std::memcpy(h, c.read_flags(5), sizeof(h));
  return compact_finish(st, h[0], h[1], h[4], nullptr).A;
}

// Stable transpose: by buckets of columns, or by an LSD radix sort of the column indices (entries already in
// row-major order, so every AT row comes out sorted by row index) carrying
// the entry positions; the row pointers come from the sorted keys (no
// per-column atomic counters), then one gather of packed (row, value) pairs
// writes rows and values.
DeviceCsrMatrix transpose_csr(const DeviceCsrMatrix& A) {
  Ctx& c = ctx();
  hipStream_t s = c.stream();
  DeviceCsrMatrix T;
  T.rows = A.cols;
  T.cols = A.rows;
  T.nnz = A.nnz;
  DBuf<int32_t> ptr(static_cast<int64_t>(A.cols) + 1, "transpose rowPtr");
  if (A.nnz == 0) {
    check(gpk_col_bounds(nullptr, 0, A.cols, ptr, s), "transpose rowPtr");
    T.rowPtr = ptr.release();
    return T;
  }
  const int32_t nnz = A.nnz;
  // Large matrices by buckets of columns.
  int32_t low = 0;
  const int32_t buckets = gpk_transpose_buckets(A.cols, nnz, &low);
  if (buckets > 0) {
    DBuf<int32_t> scratch(gpk_transpose_buckets_scratch_ints(buckets, nnz));
    check(gpk_transpose_buckets_count(A.colVal, nnz, low, buckets, scratch, s), "transpose bucket sizes");
    DBuf<gpk_row_val> rec(nnz, "transpose rows and values");
    DBuf<int32_t> idx(nnz, "transpose colVal");
    DBuf<double> val(nnz, "transpose nzVal");
    check(gpk_transpose_buckets_move(A.rowPtr, A.colVal, A.nzVal, A.rows, A.cols, nnz, low, buckets, scratch, rec, ptr,
                                     idx, val, s),
          "transpose buckets");
    T.rowPtr = ptr.release();
    T.colVal = idx.release();
    T.nzVal = val.release();
    return T;
  }
  int32_t bits = 1;
  while (bits < 31 && (int64_t{1} << bits) < A.cols) ++bits;
  DBuf<uint32_t> ka(nnz), kb(nnz);
  DBuf<int32_t> va(nnz), vb(nnz);
  int32_t in_b = 0;
  {
    DBuf<int32_t> scratch(gpk_radix_scratch_ints(nnz));
    check(gpk_transpose_sort(A.colVal, nnz, bits, ka, va, kb, vb, scratch, &in_b, s), "transpose sort");
  }
  const uint32_t* keys = in_b ? kb.get() : ka.get();
  const int32_t* perm = in_b ? vb.get() : va.get();
  check(gpk_col_bounds(keys, nnz, A.cols, ptr, s), "transpose rowPtr");
  DBuf<gpk_row_val> rv(nnz, "transpose rows and values");
  check(gpk_expand_rows(A.rowPtr, A.nzVal, A.rows, rv, s), "expand rows");
  DBuf<int32_t> idx(nnz, "transpose colVal");
  DBuf<double> val(nnz, "transpose nzVal");
  check(gpk_transpose_gather(perm, rv, nnz, idx, val, s), "transpose gather");
  T.rowPtr = ptr.release();
  T.colVal = idx.release();
  T.nzVal = val.release();
  return T;
}

void sort_rows_if_needed(const DeviceCsrMatrix& A) {
  if (A.rows <= 0 || A.nnz <= 1) return;
  Ctx& c = ctx();
  int32_t* f = c.flags();
  check(gpk_rows_unsorted(A.rowPtr, A.colVal, A.rows, f, c.stream()), "rows unsorted check");
  if (c.read_flags(1)[0] == 0) return;
  check(gpk_sort_rows_in_place(A.rowPtr, A.colVal, A.nzVal, A.rows, c.stream()), "sort rows");
}

void check_lp_arrays(const presolve::LPInfoGpu& lp, const char* who) {
  if (lp.A.rows <= 0 && lp.AT.rows <= 0) return;
  Ctx& c = ctx();
  int32_t* f = c.flags();
  const int32_t chunks = gpk_csr_check_chunks(lp.A.nnz);
  DBuf<int32_t> chunk_row(static_cast<int64_t>(chunks) + gpk_csr_check_chunks(lp.AT.nnz));
  const auto side = [](const DeviceCsrMatrix& M, int32_t* chunk_rows, int32_t* flags) {
    return gpk_csr_check_side{M.rowPtr, M.colVal, M.rows, M.cols, M.nnz, 0, chunk_rows, flags};
  };
  check(gpk_csr_check(side(lp.A, chunk_row.get(), f), side(lp.AT, chunk_row.get() + chunks, f + 4), c.stream()),
        "check A and AT");
  int32_t h[8];
  std::memcpy(h, c.read_flags(8), sizeof(h));
  const bool a_again = h[0] == 0 && h[2] == 0 && h[3] != 0, at_again = h[4] == 0 && h[6] == 0 && h[7] != 0;
  if (a_again || at_again) {  // unsorted rows: look for columns repeated at a distance
    f = c.flags();
    if (a_again) check(gpk_csr_check_rows(lp.A.rowPtr, lp.A.colVal, lp.A.rows, lp.A.cols, lp.A.nnz, f, c.stream()),
                       "check A rows");
    if (at_again)
      check(gpk_csr_check_rows(lp.AT.rowPtr, lp.AT.colVal, lp.AT.rows, lp.AT.cols, lp.AT.nnz, f + 4, c.stream()),
            "check AT rows");
    const int32_t* g = c.read_flags(8);
    for (int k = 0; k < 8; ++k) h[k] |= g[k];
  }
  static const char* const what[3] = {"row pointers are not monotone from 0 to nnz",
                                      "a column index is outside [0, cols)", "a row repeats a column index"};
  for (int m = 0; m < 2; ++m)
    for (int k = 0; k < 3; ++k)
      if (h[4 * m + k])
        throw InputError(std::string(who) + ": " + (m == 0 ? "A" : "AT") + ": " + what[k]);
}

void append_record(PostsolveTape& tape, PostsolveReductionType type, const int32_t* idx, size_t ni,
                   const double* vals, size_t nv, PostsolveDualMode mode) {
  tape.types.push_back(static_cast<int32_t>(type));
  tape.indices.insert(tape.indices.end(), idx, idx + ni);
  tape.vals.insert(tape.vals.end(), vals, vals + nv);
  tape.index_starts.push_back(static_cast<int32_t>(tape.indices.size()));
  tape.value_starts.push_back(static_cast<int32_t>(tape.vals.size()));
  tape.dual_modes.push_back(static_cast<uint8_t>(mode));
}

double fixed_col_tape(PostsolveTape* tape, const uint8_t* fixed_mask, const uint8_t* excluded,
                      const double* fixed_val, const uint8_t* keep_row, const double* cvec, const DeviceCsrMatrix& AT,
                      int32_t n) {
  if (n <= 0) return 0.0;
  Ctx& c = ctx();
  hipStream_t s = c.stream();
  const gpk_csr at = csr_view(AT);
  DBuf<uint8_t> sel(n);
  DBuf<int32_t> sel_prefix(static_cast<int64_t>(n) + 1), nnz_prefix(static_cast<int64_t>(n) + 1);
  check(gpk_fixed_col_counts(at, fixed_mask, excluded, keep_row, sel, nnz_prefix, s), "fixed col counts");
  scan_mask_launch(sel, n, sel_prefix);
  scan_counts_launch(nnz_prefix, n, nnz_prefix);
  int32_t records = 0, active = 0;  // both totals in one wait
  c.begin_copy_group();
  c.download(&records, sel_prefix.get() + n, sizeof(int32_t), "fixed col records");
  c.download(&active, nnz_prefix.get() + n, sizeof(int32_t), "fixed col entries");
  c.sync("fixed col counts");
  if (records == 0) return 0.0;
  DBuf<int32_t> cols(records), rows(active), rstart(records);
  DBuf<double> v(records), cc(records), coef(active);
  check(gpk_fixed_col_pack(at, sel, sel_prefix, nnz_prefix, fixed_val, cvec, keep_row, cols, v, cc, rstart, rows, coef,
                           s),
        "fixed col pack");
  // Everything the objective and the tape need, in one wait.
  std::vector<double> hv, hc, hcoef;
  std::vector<int32_t> hcol, hrow, starts;
  c.begin_copy_group();
  c.to_host_async(hv, v.get(), records, "fixed col values");
  c.to_host_async(hc, cc.get(), records, "fixed col costs");
  if (tape) {
    c.to_host_async(hcol, cols.get(), records, "fixed col ids");
    c.to_host_async(hrow, rows.get(), active, "fixed col rows");
    c.to_host_async(hcoef, coef.get(), active, "fixed col coefs");
    c.to_host_async(starts, rstart.get(), records, "fixed col starts");
  }
  c.sync("fixed col tape");
  long double obj = 0.0L;
  for (int32_t r = 0; r < records; ++r)
    obj += static_cast<long double>(hc[r]) * static_cast<long double>(hv[r]);
  if (tape) {
    starts.push_back(active);
    std::vector<int32_t> idx;
    std::vector<double> vals;
    for (int32_t r = 0; r < records; ++r) {
      idx.assign(1, hcol[r]);
      vals.assign({hv[r], hc[r]});
      for (int32_t q = starts[r]; q < starts[r + 1]; ++q) {
        idx.push_back(hrow[q]);
        vals.push_back(hcoef[q]);
      }
      append_record(*tape, PostsolveReductionType::FixedCol, idx.data(), idx.size(), vals.data(), vals.size(),
                    PostsolveDualMode::Minimal);
    }
  }
  return static_cast<double>(obj);
}

}  // namespace gpu_presolver::amd
