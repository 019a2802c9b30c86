// Host operands of a call: copied through pinned memory by several threads, in one transfer per few megabytes.
//
// A call on host arrays is as fast as its operands cross the bus.  Copies from and to pageable memory cost 33 us for
// 64 KB and 110 us for 256 KB and run at 29 GB/s (to the device) and 17 GB/s (back) for megabytes; the bus itself does
// 55 GB/s from pinned memory, and one thread fills pinned memory at 15 to 30 GB/s, four at 100.  So all the operands of
// a call lie in one piece of device memory, blocks of 256 KB of them are copied into pinned memory laid out the same
// way by the caller's thread and (from a megabyte on) three helpers, and whatever is filled in order is on its way
// while the rest is being filled.  The structure of a CSR matrix is checked and counted by the same pass (on the data
// as it is staged), which is what a plan needs to know of it: no kernel and no wait between the copies and the product.
//
// A result that a kernel reads and writes once per element stays in pinned memory where it is small: the kernel reaches
// it over the bus, both ways at once, and nothing is copied.
//
// A product on host arrays, fp64 7-point grids: 11^3 222 -> 26 us, 32^3 317 -> 130 us, 64^3 1.56 -> 0.70 ms,
// 128^3 10.5 -> 5.1 ms.  Bound by the bus (55 GB/s) from 32^3 on, by four launches and a wait below.
//
// Kept between calls until the library shuts down (lapis_hip_finalize): up to 4 arenas, each with two streams and pinned
// memory of up to 2 x 16 MB and 4 MB, together with at most 256 MB of memory on a device; and the helper threads, which
// sleep.  A call beyond that takes its memory and gives it back (hipMalloc 31 us, hipFree 236 us for 256 MB, where the
// call itself takes 5 ms; 1 GB: 31 and 239).  Other allocators of the process cannot ask for what is kept; a call that
// finds the device full gives back what the other arenas hold.
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>

#include "common.hpp"
#include "staging.hpp"

namespace lapis {

struct StagingArena {
  int device = -1;
  hipStream_t stream = nullptr, second = nullptr;
  char *memory = nullptr;
  size_t bytes = 0;
  char *pinned[2] = {nullptr, nullptr};
  size_t pinned_bytes = 0;  // of each half
  char *direct = nullptr;  // pinned memory that kernels work on
  size_t direct_bytes = 0;
  hipEvent_t half_done[2][2] = {};  // of each half, on each stream
  hipEvent_t joined = nullptr;
  hipEvent_t landed[16] = {};
};

namespace {
__global__ __launch_bounds__(256) void staging_copy_kernel(int n, const v4i *__restrict__ from, v4i *__restrict__ to) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) to[i] = from[i];
}

constexpr size_t kHalf = (size_t)16 << 20;      // pinned memory of a round
constexpr size_t kBlock = (size_t)256 << 10;    // what a thread copies at a time
constexpr size_t kAlign = 4096;                 // operands start here: blocks are whole groups of 1024 coordinates
constexpr size_t kAlone = (size_t)1 << 20;      // up to here the caller's thread copies alone
constexpr size_t kByKernel = (size_t)2 << 20;   // uploads up to here are one kernel's work
constexpr size_t kDirect = (size_t)4 << 20;     // direct operands up to here stay in pinned memory
constexpr size_t kKeptMemory = (size_t)256 << 20;  // device memory of all arenas at rest on a device
constexpr int kKeptArenas = 4;
constexpr int kHelpers = 3;

std::mutex g_arena_mutex;
std::vector<StagingArena *> g_arenas;

void free_arena(StagingArena *a) {
  if (a->memory) (void)hipFree(a->memory);
  for (char *p : a->pinned)
    if (p) (void)hipHostFree(p);
  if (a->direct) (void)hipHostFree(a->direct);
  for (auto &pair : a->half_done)
    for (hipEvent_t e : pair)
      if (e) (void)hipEventDestroy(e);
  if (a->joined) (void)hipEventDestroy(a->joined);
  for (hipEvent_t e : a->landed)
    if (e) (void)hipEventDestroy(e);
  if (a->stream) (void)hipStreamDestroy(a->stream);
  if (a->second) (void)hipStreamDestroy(a->second);
  delete a;
}

hipError_t prepare_arena(StagingArena *a, size_t bytes, size_t half, size_t direct) {
  hipError_t e = hipSuccess;
  if (!a->stream) {
    e = hipStreamCreateWithFlags(&a->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&a->second, hipStreamNonBlocking);
    for (auto &pair : a->half_done)
      for (hipEvent_t &ev : pair)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&a->joined, hipEventDisableTiming);
    for (hipEvent_t &ev : a->landed)
      if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  }
  if (e == hipSuccess && a->bytes < bytes) {
    if (a->memory) (void)hipFree(a->memory);
    a->memory = nullptr;
    a->bytes = 0;
    e = hipMalloc(&a->memory, bytes);
    if (e == hipSuccess) a->bytes = bytes;
  }
  if (e == hipSuccess && a->pinned_bytes < half) {
    for (char *&p : a->pinned) {
      if (p) (void)hipHostFree(p);
      p = nullptr;
    }
    a->pinned_bytes = 0;
    for (char *&p : a->pinned)
      if (e == hipSuccess) e = hipHostMalloc(&p, half, hipHostMallocDefault);
    if (e == hipSuccess) a->pinned_bytes = half;
  }
  if (e == hipSuccess && a->direct_bytes < direct) {
    if (a->direct) (void)hipHostFree(a->direct);
    a->direct = nullptr;
    a->direct_bytes = 0;
    size_t want = kBlock;
    while (want < direct) want *= 2;
    e = hipHostMalloc(&a->direct, want, hipHostMallocDefault);
    if (e == hipSuccess) a->direct_bytes = want;
  }
  return e;
}

hipError_t take_arena(StagingArena **out, size_t bytes, size_t half, size_t direct) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  StagingArena *a = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    for (size_t i = 0; i < g_arenas.size(); ++i)
      if (g_arenas[i]->device == dev && (!a || g_arenas[i]->bytes > a->bytes)) a = g_arenas[i];
    if (a) g_arenas.erase(std::find(g_arenas.begin(), g_arenas.end(), a));
  }
  if (!a) {
    a = new StagingArena();
    a->device = dev;
  }
  // sizes with room to grow, so that calls of varying size settle on one piece of memory
  size_t want = kBlock;
  while (want < bytes && want < kKeptMemory) want *= 2;
  e = prepare_arena(a, std::max(want, bytes), half, direct);
  if (e == hipErrorOutOfMemory) {  // what other arenas hold may be what is missing
    (void)hipGetLastError();
    {
      std::lock_guard<std::mutex> lock(g_arena_mutex);
      for (StagingArena *other : g_arenas) free_arena(other);
      g_arenas.clear();
    }
    e = prepare_arena(a, bytes, half, direct);
  }
  if (e != hipSuccess) {
    free_arena(a);
    return e;
  }
  *out = a;
  return hipSuccess;
}

void give_arena(StagingArena *a) {
  char *surplus = nullptr;
  bool kept = false;
  {
    std::lock_guard<std::mutex> lock(g_arena_mutex);
    size_t bytes = a->bytes;
    for (const StagingArena *other : g_arenas)
      if (other->device == a->device) bytes += other->bytes;
    kept = (int)g_arenas.size() < kKeptArenas;
    if (kept) {
      if (bytes > kKeptMemory) {
        surplus = a->memory;
        a->memory = nullptr;
        a->bytes = 0;
      }
      g_arenas.push_back(a);
    }
  }
  if (surplus) (void)hipFree(surplus);
  if (!kept) free_arena(a);
}

// ---- copying passes -----------------------------------------------------------------------------------------

// Copies of whole loops for AVX2 machines: the plain ones have no 32-bit minimum and maximum to vectorise with.
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#define LAPIS_AVX2 __attribute__((target("avx2")))
bool has_avx2() {
  static const bool yes = __builtin_cpu_supports("avx2");
  return yes;
}
#else
#define LAPIS_AVX2
bool has_avx2() { return false; }
#endif

#define LAPIS_COORDINATE_LOOP                                        \
  int mn = INT32_MAX, mx = INT32_MIN;                                \
  for (int i = 0; i < n; ++i) {                                      \
    const int32_t v = src[i];                                        \
    dst[i] = v;                                                      \
    mn = std::min(mn, v);                                            \
    mx = std::max(mx, v);                                            \
  }                                                                  \
  *lo = mn;                                                          \
  *hi = mx;
void copy_coordinates(const int32_t *src, int32_t *dst, int n, int *lo, int *hi) { LAPIS_COORDINATE_LOOP }
LAPIS_AVX2 void copy_coordinates_avx2(const int32_t *src, int32_t *dst, int n, int *lo, int *hi) { LAPIS_COORDINATE_LOOP }

// dst[0..n) = src[0..n); lengths src[i + 1] - src[i] of the first n rows (src has an element more)
struct Lengths {
  int mn, mx, empty;
  double squares;
};
#define LAPIS_POSITION_LOOP                                          \
  int mn = INT32_MAX, mx = INT32_MIN, empty = 0;                     \
  double squares = 0.0;                                              \
  for (int i = 0; i < n; ++i) {                                      \
    const int32_t v = src[i];                                        \
    const int32_t len = (int32_t)((uint32_t)src[i + 1] - (uint32_t)v); \
    dst[i] = v;                                                      \
    mn = std::min(mn, len);                                          \
    mx = std::max(mx, len);                                          \
    empty += len == 0;                                               \
  }                                                                  \
  for (int i = 0; i < n; ++i) {                                      \
    const double len = (double)(int32_t)((uint32_t)src[i + 1] - (uint32_t)src[i]); \
    squares += len * len;                                            \
  }                                                                  \
  *out = {mn, mx, empty, squares};
void copy_positions(const int32_t *src, int32_t *dst, int n, Lengths *out) { LAPIS_POSITION_LOOP }
LAPIS_AVX2 void copy_positions_avx2(const int32_t *src, int32_t *dst, int n, Lengths *out) { LAPIS_POSITION_LOOP }

std::mutex g_counts_mutex;
}  // namespace

// ---- threads ------------------------------------------------------------------------------------------------

// Blocks [0, limit) may be copied; the limit moves while they are.
struct BlockQueue {
  HostOperands *owner = nullptr;
  bool to_host = false;
  std::vector<HostOperands::Block> *blocks = nullptr;
  std::atomic<int> next{0}, limit{0};
  std::atomic<bool> closed{false};
  std::unique_ptr<std::atomic<unsigned char>[]> done;
};

struct StagingHelpers {
  std::mutex mutex;
  std::condition_variable wake, left;
  std::vector<std::thread> threads;
  BlockQueue *queue = nullptr;
  unsigned long long serial = 0;
  int inside = 0;
  bool stop = false;

  static bool copy_one(BlockQueue &q) {
    int i = q.next.load(std::memory_order_relaxed);
    while (i < q.limit.load(std::memory_order_acquire)) {
      if (!q.next.compare_exchange_weak(i, i + 1, std::memory_order_relaxed)) continue;
      q.owner->copy_block((*q.blocks)[(size_t)i], q.to_host);
      q.done[(size_t)i].store(1, std::memory_order_release);
      return true;
    }
    return false;
  }

  void run() {
    unsigned long long seen = 0;
    std::unique_lock<std::mutex> lock(mutex);
    for (;;) {
      wake.wait(lock, [&] { return stop || (queue && serial != seen); });
      if (stop) return;
      seen = serial;
      BlockQueue *q = queue;
      ++inside;
      lock.unlock();
      while (!q->closed.load(std::memory_order_acquire))
        if (!copy_one(*q)) __builtin_ia32_pause();
      lock.lock();
      if (--inside == 0) left.notify_all();
    }
  }

  // false: another call has them, or there are none
  bool open(BlockQueue *q) {
    {
      std::lock_guard<std::mutex> lock(mutex);
      if (queue || inside) return false;
      if (threads.empty()) {
        stop = false;
        const char *most = getenv("LAPIS_HIP_STAGING_HELPERS");
        const int n = std::min<int>(most ? atoi(most) : kHelpers, (int)std::thread::hardware_concurrency() / 2);
        try {
          for (int i = 0; i < n; ++i) threads.emplace_back([this] { run(); });
        } catch (const std::exception &) {
          // a process at its limit of threads copies with those it got
        }
        if (threads.empty()) return false;
      }
      queue = q;
      ++serial;
    }
    wake.notify_all();
    return true;
  }
  void close(BlockQueue *q) {
    q->closed.store(true, std::memory_order_release);
    std::unique_lock<std::mutex> lock(mutex);
    queue = nullptr;
    left.wait(lock, [&] { return inside == 0; });
  }
  void shut_down() {
    std::vector<std::thread> gone;
    {
      std::lock_guard<std::mutex> lock(mutex);
      stop = true;
      gone.swap(threads);
    }
    wake.notify_all();
    for (std::thread &t : gone) t.join();
  }
};

namespace {
// never destroyed: a process may end with the threads asleep
StagingHelpers &helpers() {
  static StagingHelpers *h = new StagingHelpers();
  return *h;
}

// Has the helpers work on a queue for as long as it lives.
struct Crew {
  BlockQueue queue;
  bool open = false;
  Crew(HostOperands *owner, bool to_host, std::vector<HostOperands::Block> *blocks, size_t bytes);
  ~Crew() {
    if (open) helpers().close(&queue);
  }
};
Crew::Crew(HostOperands *owner, bool to_host, std::vector<HostOperands::Block> *blocks, size_t bytes) {
  queue.owner = owner;
  queue.to_host = to_host;
  queue.blocks = blocks;
  queue.done.reset(new std::atomic<unsigned char>[blocks->size()]);
  for (size_t i = 0; i < blocks->size(); ++i) queue.done[i].store(0, std::memory_order_relaxed);
  open = bytes > kAlone && helpers().open(&queue);
}
}  // namespace

void HostOperands::copy_block(const Block &b, bool to_host) {
  if (to_host) {
    memcpy(b.host, b.staged, b.bytes);
    return;
  }
  const Operand &o = operands_[(size_t)b.operand];
  if (o.kind == kPlain || o.kind == kDirectly) {
    memcpy(b.staged, b.host, b.bytes);
    return;
  }
  const int32_t *src = reinterpret_cast<const int32_t *>(b.host);
  int32_t *dst = reinterpret_cast<int32_t *>(b.staged);
  const int n = (int)(b.bytes / 4);
  if (o.kind == kCoordinates) {
    unsigned long long span = 0;
    int lo = INT32_MAX, hi = INT32_MIN;
    for (int i = 0; i < n; i += 1024) {
      int l, h;
      (has_avx2() ? copy_coordinates_avx2 : copy_coordinates)(src + i, dst + i, std::min(1024, n - i), &l, &h);
      span += (unsigned long long)((long long)h - (long long)l);
      lo = std::min(lo, l);
      hi = std::max(hi, h);
    }
    std::lock_guard<std::mutex> lock(g_counts_mutex);
    counts_.span_sum += span;
    if (lo < 0 || hi >= ncols_) counts_.bad |= 2;
    return;
  }
  const int64_t first = (int64_t)(b.at / 4);
  const int rows = (int)std::min<int64_t>(n, nrows_ - first);  // the last position ends the last row
  Lengths len{INT32_MAX, 0, 0, 0.0};
  if (rows > 0) (has_avx2() ? copy_positions_avx2 : copy_positions)(src, dst, rows, &len);
  if (rows < n) dst[rows] = src[rows];
  std::lock_guard<std::mutex> lock(g_counts_mutex);
  if (len.mn < 0) counts_.bad |= 1;
  counts_.min_len = std::min(counts_.min_len, len.mn);
  counts_.max_len = std::max(counts_.max_len, len.mx);
  counts_.empty_rows += (unsigned long long)len.empty;
  counts_.sum_sq += len.squares;
}

HostOperands::~HostOperands() {
  if (!arena_) return;
  if (!idle_) {
    (void)hipStreamSynchronize(arena_->second);
    (void)hipStreamSynchronize(primary_);
  }
  give_arena(arena_);
}

int HostOperands::add(const void *host, size_t bytes) {
  operands_.push_back({static_cast<const char *>(host), bytes, 0, host ? kPlain : kDeviceOnly});
  return (int)operands_.size() - 1;
}
int HostOperands::add_direct(const void *host, size_t bytes) {
  operands_.push_back({static_cast<const char *>(host), bytes, 0, bytes <= kDirect ? kDirectly : kPlain});
  return (int)operands_.size() - 1;
}
int HostOperands::add_positions(const int32_t *host, int64_t nrows, int64_t nnz) {
  nrows_ = nrows;
  nnz_ = nnz;
  operands_.push_back({reinterpret_cast<const char *>(host), sizeof(int32_t) * ((size_t)nrows + 1), 0, kPositions});
  return (int)operands_.size() - 1;
}
int HostOperands::add_coordinates(const int32_t *host, int64_t nnz, int64_t ncols) {
  ncols_ = ncols;
  operands_.push_back({reinterpret_cast<const char *>(host), sizeof(int32_t) * (size_t)nnz, 0, kCoordinates});
  return (int)operands_.size() - 1;
}
void *HostOperands::device(int index) const {
  const Operand &o = operands_[(size_t)index];
  return !o.bytes ? nullptr : o.kind == kDirectly ? arena_->direct + o.at : arena_->memory + o.at;
}

int HostOperands::upload() {
  // values first: they are copied fastest, and the bus starts with them; what is uploaded lies together
  size_t upload_bytes = 0, direct_bytes = 0;
  for (const Kind kind : {kPlain, kCoordinates, kPositions, kDeviceOnly, kDirectly}) {
    size_t &end = kind == kDirectly ? direct_bytes : bytes_;
    for (Operand &o : operands_) {
      if (o.kind != kind) continue;
      o.at = end;
      end += (o.bytes + kAlign - 1) / kAlign * kAlign;
    }
    if (kind == kPositions) upload_bytes = bytes_;
  }
  if (bytes_ == 0) bytes_ = kAlign;
  size_t half = kBlock;
  while (half < kHalf && half < bytes_) half *= 2;
  LAPIS_HIP_TRY(take_arena(&arena_, bytes_, half, direct_bytes));
  half = arena_->pinned_bytes;
  if (own_stream_) primary_ = arena_->stream;
  counts_ = CsrCounts{};
  counts_.min_len = INT32_MAX;

  std::vector<Block> blocks;
  std::vector<size_t> rounds;  // one past the last block of each round
  for (const Kind kind : {kPlain, kCoordinates, kPositions, kDirectly})
    for (size_t i = 0; i < operands_.size(); ++i) {
      const Operand &o = operands_[i];
      if (o.kind != kind) continue;
      for (size_t done = 0; done < o.bytes;) {
        const size_t at = o.at + done, round = at / half;
        size_t bytes = std::min(kBlock, o.bytes - done);
        char *staged = arena_->direct + at;
        if (kind != kDirectly) {
          bytes = std::min(bytes, (round + 1) * half - at);
          staged = arena_->pinned[round & 1] + (at - round * half);
          rounds.resize(round + 1, blocks.size());
          rounds[round] = blocks.size() + 1;
        }
        blocks.push_back({staged, const_cast<char *>(o.host) + done, bytes, done, (int)i, at + bytes});
        done += bytes;
      }
    }
  Crew crew(this, false, &blocks, upload_bytes);
  BlockQueue &q = crew.queue;
  idle_ = false;
  // Up to 2 MB are brought over by one kernel, for which the next kernel does not wait as it does for a copy engine
  // (0.14 MB: 26 us a call against 31).  More goes in pieces of 4 MB after half a megabyte that gets the bus started, on
  // two streams in turn, so that a transfer is set up while another runs (27 MB: 0.70 ms a call against 0.85).
  const bool by_kernel = upload_bytes <= kByKernel;
  const hipStream_t streams[2] = {primary_, arena_->second};
  size_t filled = 0, sent = 0, transfers = 0;
  for (size_t r = 0; r < rounds.size(); ++r) {
    if (r >= 2)
      for (hipEvent_t e : arena_->half_done[r & 1]) LAPIS_HIP_TRY(hipEventSynchronize(e));
    q.limit.store((int)rounds[r], std::memory_order_release);
    sent = std::max(sent, r * half);
    while (filled < rounds[r]) {
      while (filled < rounds[r] && q.done[filled].load(std::memory_order_acquire)) ++filled;
      const size_t upto = filled ? blocks[filled - 1].end : 0;
      const size_t worth = by_kernel ? upload_bytes : sent == 0 ? (size_t)512 << 10 : (size_t)4 << 20;
      if (upto > sent && (filled == rounds[r] || upto - sent >= worth)) {
        if (by_kernel) {
          const int n = (int)((upto + 15) / 16);
          hipLaunchKernelGGL(staging_copy_kernel, dim3((unsigned)std::min(256, (n + 255) / 256)), dim3(256), 0, primary_,
                             n, reinterpret_cast<const v4i *>(arena_->pinned[0]), reinterpret_cast<v4i *>(arena_->memory));
          LAPIS_LAUNCH_CHECK();
        } else {
          LAPIS_HIP_TRY(hipMemcpyAsync(arena_->memory + sent, arena_->pinned[r & 1] + (sent - r * half), upto - sent,
                                       hipMemcpyHostToDevice, streams[transfers++ & 1]));
        }
        sent = upto;
      } else if (!StagingHelpers::copy_one(q)) {
        __builtin_ia32_pause();
      }
    }
    if (rounds.size() > 1)
      for (int s = 0; s < 2; ++s) LAPIS_HIP_TRY(hipEventRecord(arena_->half_done[r & 1][s], streams[s]));
  }
  if (transfers > 1) {
    LAPIS_HIP_TRY(hipEventRecord(arena_->joined, arena_->second));
    LAPIS_HIP_TRY(hipStreamWaitEvent(primary_, arena_->joined, 0));
  }
  q.limit.store((int)blocks.size(), std::memory_order_release);
  while (filled < blocks.size()) {
    if (!StagingHelpers::copy_one(q)) __builtin_ia32_pause();
    while (filled < blocks.size() && q.done[filled].load(std::memory_order_acquire)) ++filled;
  }
  return LAPIS_HIP_OK;
}

int HostOperands::create_plan(int positions, int coordinates, int value_bytes, lapis_hip_csr_plan **plan) {
  const int32_t *host = reinterpret_cast<const int32_t *>(operands_[(size_t)positions].host);
  CsrCounts counts = counts_;
  if (nrows_ == 0) counts.min_len = 0;
  return create_counted_plan(plan, nrows_, ncols_, nnz_, at<int32_t>(positions), at<int32_t>(coordinates), value_bytes, counts,
                             host[0], host[nrows_], primary_);
}

int HostOperands::synchronize() {
  LAPIS_HIP_TRY(hipStreamSynchronize(primary_));
  idle_ = true;
  return LAPIS_HIP_OK;
}

int HostOperands::download(int index, void *host) {
  const Operand &o = operands_[(size_t)index];
  if (o.bytes == 0) return LAPIS_HIP_OK;
  if (o.kind == kDirectly) {
    const int rc = synchronize();
    if (rc != LAPIS_HIP_OK) return rc;
    std::vector<Block> blocks;
    for (size_t done = 0; done < o.bytes; done += kBlock)
      blocks.push_back({arena_->direct + o.at + done, static_cast<char *>(host) + done, std::min(kBlock, o.bytes - done), done, index, 0});
    Crew crew(this, true, &blocks, o.bytes);
    crew.queue.limit.store((int)blocks.size(), std::memory_order_release);
    for (size_t i = 0; i < blocks.size();)
      if (crew.queue.done[i].load(std::memory_order_acquire))
        ++i;
      else if (!StagingHelpers::copy_one(crew.queue))
        __builtin_ia32_pause();
    return LAPIS_HIP_OK;
  }
  return download(arena_->memory + o.at, o.bytes, host);
}

int HostOperands::download(const void *from, size_t total, void *host) {
  if (total == 0) return LAPIS_HIP_OK;
  const char *source = static_cast<const char *>(from);
  const size_t half = arena_->pinned_bytes;
  if (total <= half && total <= kAlone / 2) {
    LAPIS_HIP_TRY(hipMemcpyAsync(arena_->pinned[0], source, total, hipMemcpyDeviceToHost, primary_));
    const int rc = synchronize();
    if (rc == LAPIS_HIP_OK) memcpy(host, arena_->pinned[0], total);
    return rc;
  }
  // pieces of up to 2 MB through the slots of both halves, copied out as they land
  const size_t piece = std::min(half, std::max(kBlock, std::min((size_t)2 << 20, (total / 4 + kBlock - 1) / kBlock * kBlock)));
  const size_t per_half = half / piece, slots = std::min<size_t>(16, 2 * per_half);
  const size_t pieces = (total + piece - 1) / piece;
  auto slot_of = [&](size_t p) {
    const size_t s = p % slots;
    return arena_->pinned[s / per_half] + (s % per_half) * piece;
  };
  std::vector<Block> blocks;
  std::vector<size_t> last(pieces);  // one past the last block of each piece
  for (size_t p = 0; p < pieces; ++p) {
    const size_t at = p * piece, bytes = std::min(piece, total - at);
    for (size_t done = 0; done < bytes; done += kBlock)
      blocks.push_back({slot_of(p) + done, static_cast<char *>(host) + at + done, std::min(kBlock, bytes - done), at + done, 0, 0});
    last[p] = blocks.size();
  }
  Crew crew(this, true, &blocks, total);
  BlockQueue &q = crew.queue;
  size_t queued = 0, landed = 0, emptied = 0, block = 0;
  idle_ = false;
  while (emptied < pieces) {
    while (queued < pieces && queued < emptied + slots) {
      const size_t at = queued * piece;
      LAPIS_HIP_TRY(hipMemcpyAsync(slot_of(queued), source + at, std::min(piece, total - at),
                                   hipMemcpyDeviceToHost, primary_));
      LAPIS_HIP_TRY(hipEventRecord(arena_->landed[queued % slots], primary_));
      ++queued;
    }
    if (landed < queued) {
      const hipError_t e = hipEventQuery(arena_->landed[landed % slots]);
      if (e == hipSuccess)
        q.limit.store((int)last[landed++], std::memory_order_release);
      else if (e == hipErrorNotReady)
        (void)hipGetLastError();
      else
        LAPIS_HIP_TRY(e);
    }
    if (!StagingHelpers::copy_one(q)) __builtin_ia32_pause();
    while (emptied < landed) {
      while (block < last[emptied] && q.done[block].load(std::memory_order_acquire)) ++block;
      if (block < last[emptied]) break;
      ++emptied;
    }
  }
  idle_ = true;
  return LAPIS_HIP_OK;
}

void release_staging() {
  helpers().shut_down();
  std::lock_guard<std::mutex> lock(g_arena_mutex);
  for (StagingArena *a : g_arenas) free_arena(a);
  g_arenas.clear();
}

}  // namespace lapis
