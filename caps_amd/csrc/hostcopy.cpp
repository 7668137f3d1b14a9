#include "hostcopy.h"

#include <emmintrin.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace caps {

namespace {

// 2 MiB per DMA: 1 MiB chunks lose 15 to 30 % to the gaps between copies
constexpr size_t CHUNK = (size_t)2 << 20;
// unit of the threads' work: the last chunk's memcpy, which nothing hides, is
// shared
constexpr int PIECES = 4;
constexpr size_t PIECE = CHUNK / PIECES;
// with the calling thread: more than four gain nothing (memory bound)
constexpr int MAX_HELPERS = 3;
constexpr size_t BYTES_PER_HELPER = 2 * CHUNK;
// What a helper reads stays in its core's caches too: a caller that refills
// operands of 10 or 26 MB after the call then takes 8 and 18 ms, 2.4 and 6.6 if
// it read them itself, which up to there is as quick (n = 800 550 and 564 us, n =
// 1280 1098 and 1041).  From 32 MiB on little of them is left in those caches
// (36 MB: 11.5 and 10.2 ms) and helpers pay (n = 1536 2042 -> 1379 us, n = 2048
// 3475 -> 2634).
constexpr size_t UP_HELPER_BYTES = (size_t)32 << 20;
// smaller copies are the runtime's: it is as quick or quicker below (a multiply
// of host arrays of 0.5 MiB 114 us against 137, of 1.25 MiB 229 against 205)
constexpr size_t DIRECT_BYTES = (size_t)1 << 20;

// memcpy past the caches: what a helper writes would else stay in its core's
// caches, and the caller's next pass over the array would fetch it from there
void stream_copy(char *dst, const char *src, size_t n) {
  const size_t head = std::min(n, (size_t)(-reinterpret_cast<uintptr_t>(dst) & 15));
  memcpy(dst, src, head);
  dst += head;
  src += head;
  n -= head;
  for (; n >= 64; n -= 64, dst += 64, src += 64) {
    _mm_prefetch(src + 512, _MM_HINT_NTA);
    const __m128i a = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src));
    const __m128i b = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + 16));
    const __m128i c = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + 32));
    const __m128i d = _mm_loadu_si128(reinterpret_cast<const __m128i *>(src + 48));
    _mm_stream_si128(reinterpret_cast<__m128i *>(dst), a);
    _mm_stream_si128(reinterpret_cast<__m128i *>(dst + 16), b);
    _mm_stream_si128(reinterpret_cast<__m128i *>(dst + 32), c);
    _mm_stream_si128(reinterpret_cast<__m128i *>(dst + 48), d);
  }
  memcpy(dst, src, n);
  _mm_sfence();  // the stores are visible before the piece counts as done
}

struct Chunk {
  char *dev, *host;
  size_t bytes;
};

// memory that HIP does not know (pinned and device memory: the runtime's copy)
bool pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

void add_chunks(std::vector<Chunk> &v, const HostRange &r) {
  for (size_t o = 0; o < r.bytes; o += CHUNK)
    v.push_back({(char *)r.dev + o, (char *)r.host + o, std::min(CHUNK, r.bytes - o)});
}

// The memcpy half of a copy: pieces in order, chunk c's once c < avail.
class Pieces {
 public:
  Pieces(const std::vector<Chunk> &chunks, char *ring, int slots, bool up)
      : chunks_(chunks), ring_(ring), slots_(slots), up_(up),
        done_(new std::atomic<int>[chunks.size()]) {
    for (size_t c = 0; c < chunks.size(); c++) done_[c].store(0, std::memory_order_relaxed);
  }
  ~Pieces() {
    stop_.store(true);
    for (auto &t : helpers_) t.join();
  }
  void start_helpers() {
    const size_t total = chunks_.size() * CHUNK;
    const int cpus = (int)std::thread::hardware_concurrency();
    const int want = std::min({MAX_HELPERS, (int)(total / BYTES_PER_HELPER), cpus - 1});
    try {
      helpers_.reserve(MAX_HELPERS);
      for (int t = 0; t < want; t++) helpers_.emplace_back([this] { run(); });
    } catch (const std::system_error &) {  // fewer threads then
    } catch (const std::bad_alloc &) {
    }
  }
  void set_avail(int chunks) { avail_.store(chunks, std::memory_order_release); }
  bool done(int c) const { return done_[c].load(std::memory_order_acquire) == PIECES; }
  // the calling thread's share: one piece if one can be taken now
  bool help() {
    int p = next_.load(std::memory_order_relaxed);
    while (p / PIECES < avail_.load(std::memory_order_acquire))
      if (next_.compare_exchange_weak(p, p + 1, std::memory_order_relaxed)) {
        copy(p);
        return true;
      }
    return false;
  }

 private:
  void run() {
    const int total = (int)chunks_.size() * PIECES;
    for (;;) {
      const int p = next_.fetch_add(1, std::memory_order_relaxed);
      if (p >= total) return;
      while (avail_.load(std::memory_order_acquire) <= p / PIECES) {
        if (stop_.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      copy(p);
    }
  }
  void copy(int p) {
    const int c = p / PIECES;
    const Chunk &k = chunks_[(size_t)c];
    const size_t off = (size_t)(p % PIECES) * PIECE;
    if (off < k.bytes) {
      const size_t n = std::min(PIECE, k.bytes - off);
      char *slot = ring_ + (size_t)(c % slots_) * CHUNK + off;
      if (up_)
        stream_copy(slot, k.host + off, n);
      else
        stream_copy(k.host + off, slot, n);
    }
    done_[c].fetch_add(1, std::memory_order_release);
  }

  const std::vector<Chunk> &chunks_;
  char *ring_;
  const int slots_;
  const bool up_;
  std::unique_ptr<std::atomic<int>[]> done_;
  std::atomic<int> next_{0}, avail_{0};
  std::atomic<bool> stop_{false};
  std::vector<std::thread> helpers_;
};

// has the event's copy landed?  (its "not ready" is not left as the last error)
hipError_t landed(hipEvent_t e, bool &yes) {
  const hipError_t r = hipEventQuery(e);
  yes = r == hipSuccess;
  if (r != hipErrorNotReady) return r;
  (void)hipGetLastError();
  return hipSuccess;
}

}  // namespace

#define HC_TRY(expr)                      \
  do {                                    \
    const hipError_t e_ = (expr);         \
    if (e_ != hipSuccess) return e_;      \
  } while (0)

bool HostCopy::prepare() {
  if (ring_) return true;
  bool ok = hipStreamCreateWithFlags(&side_, hipStreamNonBlocking) == hipSuccess &&
            hipEventCreateWithFlags(&order_, hipEventDisableTiming) == hipSuccess;
  for (auto &e : landed_)
    ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
  ok = ok && hipHostMalloc((void **)&ring_, SLOTS * CHUNK, hipHostMallocPortable) == hipSuccess;
  if (!ok) {  // the runtime's copy then
    release();
    (void)hipGetLastError();
  }
  return ok;
}

void HostCopy::release() {
  if (side_) (void)hipStreamDestroy(side_);
  if (order_) (void)hipEventDestroy(order_);
  for (auto &e : landed_) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (ring_) (void)hipHostFree(ring_);
  side_ = nullptr;
  order_ = nullptr;
  ring_ = nullptr;
}

hipError_t HostCopy::send(const HostRange *r, int count, hipStream_t s) try {
  std::vector<Chunk> chunks;
  for (int i = 0; i < count; i++) {
    if (r[i].bytes >= DIRECT_BYTES && pageable(r[i].host) && prepare())
      add_chunks(chunks, r[i]);
    else
      HC_TRY(hipMemcpyAsync(r[i].dev, r[i].host, r[i].bytes, hipMemcpyHostToDevice, s));
  }
  if (chunks.empty()) return hipSuccess;
  const int n = (int)chunks.size();
  const bool two = n > 1;
  Pieces pieces(chunks, ring_, SLOTS, true);
  pieces.set_avail(std::min(n, SLOTS));
  size_t bytes = 0;
  for (const Chunk &c : chunks) bytes += c.bytes;
  if (bytes >= UP_HELPER_BYTES) pieces.start_helpers();
  int issued = 0, retired = 0;  // chunks given to the DMA, chunks it is done with
  while (issued < n) {
    if (pieces.done(issued)) {
      const Chunk &c = chunks[(size_t)issued];
      const int slot = issued % SLOTS;
      const hipStream_t q = two && slot & 1 ? side_ : s;
      HC_TRY(hipMemcpyAsync(c.dev, ring_ + slot * CHUNK, c.bytes, hipMemcpyHostToDevice, q));
      HC_TRY(hipEventRecord(landed_[slot], q));
      issued++;
      continue;
    }
    if (pieces.help()) continue;
    bool yes = false;
    if (retired < issued) HC_TRY(landed(landed_[retired % SLOTS], yes));
    if (yes)
      pieces.set_avail(std::min(n, ++retired + SLOTS));
    else
      std::this_thread::yield();
  }
  if (!two) return hipSuccess;
  HC_TRY(hipEventRecord(order_, side_));
  return hipStreamWaitEvent(s, order_, 0);
} catch (const std::bad_alloc &) {
  return hipErrorOutOfMemory;
}

hipError_t HostCopy::receive(const HostRange &r, hipStream_t s) try {
  if (r.bytes < DIRECT_BYTES || !pageable(r.host) || !prepare()) {
    HC_TRY(hipMemcpyAsync(r.host, r.dev, r.bytes, hipMemcpyDeviceToHost, s));
    return hipStreamSynchronize(s);
  }
  std::vector<Chunk> chunks;
  add_chunks(chunks, r);
  const int n = (int)chunks.size();
  const bool two = n > 1;
  if (two) {
    HC_TRY(hipEventRecord(order_, s));
    HC_TRY(hipStreamWaitEvent(side_, order_, 0));
  }
  int issued = 0, arrived = 0, freed = 0;  // chunks given to the DMA, in the ring, copied out
  Pieces pieces(chunks, ring_, SLOTS, false);
  while (freed < n) {
    if (issued < n && issued < freed + SLOTS) {
      const Chunk &c = chunks[(size_t)issued];
      const int slot = issued % SLOTS;
      const hipStream_t q = two && slot & 1 ? side_ : s;
      HC_TRY(hipMemcpyAsync(ring_ + slot * CHUNK, c.dev, c.bytes, hipMemcpyDeviceToHost, q));
      HC_TRY(hipEventRecord(landed_[slot], q));
      issued++;
      continue;
    }
    if (arrived == 0) {  // the work on s may be long: no thread spins through it
      HC_TRY(hipEventSynchronize(landed_[0]));
      pieces.set_avail(++arrived);
      pieces.start_helpers();
    }
    bool yes = false;
    if (arrived < issued) HC_TRY(landed(landed_[arrived % SLOTS], yes));
    if (yes) pieces.set_avail(++arrived);
    if (pieces.done(freed))
      freed++;
    else if (!pieces.help() && !yes)
      std::this_thread::yield();
  }
  return hipSuccess;
} catch (const std::bad_alloc &) {
  return hipErrorOutOfMemory;
}

// after an error nothing still uses the ring
hipError_t HostCopy::settled(hipError_t e, hipStream_t s) {
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(s);
    if (side_) (void)hipStreamSynchronize(side_);
  }
  return e;
}

hipError_t HostCopy::up(const HostRange *r, int count, hipStream_t s) {
  return settled(send(r, count, s), s);
}

hipError_t HostCopy::down(const HostRange &r, hipStream_t s) { return settled(receive(r, s), s); }

}  // namespace caps
