#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace ihip {
namespace {

// Pieces of host memory to copy, cut into shares that whoever has time takes in order.
struct Job {
  std::vector<CopyPiece> pieces;
  std::vector<std::pair<size_t, size_t>> shares;  // (piece, offset)
  std::unique_ptr<std::atomic<size_t>[]> left;    // shares of a piece that are not done
  std::atomic<size_t> next{0}, active{0};         // the share that is taken next; threads that are in step()

  // A share is what a thread copies in about 10 us, the time it takes to wake one; 1 MiB of the 8 MiB chunks that both
  // directions of a large call fill and empty side by side (row softmax of 16384 x 4096 through the host entry: 7.5 ms, with
  // shares of 128 KiB 8.1; 33 MB through the mirror 0.82 ms with those, 0.92 with 1 MiB).
  static size_t share_of(const CopyPiece& piece) { return piece.bytes >= size_t(8) << 20 ? size_t(1) << 20 : size_t(128) << 10; }
  explicit Job(std::vector<CopyPiece> given) : pieces(std::move(given)), left(new std::atomic<size_t>[pieces.size() + 1]) {
    for (size_t p = 0; p < pieces.size(); ++p) {
      size_t count = 0;
      for (size_t at = 0; at < pieces[p].bytes; at += share_of(pieces[p]), ++count) shares.push_back({p, at});
      left[p].store(count);
    }
  }
  // takes the next share, if there is one
  bool step() {
    active.fetch_add(1);
    const size_t n = next.fetch_add(1);
    if (n >= shares.size()) {
      active.fetch_sub(1);
      return false;
    }
    const auto [p, at] = shares[n];
    const CopyPiece& piece = pieces[p];
    std::memcpy(static_cast<char*>(piece.dst) + at, static_cast<const char*>(piece.src) + at, std::min(share_of(piece), piece.bytes - at));
    left[p].fetch_sub(1, std::memory_order_release);
    active.fetch_sub(1);
    return true;
  }
  // no share is begun any more, and none is being copied
  void stop() {
    next.store(shares.size());
    while (active.load() != 0) std::this_thread::yield();
  }
  bool done(size_t p) const { return left[p].load(std::memory_order_acquire) == 0; }
  // returns when piece p is copied; the caller copies too
  void wait(size_t p) {
    while (!done(p))
      if (!step()) std::this_thread::yield();  // (its last shares are with other threads, for 10 us, or about 80 where a share is 1 MiB)
  }
};

// A few threads that copy shares of the jobs at hand (one thread moves 10-15 GB/s, the link to the device four times
// that).  ILANG_HIP_COPY_THREADS sets their number (default 8, the caller included; 1: the caller alone).  The threads
// are started by the first job that is worth waking them and live until the process ends; where the system has no more
// threads to give, those that there are do the work, or the caller alone.
class CopyCrew {
 public:
  static CopyCrew& get() {
    static CopyCrew* crew = new CopyCrew();  // (never destroyed: its threads may outlive static destructors)
    return *crew;
  }
  // Waking the others costs the caller 15 us, and what is in its caches it copies alone at 40 GB/s: a host call that sums rows
  // of 0.6 MB takes 53 us alone and 59 with the others, of 1.0 MB 68 either way, of 1.6 MB 96 and 81.
  static constexpr size_t kWorthWaking = size_t(1) << 20;
  void post(const std::shared_ptr<Job>& job) {
    std::call_once(started_, [this] { start(); });
    if (threads_ == 0) return;
    {
      std::lock_guard<std::mutex> lock(mu_);
      jobs_.push_back(job);
    }
    wake_.notify_all();
  }
  void copy(void* dst, const void* src, size_t bytes) {
    if (bytes < kWorthWaking) {
      if (bytes) std::memcpy(dst, src, bytes);
      return;
    }
    auto job = std::make_shared<Job>(std::vector<CopyPiece>{{dst, src, bytes}});
    post(job);
    job->wait(0);
  }

 private:
  CopyCrew() = default;
  void start() {
    size_t n = 8;
    if (const char* v = std::getenv("ILANG_HIP_COPY_THREADS")) n = (size_t)std::max(1, std::atoi(v));
    n = std::min<size_t>(n, std::max(1u, std::thread::hardware_concurrency()));
    for (size_t t = 1; t < n; ++t) {
      try {
        std::thread([this] { work(); }).detach();
      } catch (const std::system_error&) {
        return;
      }
      ++threads_;
    }
  }
  void work() {
    std::unique_lock<std::mutex> lock(mu_);
    for (;;) {
      wake_.wait(lock, [&] { return !jobs_.empty(); });
      const std::shared_ptr<Job> job = jobs_.front();
      lock.unlock();
      while (job->step()) {
      }
      lock.lock();
      if (!jobs_.empty() && jobs_.front() == job) jobs_.pop_front();  // (every share is taken)
    }
  }
  std::mutex mu_;
  std::condition_variable wake_;
  std::deque<std::shared_ptr<Job>> jobs_;
  std::once_flag started_;
  size_t threads_ = 0;
};

// A ring of page-locked chunks of one device (one for each direction): four chunks of 8 MiB (small enough that the first chunk's fill and
// the last chunk's transfer, which nothing overlaps, are a small part of a 64 MiB operand), allocated by the first
// large host call on that device and kept until the process ends.  One transfer uses the ring at a time; a chunk
// whose last transfer may still be in flight (in_flight) is awaited before it is touched again, not before: the
// upload of one operand runs into the upload of the next.
constexpr size_t kChunkBytes = size_t(8) << 20;
constexpr int kChunks = 4;
struct Ring {
  void* chunk[kChunks] = {};
  hipEvent_t landed[kChunks] = {};
  bool in_flight[kChunks] = {};
  size_t next = 0;  // the chunk that the next transfer step takes
  bool ready = false, failed = false;
  std::mutex busy;
  Err settle(int slot) {
    if (!in_flight[slot]) return {};
    in_flight[slot] = false;
    return check(hipEventSynchronize(landed[slot]), "hipEventSynchronize");
  }
};

struct RingTable {
  std::mutex mu;
  std::map<int, std::unique_ptr<Ring>> rings;
};
RingTable& ring_table() {
  static RingTable* table = new RingTable();
  return *table;
}
// (a ring for uploads and one for downloads per device, so that a download on one thread can run beside an upload
// on another: the link carries both directions at once)
Ring* ring_of_current_device(bool download) {
  RingTable& t = ring_table();
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lock(t.mu);
  auto& ring = t.rings[2 * device + (download ? 1 : 0)];
  if (!ring) ring = std::make_unique<Ring>();
  return ring.get();
}

// with ring->busy held
bool prepare(Ring* ring) {
  if (ring->ready) return true;
  if (ring->failed) return false;
  for (int c = 0; c < kChunks; ++c)
    if (hipHostMalloc(&ring->chunk[c], kChunkBytes, hipHostMallocDefault) != hipSuccess ||
        hipEventCreateWithFlags(&ring->landed[c], hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      ring->failed = true;  // (no page-locked memory to be had: plain copies from now on)
      return false;
    }
  ring->ready = true;
  return true;
}

}  // namespace

size_t release_copy_chunks() {
  RingTable& t = ring_table();
  std::lock_guard<std::mutex> lock(t.mu);
  size_t released = 0;
  for (auto& [device, ring] : t.rings) {
    std::unique_lock<std::mutex> idle(ring->busy, std::try_to_lock);
    if (!idle.owns_lock() || !ring->ready) continue;
    for (int c = 0; c < kChunks; ++c) {
      (void)ring->settle(c);
      (void)hipHostFree(ring->chunk[c]);
      (void)hipEventDestroy(ring->landed[c]);
      ring->chunk[c] = nullptr;
      ring->landed[c] = nullptr;
      released += kChunkBytes;
    }
    ring->ready = false;
  }
  return released;
}

void copy_by_threads(void* dst, const void* src, size_t bytes) { CopyCrew::get().copy(dst, src, bytes); }

struct CopyAhead::State {
  std::shared_ptr<Job> job;
};
CopyAhead::CopyAhead(std::vector<CopyPiece> pieces) {
  size_t bytes = 0;
  for (const CopyPiece& piece : pieces) bytes += piece.bytes;
  if (bytes < CopyCrew::kWorthWaking) {  // (the caller alone, at once and without a job)
    for (const CopyPiece& piece : pieces)
      if (piece.bytes) std::memcpy(piece.dst, piece.src, piece.bytes);
    return;
  }
  state_.reset(new State{std::make_shared<Job>(std::move(pieces))});
  CopyCrew::get().post(state_->job);
}
CopyAhead::~CopyAhead() {
  if (state_) state_->job->stop();
}
void CopyAhead::wait(size_t piece) {
  if (state_) state_->job->wait(piece);
}

Err upload_pipelined(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  Ring* ring = bytes >= kPipelinedCopyBytes ? ring_of_current_device(false) : nullptr;
  std::unique_lock<std::mutex> lock;
  if (ring) lock = std::unique_lock<std::mutex>(ring->busy, std::try_to_lock);
  if (!ring || !lock.owns_lock() || !prepare(ring)) return h2d(dst, src, bytes, stream);
  for (size_t at = 0; at < bytes; at += kChunkBytes) {
    const int slot = (int)(ring->next++ % kChunks);
    const size_t len = std::min(kChunkBytes, bytes - at);
    if (Err e = ring->settle(slot); !e.empty()) return e;  // the chunk's last transfer has left it
    CopyCrew::get().copy(ring->chunk[slot], static_cast<const char*>(src) + at, len);
    if (Err e = check(hipMemcpyAsync(static_cast<char*>(dst) + at, ring->chunk[slot], len, hipMemcpyHostToDevice, stream), "hipMemcpy H2D");
        !e.empty())
      return e;
    if (Err e = check(hipEventRecord(ring->landed[slot], stream), "hipEventRecord"); !e.empty()) return e;
    ring->in_flight[slot] = true;
  }
  return {};
}

Err download_pipelined(void* dst, const void* src, size_t bytes, hipStream_t stream) {
  Ring* ring = bytes >= kPipelinedCopyBytes ? ring_of_current_device(true) : nullptr;
  std::unique_lock<std::mutex> lock;
  if (ring) lock = std::unique_lock<std::mutex>(ring->busy, std::try_to_lock);
  if (!ring || !lock.owns_lock() || !prepare(ring)) {
    if (Err e = d2h(dst, src, bytes, stream); !e.empty()) return e;
    return sync(stream);
  }
  const size_t chunks = (bytes + kChunkBytes - 1) / kChunkBytes, first = ring->next;
  ring->next += chunks;
  auto request = [&](size_t c) -> Err {
    const size_t at = c * kChunkBytes, len = std::min(kChunkBytes, bytes - at);
    const int slot = (int)((first + c) % kChunks);
    if (Err e = ring->settle(slot); !e.empty()) return e;
    if (Err e = check(hipMemcpyAsync(ring->chunk[slot], static_cast<const char*>(src) + at, len, hipMemcpyDeviceToHost, stream), "hipMemcpy D2H");
        !e.empty())
      return e;
    if (Err e = check(hipEventRecord(ring->landed[slot], stream), "hipEventRecord"); !e.empty()) return e;
    ring->in_flight[slot] = true;
    return {};
  };
  // transfers in flight ahead of the chunk that the host threads are emptying: all chunks of the ring but one
  for (size_t c = 0; c < std::min<size_t>(chunks, kChunks - 1); ++c)
    if (Err e = request(c); !e.empty()) return e;
  for (size_t c = 0; c < chunks; ++c) {
    const size_t at = c * kChunkBytes, len = std::min(kChunkBytes, bytes - at);
    const int slot = (int)((first + c) % kChunks);
    if (c + kChunks - 1 < chunks)
      if (Err e = request(c + kChunks - 1); !e.empty()) return e;  // (into the chunk emptied in the step before)
    if (Err e = ring->settle(slot); !e.empty()) return e;
    CopyCrew::get().copy(static_cast<char*>(dst) + at, ring->chunk[slot], len);
  }
  return {};
}

}  // namespace ihip
