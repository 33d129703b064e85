// host_copy.hip -- device-to-host copies into a caller's ordinary memory.
//
// The runtime's own copy stages such a transfer through pinned memory with one
// host thread, which also takes the page faults of a fresh destination: 10 to
// 14 GB/s on the machine this is written for, where the link moves 50.  Here
// the pieces of a large copy go through a ring of pinned buffers that several
// threads empty.  Five fields into fresh memory, before and after: 0.28 -> 0.26
// ms at 4.4 MB (40^3), 1.0 -> 0.73 at 15 MB (64^3), 9.6 -> 3.3 at 101 MB
// (128^3), 68 -> 20 at 736 MB (256^3).  What bounds the large copy is the link
// and about 14 us between two pieces; the small one, the start of the threads.
// The ring is shared by the blocks of the process (16 MiB, made once they have read
// enough and given back with the last of them) and used by one copy at a time; a
// copy that finds it taken, or no threads to be had, goes the runtime's way.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "cbns_internal.hpp"

namespace cbns {

namespace {

constexpr size_t RING = 16u << 20;
constexpr int MAX_THREADS = 8;  // 4 and 12 are within the noise of 8
// Copies below this go the runtime's way: at 2.6 MB (32^3) its 0.15 ms are no
// more than the ring's.
constexpr size_t LEAST = 4u << 20;
// Bytes read since the last ring was given back that are worth a new one.  Its pinned
// memory takes 1.5 ms to make where the runtime does not hold some, and given back
// it takes the place of a block's arrays among what the runtime holds.  A program
// that makes a block of 64^3, reads its state once (15 MB) and frees it, again and
// again, waited 2.3 ms for the read with a ring each time, 1.1 without; the ring saves
// 0.3 of them.  A copy of 64 MiB pays for it at once.
constexpr size_t WORTH = 64u << 20;
// A copy without the ring goes in parts below 1 MiB, from where on the runtime pins the
// destination for the copy instead of staging it: five fields into memory fresh from
// the kernel, one by one / one copy / parts, us: 24^3 292 / 316 / 262, 32^3 528 / 618 /
// 498, 38^3 766 / 924 / 740; into memory used before 105 / 80 / 72, 155 / 148 / 128, 207 /
// 219 / 186.  Up to 32 MiB: 16 MiB fresh / used whole 5.2 / 0.99 ms, in parts 4.4 / 0.90,
// 48 MiB 15.7 / 2.9 and 14.4 / 3.3.
constexpr size_t PART = 1020u << 10, MOST_PARTED = 32u << 20;
// Bytes of a piece.  2 MiB fill the pipeline sooner (0.27 ms against 0.35 at
// 4.4 MB), 4 MiB have fewer gaps (43 GB/s against 38 at 736 MB; 1 MiB 30).
inline size_t piece_of(size_t bytes) { return bytes < (32u << 20) ? 2u << 20 : 4u << 20; }
constexpr int BUFFERS = 8;  // of the smaller pieces

struct Ring {
  std::mutex mu;      // held by the copy that uses the buffers
  std::mutex refs_mu;
  int refs = 0;
  char* buf = nullptr;
  size_t without = 0;  // bytes copied since there was no ring, up to WORTH
};
Ring ring;

struct Events {
  hipEvent_t ev[BUFFERS] = {};
  ~Events() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  }
  bool create() {
    for (hipEvent_t& e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return false;
    return true;
  }
};

// Pieces of one copy: the calling thread moves them into the ring in order,
// the workers take them out.
struct Copy {
  const char* dev;
  char* host;
  size_t bytes, piece;
  int buffers, pieces;
  int issued = 0;              // pieces on their way into the ring, or past it
  std::atomic<int> next{0};    // piece the next free worker takes
  std::atomic<int> landed{0};  // pieces that have arrived in the ring
  std::atomic<bool> failed{false};
  std::unique_ptr<std::atomic<bool>[]> out;  // piece has left the ring

  size_t size(int p) const { return std::min(piece, bytes - p * piece); }
  void work() {
    for (;;) {
      const int p = next.fetch_add(1);
      if (p >= pieces) return;
      while (landed.load(std::memory_order_acquire) <= p) {
        if (failed.load()) return;
        std::this_thread::yield();
      }
      std::memcpy(host + p * piece, ring.buf + p % buffers * piece, size(p));
      out[p].store(true, std::memory_order_release);
    }
  }
  // issues the pieces that piece p's turn leaves room for; false after a HIP error
  bool issue(int p, hipStream_t s, Events& e) {
    for (; issued < pieces && issued < p + buffers; issued++) {
      if (issued >= buffers) {
        // has the buffer's last piece left it?  Only the piece that is due
        // next is waited for: the others can be issued a round later
        if (issued > p && !out[issued - buffers].load(std::memory_order_acquire)) break;
        while (!out[issued - buffers].load(std::memory_order_acquire)) std::this_thread::yield();
      }
      const int b = issued % buffers;
      if (hipMemcpyAsync(ring.buf + b * piece, dev + issued * piece, size(issued),
                         hipMemcpyDeviceToHost, s) != hipSuccess ||
          hipEventRecord(e.ev[b], s) != hipSuccess)
        return false;
    }
    return true;
  }
  // moves the pieces into the ring; false after a HIP error
  bool feed(hipStream_t s, Events& e) {
    for (int p = 0; p < pieces; p++) {
      if (!issue(p, s, e)) return false;
      if (hipEventSynchronize(e.ev[p % buffers]) != hipSuccess) return false;
      landed.store(p + 1, std::memory_order_release);
    }
    return true;
  }
};

// Memory that HIP does not know, as malloc returns it.  What a caller has pinned
// (or allocated on a device) is the runtime's to copy to: it writes pinned memory
// over the link at once, and the ring would add a pass of the host over every byte
// (one field into pinned memory, ring / runtime: 0.65 / 0.37 ms at 20 MB, 1.9 / 1.4
// at 76 MB).
bool ordinary_memory(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

// the ring's way; false if it could not be taken (nothing copied, or not all)
bool ring_copy(hipStream_t s, const void* dev, void* host, size_t bytes) {
  std::unique_lock<std::mutex> lock(ring.mu, std::try_to_lock);
  if (!lock.owns_lock()) return false;
  if (!ring.buf) {
    ring.without = std::min(WORTH, ring.without + std::min(bytes, WORTH));
    if (ring.without < WORTH) return false;
  }
  Events e;
  Copy c;
  std::vector<std::thread> threads;
  bool ok = false;
  try {
    if (!ring.buf && hipHostMalloc((void**)&ring.buf, RING, hipHostMallocPortable) != hipSuccess) {
      ring.buf = nullptr;
      (void)hipGetLastError();
      return false;
    }
    if (!e.create()) return false;
    c.dev = static_cast<const char*>(dev);
    c.host = static_cast<char*>(host);
    c.bytes = bytes;
    c.piece = piece_of(bytes);
    c.buffers = (int)(RING / c.piece);
    c.pieces = (int)((bytes + c.piece - 1) / c.piece);
    c.out.reset(new std::atomic<bool>[c.pieces]);
    for (int p = 0; p < c.pieces; p++) c.out[p].store(false, std::memory_order_relaxed);
    const unsigned cores = std::max(2u, std::thread::hardware_concurrency());
    const int n = std::min({MAX_THREADS, c.pieces, (int)(cores / 2)});
    threads.reserve(n);
    // the first pieces are on their way while the threads start
    ok = c.issue(0, s, e);
    for (int t = 0; ok && t < n; t++) threads.emplace_back([&c] { c.work(); });
  } catch (...) {  // no memory or no thread: those that run do the copy
    if (threads.empty()) ok = false;
  }
  ok = ok && c.feed(s, e);
  if (!ok) c.failed.store(true);
  for (std::thread& t : threads) t.join();
  if (!ok) (void)hipStreamSynchronize(s);  // nothing writes the ring any more
  return ok;
}

}  // namespace

void host_copy_ref() {
  std::lock_guard<std::mutex> lock(ring.refs_mu);
  ring.refs++;
}

void host_copy_unref() {
  std::lock_guard<std::mutex> lock(ring.refs_mu);
  if (--ring.refs > 0) return;
  std::lock_guard<std::mutex> use(ring.mu);
  if (ring.buf) (void)hipHostFree(ring.buf);
  ring.buf = nullptr;
  ring.without = 0;
}

int copy_to_host(cbns_block* b, const void* dev, void* host, size_t bytes) {
  const bool ordinary = bytes > PART && ordinary_memory(host);
  if (ordinary && bytes >= LEAST) {
    // what is queued ahead of the copy is waited for by this thread alone: the ring's
    // would poll all that time, and other blocks' copies would find the ring taken
    CBNS_HIP(b, hipStreamSynchronize(b->stream));
    if (ring_copy(b->stream, dev, host, bytes)) return CBNS_OK;
  }
  const size_t parts = ordinary && bytes <= MOST_PARTED ? (bytes + PART - 1) / PART : 1;
  for (size_t p = 0; p < parts; p++) {
    const size_t from = bytes * p / parts, to = bytes * (p + 1) / parts;
    CBNS_HIP(b, hipMemcpyAsync(static_cast<char*>(host) + from,
                               static_cast<const char*>(dev) + from, to - from,
                               hipMemcpyDeviceToHost, b->stream));
  }
  CBNS_HIP(b, hipStreamSynchronize(b->stream));
  return CBNS_OK;
}

}  // namespace cbns
