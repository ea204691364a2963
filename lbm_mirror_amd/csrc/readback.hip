// Read-back of device arrays.  A copy straight into the caller's (pageable)
// memory goes through the runtime's own staging in one thread at about 10 GB/s,
// most of which is the kernel handing out the caller's fresh pages; widening
// FP32 to the interface's doubles on the device doubles what crosses the bus and
// takes a device allocation per call.  Here the device's own type crosses into
// pinned slots, and threads widen it from there into the caller's pages while
// the next slots fill.  Density and velocity of 512 x 128 x 128 cells (FP32, 268
// MB of doubles): 27 ms before, about 5 ms now; of 256 x 64 cells (FP64) about
// 110 us before, 50 us now (one wait for both arrays, no allocation).
#include "readback.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

namespace lbmx {
namespace {

constexpr int kSlots = 4;                  // pinned slots in flight
constexpr size_t kSlot = size_t(8) << 20;  // their most
constexpr size_t kPiece = size_t(1) << 20;  // of a slot per thread at a time: 2 MiB of doubles, one huge page
// Up to here the calling thread copies and widens by itself: a thread costs some
// 70 us to start and join (3 MB of FP32 176 us alone, 610 us with 8 threads; 6 MB 291
// and 690; 12 MB 645 alone, 476 with 4).  Beyond it a thread per kPerThread bytes.
constexpr size_t kAlone = size_t(8) << 20;
constexpr size_t kPerThread = size_t(4) << 20;
constexpr unsigned kThreads = 8;
constexpr size_t kKept = 2;  // stages kept between calls

struct Stage {
  int device = 0;
  char* mem = nullptr;
  size_t size = 0;
  bool pinned = true;
  hipEvent_t ev[kSlots] = {};
};

std::mutex g_mu;
int g_users = 0;
Stage g_free[kKept];  // (never destroyed: no HIP call after main)
size_t g_kept = 0;

void drop(Stage& t) {
  for (hipEvent_t e : t.ev)
    if (e) (void)hipEventDestroy(e);
  if (t.mem && t.pinned) (void)hipHostFree(t.mem);
  else std::free(t.mem);
  t = Stage();
}

hipError_t take(int device, size_t size, Stage& t) {
  Stage small;  // one that is in the way
  {
    std::lock_guard<std::mutex> lock(g_mu);
    auto pick = [](size_t i) {  // (the others stay in order)
      const Stage f = g_free[i];
      for (--g_kept; i < g_kept; ++i) g_free[i] = g_free[i + 1];
      return f;
    };
    for (size_t i = 0; i < g_kept; ++i) {
      if (g_free[i].device != device || g_free[i].size < size) continue;
      t = pick(i);
      return hipSuccess;
    }
    if (g_kept == kKept) small = pick(0);
  }
  drop(small);
  t = Stage();
  t.device = device;
  t.size = size;
  hipError_t e = hipHostMalloc((void**)&t.mem, size, hipHostMallocDefault);
  if (e != hipSuccess) {  // no pinned memory: ordinary memory, through the runtime's own staging
    (void)hipGetLastError();
    t.pinned = false;
    t.mem = static_cast<char*>(std::malloc(size));
    e = t.mem ? hipSuccess : hipErrorOutOfMemory;
  }
  for (int i = 0; i < kSlots && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&t.ev[i], hipEventDisableTiming);
  if (e != hipSuccess) drop(t);
  return e;
}

void give(Stage& t) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_users > 0 && t.pinned && g_kept < kKept) {
      g_free[g_kept++] = t;
      return;
    }
  }
  drop(t);
}

struct Chunk {
  const ReadBack* of;
  size_t offset, bytes, piece;
  size_t pieces() const { return (bytes + piece - 1) / piece; }
};

hipError_t read_chunks(hipStream_t s, Stage& t, size_t slot, const std::vector<Chunk>& chunks, unsigned want) {
  std::mutex mu;
  std::condition_variable cv;
  size_t ready = 0, chunk = 0, piece = 0;  // chunks that arrived; the next piece to take
  std::vector<size_t> left(chunks.size());
  for (size_t i = 0; i < chunks.size(); ++i) left[i] = chunks[i].pieces();
  bool stop = false;
  // takes pieces in order; `all`: until none is left, else those that arrived
  auto work = [&](bool all) {
    std::unique_lock<std::mutex> lock(mu);
    while (chunk < chunks.size()) {
      if (chunk >= ready) {
        if (stop || !all) return;
        cv.wait(lock);
        continue;
      }
      const size_t c = chunk, p = piece;
      if (++piece == chunks[c].pieces()) {
        piece = 0;
        ++chunk;
      }
      lock.unlock();
      const Chunk& k = chunks[c];
      const size_t at = p * k.piece;
      k.of->use(t.mem + (c % kSlots) * slot + at, k.offset + at, std::min(k.piece, k.bytes - at));
      lock.lock();
      if (--left[c] == 0) cv.notify_all();
    }
  };
  std::thread th[kThreads];
  unsigned n = 0;
  try {
    for (; n < want; ++n) th[n] = std::thread(work, true);
  } catch (...) {  // as many as there are; the calling thread works if there is none
  }
  hipError_t e = hipSuccess;
  auto arrived = [&](size_t i) {
    e = hipEventSynchronize(t.ev[i % kSlots]);
    if (e != hipSuccess) return;
    {
      std::lock_guard<std::mutex> lock(mu);
      ready = i + 1;
    }
    cv.notify_all();
    if (n == 0) work(false);
  };
  for (size_t i = 0; i < chunks.size() && e == hipSuccess; ++i) {
    if (i >= kSlots) {
      std::unique_lock<std::mutex> lock(mu);
      cv.wait(lock, [&] { return left[i - kSlots] == 0; });
    }
    e = hipMemcpyAsync(t.mem + (i % kSlots) * slot, (const char*)chunks[i].of->src + chunks[i].offset, chunks[i].bytes,
                       hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipEventRecord(t.ev[i % kSlots], s);
    // (keep kSlots - 1 copies queued behind the one waited for)
    if (e == hipSuccess && i + 1 >= kSlots) arrived(i + 1 - kSlots);
  }
  for (size_t i = chunks.size() < kSlots ? 0 : chunks.size() - kSlots + 1; i < chunks.size() && e == hipSuccess; ++i)
    arrived(i);
  {
    std::lock_guard<std::mutex> lock(mu);
    stop = true;
  }
  cv.notify_all();
  for (unsigned i = 0; i < n; ++i) th[i].join();
  return e;
}

}  // namespace

void read_back_user(int change) {
  Stage gone[kKept];
  {
    std::lock_guard<std::mutex> lock(g_mu);
    g_users += change;
    if (g_users == 0)
      for (; g_kept > 0; --g_kept) gone[g_kept - 1] = g_free[g_kept - 1];
  }
  for (Stage& t : gone) drop(t);
}

hipError_t read_back(int device, hipStream_t s, const ReadBack* what, int count) {
  size_t total = 0;
  for (int i = 0; i < count; ++i) total += what[i].bytes;
  if (total == 0) return hipStreamSynchronize(s);
  Stage t;
  hipError_t e;
  if (total <= kAlone) {
    size_t size = kAlone / 16;
    while (size < total) size *= 2;
    e = take(device, size, t);
    size_t at = 0;
    for (int i = 0; i < count && e == hipSuccess; ++i) {
      if (what[i].bytes) e = hipMemcpyAsync(t.mem + at, what[i].src, what[i].bytes, hipMemcpyDeviceToHost, s);
      at += what[i].bytes;
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    at = 0;
    for (int i = 0; i < count && e == hipSuccess; ++i) {
      if (what[i].bytes) what[i].use(t.mem + at, 0, what[i].bytes);
      at += what[i].bytes;
    }
  } else {
    // slots of whole pieces; arrays of a few slots' size in smaller ones, so
    // that their threads start before the last byte has arrived
    const size_t piece = std::min(kPiece, total / 32 / 4096 * 4096);
    const size_t slot = std::min(kSlot, total / (2 * kSlots) / piece * piece);
    try {
      std::vector<Chunk> chunks;
      for (int i = 0; i < count; ++i) {
        const size_t p = piece / what[i].unit * what[i].unit, c = slot / piece * p;
        for (size_t o = 0; o < what[i].bytes; o += c) chunks.push_back({&what[i], o, std::min(c, what[i].bytes - o), p});
      }
      e = take(device, kSlots * slot, t);
      const unsigned cpu = std::max(2u, std::thread::hardware_concurrency()) / 2;
      if (e == hipSuccess)
        e = read_chunks(s, t, slot, chunks, unsigned(std::min<size_t>({kThreads, cpu, total / kPerThread})));
    } catch (const std::bad_alloc&) {
      e = hipErrorOutOfMemory;
    }
  }
  if (t.mem) {
    if (e != hipSuccess) {  // copies may still be under way
      (void)hipStreamSynchronize(s);
      drop(t);
    } else {
      give(t);
    }
  }
  return e;
}

}  // namespace lbmx
