// Device-to-host copies of state arrays into the caller's (pageable) memory.
//
// A copy into pageable memory runs through the runtime's own staging buffer on
// one host thread: 61 ms for the 655 MB state of 2,048 cubes (10.7 GB/s), bound
// by that thread's copy and by the page faults of fresh memory.  Here four host
// threads each hold two pinned chunks: one is filled by the device while the
// other is copied on, and the link (57 GB/s) becomes the bound: 16 ms for 655
// MB, 0.6 ms for 20 MB (1.2 ms before).  Chunks of 2 MB: 1 MB chunks
// take 21 ms for 655 MB, 4 MB chunks 15 ms but twice the pinned memory.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "bcm_engine.h"

namespace bcm {

namespace {
constexpr size_t CHUNK = (size_t)2 << 20;
constexpr int THREADS = 4;
// Below this an engine's first download would pay more for the pinned chunks
// than it saves (9 MB: 0.31 ms against 0.53 ms directly, and 2 ms once).
constexpr size_t DIRECT_BELOW = (size_t)16 << 20;
}  // namespace

// Pinned chunks and their events, two per thread; kept by the engine from the
// first large download until it is destroyed (16 MB).
struct HostChunks {
  char* pin = nullptr;
  hipEvent_t ready[2 * THREADS] = {};
};

namespace {

// The engine's chunks, or null when they cannot be had.
HostChunks* host_chunks(Engine* e) {
  if (e->chunks) return e->chunks;
  const bool clean = hipPeekAtLastError() == hipSuccess;
  e->chunks = new (std::nothrow) HostChunks();
  if (!e->chunks) return nullptr;
  bool ok = hipHostMalloc((void**)&e->chunks->pin, 2 * THREADS * CHUNK) == hipSuccess;
  for (hipEvent_t& ev : e->chunks->ready)
    ok = ok && hipEventCreateWithFlags(&ev, hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    engine_chunks_free(e);
    if (clean) (void)hipGetLastError();   // (no error but the allocation's)
  }
  return e->chunks;
}

}  // namespace

void engine_chunks_free(Engine* e) {
  if (!e->chunks) return;
  if (e->chunks->pin) (void)hipHostFree(e->chunks->pin);
  for (hipEvent_t ev : e->chunks->ready)
    if (ev) (void)hipEventDestroy(ev);
  delete e->chunks;
  e->chunks = nullptr;
}

hipError_t engine_to_host(Engine* e, void* dst, const void* src, size_t bytes) {
  HostChunks* h = bytes < DIRECT_BELOW ? nullptr : host_chunks(e);
  if (!h) {
    const hipError_t rc = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, e->stream);
    return rc != hipSuccess ? rc : hipStreamSynchronize(e->stream);
  }
  const size_t n = (bytes + CHUNK - 1) / CHUNK;
  std::atomic<size_t> next{0};
  std::atomic<int> error{(int)hipSuccess};
  // Thread w takes the next chunk for each of its two slots in turn.  Copies
  // of all threads go to the engine stream, each with its slot's event.
  auto work = [&](int w) {
    auto fail = [&](hipError_t rc) { error = (int)rc; };
    if (hipSetDevice(e->device) != hipSuccess) return fail(hipErrorInvalidDevice);
    size_t at[2];
    auto issue = [&](int s) {
      const size_t q = error == (int)hipSuccess ? next++ : n;
      if (q >= n) return false;
      at[s] = q * CHUNK;
      const size_t len = std::min(CHUNK, bytes - at[s]);
      hipError_t rc = hipMemcpyAsync(h->pin + (2 * w + s) * CHUNK, (const char*)src + at[s], len,
                                     hipMemcpyDeviceToHost, e->stream);
      if (rc == hipSuccess) rc = hipEventRecord(h->ready[2 * w + s], e->stream);
      if (rc != hipSuccess) fail(rc);
      return rc == hipSuccess;
    };
    bool busy[2] = {issue(0), false};
    busy[1] = busy[0] && issue(1);
    for (int s = 0; busy[s]; s ^= 1) {
      const hipError_t rc = hipEventSynchronize(h->ready[2 * w + s]);
      if (rc != hipSuccess) return fail(rc);
      memcpy((char*)dst + at[s], h->pin + (2 * w + s) * CHUNK, std::min(CHUNK, bytes - at[s]));
      busy[s] = issue(s);
    }
  };
  std::vector<std::thread> others;
  try {
    others.reserve(THREADS - 1);
    for (int w = 1; w < THREADS; ++w) others.emplace_back(work, w);
  } catch (const std::exception&) {
    // Fewer threads: the chunks are taken by those that run.
  }
  work(0);
  for (std::thread& t : others) t.join();
  const hipError_t rc = hipStreamSynchronize(e->stream);
  return error != (int)hipSuccess ? (hipError_t)error.load() : rc;
}

}  // namespace bcm
