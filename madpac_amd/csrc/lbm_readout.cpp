// Readout of large results: device -> pinned staging -> the caller's memory.
//
// hipMemcpy into pageable memory runs at 8-9 GB/s: the runtime pins the destination piece by piece, on
// one thread, which also takes the page faults of a fresh array.  Here the DMA engine fills a ring of
// pinned pieces at the bus rate and a few threads move the pieces on, so that the page faults and the
// copies of different pieces overlap with each other and with the transfer.
#include "lbm_readout.h"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace lbm {

namespace {

// Measured for rho and u of n^3 cells (32 n^3 bytes; ms, first call of a process / later ones): 256^3
// hipMemcpy 56 / 53, this 16 / 15; 128^3 6.6 / 5.8 and 3.9 / 2.1; 96^3 2.8 / 1.6 and 2.9 / 1.0; 64^3 1.0 / 0.5 and,
// had it taken this way, 2.0 / 0.4: below DIRECT the ring's allocation costs a first call more than later
// ones gain.  Pieces of 0.5 and 1 MB take 26 and 18 ms at 256^3; 4, 8 and 12 threads are within 5 %.
constexpr size_t PIECE = (size_t)2 << 20;
constexpr int RING = 8;
constexpr int THREADS = 8;
constexpr size_t DIRECT = (size_t)24 << 20;

struct Staging {
  char* mem = nullptr;
  hipEvent_t arrived[RING] = {};
  int device = -1;  // of the events
  bool busy = false;
};

// Two rings: one per call in flight; a third concurrent call copies directly.
constexpr int RINGS = 2;
std::mutex g_mutex;
int64_t g_holders = 0;
Staging g_rings[RINGS];

void free_ring(Staging& r) {
  for (hipEvent_t& e : r.arrived) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
  if (r.mem) (void)hipHostFree(r.mem);
  r.mem = nullptr;
  r.device = -1;
}

// A ring whose events belong to the current device, or null (all in use, or no pinned memory).
Staging* take_ring() {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return nullptr;
  std::lock_guard<std::mutex> lock(g_mutex);
  Staging* r = nullptr;
  for (Staging& s : g_rings)
    if (!s.busy && (!r || s.device == device)) r = &s;
  if (!r) return nullptr;
  if (r->device != device) {
    free_ring(*r);
    bool ok = hipHostMalloc((void**)&r->mem, RING * PIECE, hipHostMallocPortable) == hipSuccess;
    for (int k = 0; ok && k < RING; k++) ok = hipEventCreateWithFlags(&r->arrived[k], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
      (void)hipGetLastError();
      free_ring(*r);
      return nullptr;
    }
    r->device = device;
  }
  r->busy = true;
  return r;
}

void give_ring(Staging* r) {
  std::lock_guard<std::mutex> lock(g_mutex);
  r->busy = false;
  if (g_holders == 0) free_ring(*r);
}

// Memory that the runtime knows (pinned above all) takes the transfer itself: rho and u of 256^3 cells into
// pinned memory 10.0 ms, through the ring 14.0; 96^3 0.56 and 0.97.
bool known(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return false;
}

struct Piece {
  char* dst;
  const char* src;
  size_t bytes;
};

hipError_t through_ring(Staging& r, const HostCopy* parts, int nparts, hipStream_t stream) {
  std::vector<Piece> pieces;
  for (int p = 0; p < nparts; p++)
    for (size_t o = 0; o < parts[p].bytes; o += PIECE)
      pieces.push_back(Piece{(char*)parts[p].dst + o, (const char*)parts[p].src + o, std::min(PIECE, parts[p].bytes - o)});
  const int n = (int)pieces.size();
  std::mutex m;
  std::condition_variable cv;
  int queued = 0, next = 0;          // pieces handed to the DMA engine; pieces taken by a thread
  std::vector<char> done(n, 0);
  bool stop = false;
  std::atomic<int> error{(int)hipSuccess};
  auto worker = [&] {
    if (hipSetDevice(r.device) != hipSuccess) error = (int)hipErrorInvalidDevice;
    std::unique_lock<std::mutex> lock(m);
    for (;;) {
      cv.wait(lock, [&] { return stop || next < queued || next == n; });
      if (next == n || (stop && next >= queued)) return;
      const int k = next++;
      lock.unlock();
      const hipError_t e = hipEventSynchronize(r.arrived[k % RING]);
      if (e == hipSuccess) std::memcpy(pieces[k].dst, r.mem + (size_t)(k % RING) * PIECE, pieces[k].bytes);
      else error = (int)e;
      lock.lock();
      done[k] = 1;
      cv.notify_all();
    }
  };
  std::vector<std::thread> threads;
  const int want = std::min(THREADS, n);
  threads.reserve(want);
  for (int t = 0; t < want; t++) {
    try {
      threads.emplace_back(worker);
    } catch (const std::exception&) {  // no thread or no memory for one: those that run move all pieces
      break;
    }
  }
  hipError_t e = threads.empty() ? hipErrorOutOfMemory : hipSuccess;
  for (int k = 0; k < n && e == hipSuccess; k++) {
    if (k >= RING) {
      std::unique_lock<std::mutex> lock(m);
      cv.wait(lock, [&] { return done[k - RING] != 0; });
    }
    e = hipMemcpyAsync(r.mem + (size_t)(k % RING) * PIECE, pieces[k].src, pieces[k].bytes, hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipEventRecord(r.arrived[k % RING], stream);
    if (e == hipSuccess) {
      std::lock_guard<std::mutex> lock(m);
      queued = k + 1;
      cv.notify_all();
    }
  }
  {
    std::lock_guard<std::mutex> lock(m);
    stop = true;
    cv.notify_all();
  }
  for (std::thread& t : threads) t.join();
  if (e == hipSuccess) e = (hipError_t)error.load();
  return e;
}

}  // namespace

hipError_t read_back(const HostCopy* parts, int n, hipStream_t stream) {
  constexpr int MOST = 4;
  HostCopy staged[MOST];
  int nstaged = 0;
  size_t total = 0, large = 0;
  for (int p = 0; p < n; p++) total += parts[p].bytes;
  for (int p = 0; p < n && n <= MOST && total >= DIRECT; p++)
    if (!known(parts[p].dst)) {
      staged[nstaged++] = parts[p];
      large += parts[p].bytes;
    }
  bool arrived = false;  // the staged parts
  if (large >= DIRECT) {
    if (Staging* r = take_ring()) {
      hipError_t e;
      try {
        e = through_ring(*r, staged, nstaged, stream);
      } catch (const std::bad_alloc&) {  // from the lists, before any thread is started
        e = hipErrorOutOfMemory;
      }
      (void)hipStreamSynchronize(stream);  // nothing is on its way into the ring when it is given back
      give_ring(r);
      arrived = e == hipSuccess;
    }
  }
  for (int p = 0; p < n; p++) {
    if (arrived && !known(parts[p].dst)) continue;
    const hipError_t e = hipMemcpyAsync(parts[p].dst, parts[p].src, parts[p].bytes, hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess) return e;
  }
  return hipStreamSynchronize(stream);
}

void readout_hold() {
  std::lock_guard<std::mutex> lock(g_mutex);
  g_holders++;
}

void readout_release() {
  std::lock_guard<std::mutex> lock(g_mutex);
  if (--g_holders == 0)
    for (Staging& r : g_rings)
      if (!r.busy) free_ring(r);
}

}  // namespace lbm
