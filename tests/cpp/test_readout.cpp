// Host-only driver of the large readouts (madpac_amd/csrc/lbm_readout.cpp) over a stand-in for the few
// runtime calls they make: "device" memory is host memory and copies happen at once.
//
// usage: test_readout whole | nothreads K | known
//   whole        parts around the switch to the ring and with ragged last pieces arrive whole
//   nothreads K  creating a thread runs out of memory after K of them were started
//   known        parts in memory that the runtime knows (pinned) are copied there directly, others not
#include <dlfcn.h>
#include <pthread.h>
#include <stdlib.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <new>
#include <vector>

#include "lbm_readout.h"

namespace {
int g_allowed = -1;                          // threads that may still be started, -1: any number
thread_local bool g_out_of_memory = false;   // operator new of this thread fails
int g_started = 0;
std::atomic<size_t> g_direct{0};             // bytes that a copy moved straight into the caller's memory
const char *g_user = nullptr, *g_user_end = nullptr;
const char *g_known = nullptr, *g_known_end = nullptr;  // pinned memory
}  // namespace

void* operator new(size_t n) {
  if (g_out_of_memory) throw std::bad_alloc();
  if (void* p = malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
  using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Create real = (Create)dlsym(RTLD_NEXT, "pthread_create");
  g_started++;
  if (g_allowed > 0 && --g_allowed == 0) g_out_of_memory = true;
  return real(t, a, f, arg);
}

extern "C" {
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)malloc(1), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return free((void*)e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::memset(a, 0, sizeof(*a));
  a->type = (const char*)p >= g_known && (const char*)p < g_known_end ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(dst, src, n);
  if ((const char*)dst >= g_user && (const char*)dst < g_user_end) g_direct += n;
  return hipSuccess;
}
}

namespace {
// `sizes` bytes from as many sources into one destination, part `pinned` into pinned memory; whether every byte
// arrived and nothing else changed
bool arrives(const std::vector<size_t>& sizes, int pinned = -1) {
  size_t total = 0;
  for (size_t s : sizes) total += s;
  std::vector<unsigned char> src(total), dst(total + 64, 0xA5);
  uint32_t r = 12345;
  for (unsigned char& v : src) v = (unsigned char)((r = r * 1664525u + 1013904223u) >> 24);
  std::vector<lbm::HostCopy> parts;
  size_t o = 0;
  for (size_t s : sizes) {
    parts.push_back(lbm::HostCopy{dst.data() + o, src.data() + o, s});
    if ((int)parts.size() - 1 == pinned) {
      g_known = (const char*)dst.data() + o;
      g_known_end = g_known + s;
    }
    o += s;
  }
  g_user = (const char*)dst.data();
  g_user_end = g_user + total;
  g_direct = 0;
  const hipError_t e = lbm::read_back(parts.data(), (int)parts.size(), nullptr);
  g_out_of_memory = false;
  if (e != hipSuccess || std::memcmp(src.data(), dst.data(), total) != 0) return false;
  for (int k = 0; k < 64; k++)
    if (dst[total + k] != 0xA5) return false;
  return true;
}

constexpr size_t MB = (size_t)1 << 20;
}  // namespace

int main(int argc, char** argv) {
  bool ok = false;
  lbm::readout_hold();
  if (argc == 2 && !std::strcmp(argv[1], "whole")) {
    ok = arrives({24 * MB - 1}) && g_direct == 24 * MB - 1;
    ok = ok && arrives({24 * MB}) && g_direct == 0;
    ok = ok && arrives({8 * MB, 24 * MB + 8}) && arrives({2 * MB - 8, 30 * MB, 8, 2 * MB + 1}) && g_direct == 0;
  } else if (argc == 3 && !std::strcmp(argv[1], "nothreads")) {
    g_allowed = atoi(argv[2]);
    ok = arrives({40 * MB + 24}) && g_started == atoi(argv[2]);
    g_allowed = -1;
    ok = ok && arrives({40 * MB + 24});
  } else if (argc == 2 && !std::strcmp(argv[1], "known")) {
    ok = arrives({32 * MB + 8}, 0) && g_direct == 32 * MB + 8;
    ok = ok && arrives({30 * MB, 30 * MB + 16}, 0) && g_direct == 30 * MB;
    ok = ok && arrives({30 * MB, 30 * MB + 16}, 1) && g_direct == 30 * MB + 16;
    ok = ok && arrives({8 * MB, 23 * MB, 8}, 0) && g_direct == 31 * MB + 8;  // the rest is below the switch
  }
  lbm::readout_release();
  std::printf("%s\n", ok ? "ok" : "failed");
  return ok ? 0 : 1;
}
