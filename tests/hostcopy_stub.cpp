// The pinned copy pipeline (mfm_hostcopy.cpp) on host memory: the HIP calls it
// makes, as plain memory operations, and programs over it.
//   race:  eight threads copy through one link at a time, every copy checked
//          (built with the thread sanitizer)
//   pinned: memory that the runtime knows
//   small: segments below the pipeline's size
//   alloc: a thread that cannot be started for want of memory
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <thread>
#include <vector>

#include "../ms-flukss-multifluid_amd/csrc/mfm_host.hpp"

static const void* pinned = nullptr;  // memory the runtime knows
static std::atomic<int> whole_copies{0}, chunks{0};

static thread_local int countdown = 0;  // the allocation that fails, 0: none

#if !__has_feature(thread_sanitizer)  // (it brings its own)
void* operator new(std::size_t n) {
  if (countdown > 0 && --countdown == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
#endif

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { *p = std::malloc(n); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) { *s = (hipStream_t)s; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)e; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = p == pinned ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  ++whole_copies;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  ++chunks;
  return hipSuccess;
}
}

using namespace mfm::host;

// up and down again, in three segments with a gap between them
static bool round_trip(HostLink& link, unsigned char seed) {
  const size_t n = (size_t)7 << 20;
  std::vector<char> host(n), dev(n), back(n, 1);
  for (size_t i = 0; i < n; ++i) host[i] = (char)(seed + i * 7 + (i >> 12));
  const CopySeg seg[3] = {{0, n / 2}, {n / 2, n / 4 + 13}, {n - 1000, 1000}};
  if (host_copy(link, dev.data(), host.data(), seg, 3, true) != hipSuccess) return false;
  if (host_copy(link, dev.data(), back.data(), seg, 3, false) != hipSuccess) return false;
  for (const CopySeg& s : seg)
    if (std::memcmp(&back[s.off], &host[s.off], s.bytes)) return false;
  const size_t gap = n / 2 + n / 4 + 13;
  for (size_t i = gap; i < n - 1000; ++i)
    if (dev[i] != 0 || back[i] != 1) return false;
  return true;
}

int main(int argc, char** argv) {
  std::atomic<int> bad{0};
  if (argc > 1 && !std::strcmp(argv[1], "pinned")) {
    HostLink link;
    const size_t n = (size_t)6 << 20;
    std::vector<char> host(n, 3), dev(n), other(n);
    const CopySeg all{0, n};
    pinned = host.data();
    if (host_copy(link, dev.data(), host.data(), &all, 1, true) != hipSuccess) ++bad;
    if (whole_copies != 1 || chunks != 0) ++bad;
    if (host_copy(link, dev.data(), other.data(), &all, 1, false) != hipSuccess) ++bad;
    if (whole_copies != 1 || chunks != 3 || std::memcmp(other.data(), host.data(), n)) ++bad;
  } else if (argc > 1 && !std::strcmp(argv[1], "small")) {
    HostLink link;
    const size_t n = (size_t)1 << 20;
    std::vector<char> host(n, 3), dev(n, 5);
    const CopySeg seg[3] = {{100, 1000}, {5000, 70000}, {n - 50, 40}};
    if (host_copy(link, dev.data(), host.data(), seg, 3, false) != hipSuccess) ++bad;
    if (whole_copies != 3) ++bad;
    for (size_t i = 0; i < n; ++i) {
      bool in = false;
      for (const CopySeg& s : seg) in = in || (i >= s.off && i < s.off + s.bytes);
      if (host[i] != (in ? 5 : 3)) { ++bad; break; }
    }
    // the gaps may go along: one copy, nothing outside it
    std::fill(host.begin(), host.end(), (char)3);
    if (host_copy(link, dev.data(), host.data(), seg, 3, false, true) != hipSuccess) ++bad;
    if (whole_copies != 4 || chunks != 0) ++bad;
    for (size_t i = 0; i < n; ++i)
      if (host[i] != (i >= 100 && i < n - 10 ? 5 : 3)) { ++bad; break; }
  } else if (argc > 1 && !std::strcmp(argv[1], "alloc")) {
    HostLink link;
    if (!round_trip(link, 1)) return 1;
    for (int nth = 1; nth <= 4; ++nth) {  // of a copy's allocations
      const size_t n = (size_t)6 << 20;
      std::vector<char> host(n, (char)nth), dev(n);
      const CopySeg all{0, n};
      countdown = nth;
      const hipError_t e = host_copy(link, dev.data(), host.data(), &all, 1, true);
      countdown = 0;
      if (e != hipSuccess || std::memcmp(host.data(), dev.data(), n)) ++bad;
    }
  } else {
    for (int turn = 0; turn < 6; ++turn) {
      HostLink link;  // its first copy makes the pipeline, with others beside it
      std::vector<std::thread> th;
      for (int t = 0; t < 8; ++t)
        th.emplace_back([&, t]() { if (!round_trip(link, (unsigned char)(t + 9 * turn))) ++bad; });
      for (std::thread& t : th) t.join();
    }
  }
  std::printf("%s\n", bad ? "wrong copies" : "copies right");
  return bad ? 1 : 0;
}
