// Runtime part of the C ABI: errors, device memory, streams, events.
#include <cstdio>
#include <cstring>
#include <exception>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

#include "fvm_internal.hpp"

namespace fvm {
namespace {
thread_local std::string g_last_error;
}
void set_error(const std::string& msg) { g_last_error = msg; }
int hip_fail(hipError_t e, const char* what) {
  // reported here: the runtime keeps its last error until it is read, and the next check of a
  // launch, of a caller that goes on after this failure, would take it for its own
  (void)hipGetLastError();
  g_last_error = std::string(what) + ": " + hipGetErrorString(e);
  return e == hipErrorOutOfMemory ? FVM_ERR_ALLOC : FVM_ERR_HIP;
}
const std::string& last_error() { return g_last_error; }

// Device memory: a block of 1 to 128 MiB is kept when it is freed and handed out again for
// the same size on the same device.  hipMalloc and hipFree map and unmap such a block
// (12 us each, measured at 8 and 64 MiB; 0.7 us below 1 MiB, which stay with HIP): a
// gradient of 10^6 nodes, whose five arrays come and go with each call, 213 -> 110 us.
// A free waits for the device first, as hipFree does, so whatever stream used the block
// has finished with it and any stream may have it next.  At most 512 MiB are kept, none
// longer than the next 64 frees, and all are given back when an allocation of the library
// would fail (dev_malloc, for every array).
namespace {
thread_local int64_t g_fail_after = 0, g_fail_count = 0;  // fvm_test_fail_allocations
hipError_t raw_malloc(void** p, size_t bytes) {
  if (g_fail_after > 0) {
    --g_fail_after;
  } else if (g_fail_count > 0) {
    --g_fail_count;
    bytes = (size_t)1 << 60;  // more than any device holds: HIP's own failure
  }
  return hipMalloc(p, bytes > 0 ? bytes : 1);
}

constexpr size_t kKeepMin = (size_t)1 << 20, kKeepMax = (size_t)128 << 20, kKeepTotal = (size_t)512 << 20;
constexpr uint64_t kKeepFrees = 64;
struct Block {
  void* p;
  size_t bytes;
  int dev;
  uint64_t freed;  // number of the free that kept it
};
std::mutex g_mem;
std::unordered_map<void*, Block>* const g_live = new std::unordered_map<void*, Block>;  // handed out, of kept sizes
std::vector<Block>* const g_kept = new std::vector<Block>;  // (never destroyed: frees may come at exit)
size_t g_kept_bytes = 0;
uint64_t g_frees = 0;

// with g_mem held: give back the kept blocks that go(block) names
template <class F>
void give_back(F go) {
  size_t w = 0;
  for (Block& b : *g_kept) {
    if (go(b)) {
      g_kept_bytes -= b.bytes;
      (void)hipFree(b.p);
    } else {
      (*g_kept)[w++] = b;
    }
  }
  g_kept->resize(w);
}
}  // namespace

hipError_t dev_malloc(void** p, size_t bytes) {
  *p = nullptr;
  const hipError_t e = raw_malloc(p, bytes);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  {
    std::lock_guard<std::mutex> lock(g_mem);
    give_back([](const Block&) { return true; });
  }
  return raw_malloc(p, bytes);
}

hipError_t dev_alloc(void** p, size_t bytes) {
  *p = nullptr;
  if (bytes < kKeepMin || bytes > kKeepMax) return dev_malloc(p, bytes);
  Block b{nullptr, (bytes + 0xffff) & ~(size_t)0xffff, 0, 0};
  hipError_t e = hipGetDevice(&b.dev);
  if (e != hipSuccess) return e;
  {
    std::lock_guard<std::mutex> lock(g_mem);
    for (size_t k = g_kept->size(); k-- > 0;) {
      const Block& c = (*g_kept)[k];
      if (c.bytes != b.bytes || c.dev != b.dev) continue;
      b.p = c.p;
      g_kept_bytes -= b.bytes;
      g_kept->erase(g_kept->begin() + (long)k);
      break;
    }
  }
  if (!b.p && (e = dev_malloc(&b.p, b.bytes)) != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_mem);
  try {
    (*g_live)[b.p] = b;
  } catch (const std::exception&) {  // no host memory for the entry
    (void)hipFree(b.p);
    return hipErrorOutOfMemory;
  }
  *p = b.p;
  return hipSuccess;
}

hipError_t dev_free(void* p) {
  if (!p) return hipSuccess;
  int dev = 0;
  {
    std::lock_guard<std::mutex> lock(g_mem);
    auto it = g_live->find(p);
    if (it == g_live->end()) return hipFree(p);
    dev = it->second.dev;
  }
  // the wait outside the lock: other threads allocate and free meanwhile
  int now = 0;
  hipError_t e = hipGetDevice(&now);
  if (e == hipSuccess && now != dev) e = hipSetDevice(dev);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (now != dev) (void)hipSetDevice(now);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(g_mem);
  auto it = g_live->find(p);
  if (it == g_live->end()) return hipErrorInvalidValue;
  Block b = it->second;
  g_live->erase(it);
  b.freed = ++g_frees;
  try {
    g_kept->push_back(b);
  } catch (const std::exception&) {
    return hipFree(p);
  }
  g_kept_bytes += b.bytes;
  // the oldest first (the list is in the order of the frees)
  size_t over = g_kept_bytes > kKeepTotal ? g_kept_bytes - kKeepTotal : 0;
  give_back([&](const Block& c) {
    const bool go = over > 0 || g_frees - c.freed >= kKeepFrees;
    if (go) over -= c.bytes < over ? c.bytes : over;
    return go;
  });
  return hipSuccess;
}

namespace {
thread_local int64_t g_resident_limit = 0;  // fvm_test_resident_limit
std::mutex g_occupancy;
std::map<std::pair<const void*, int>, int64_t>* const g_resident = new std::map<std::pair<const void*, int>, int64_t>;
}  // namespace

hipError_t grid_fits(const void* kernel, int threads, int64_t wgs, bool* fits) {
  *fits = false;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  int64_t most = -1;
  {
    std::lock_guard<std::mutex> lock(g_occupancy);
    const auto it = g_resident->find({kernel, dev});
    if (it != g_resident->end()) most = it->second;
  }
  if (most < 0) {
    int per = 0, cus = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, 0);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    most = (int64_t)per * cus;
    std::lock_guard<std::mutex> lock(g_occupancy);
    try {
      (*g_resident)[{kernel, dev}] = most;
    } catch (const std::exception&) {  // no host memory: asked again the next time
    }
  }
  if (g_resident_limit > 0 && g_resident_limit < most) most = g_resident_limit;
  *fits = wgs <= most;
  return hipSuccess;
}
}  // namespace fvm

extern "C" {

// For tests (not in fvm_hip.h): of the calling thread's following device allocations the first
// `after` are made as usual and the next `count` attempts fail as without memory.
void fvm_test_fail_allocations(int64_t after, int64_t count) {
  fvm::g_fail_after = after;
  fvm::g_fail_count = count;
}

// And: the device holds at most wgs workgroups of the kernels that need to be resident, for the
// calling thread (0: what it does hold).
void fvm_test_resident_limit(int64_t wgs) { fvm::g_resident_limit = wgs; }

int fvm_last_error(char* buf, size_t n) {
  if (!buf || n == 0) return FVM_ERR_ARG;
  const std::string& s = fvm::last_error();
  size_t k = s.size() < n - 1 ? s.size() : n - 1;
  std::memcpy(buf, s.data(), k);
  buf[k] = 0;
  return FVM_OK;
}

int fvm_build_info(char* buf, size_t n) {
  FVM_CHECK(buf && n > 0, "fvm_build_info: null buffer");
  std::snprintf(buf, n, "gfx950 rhs_rev=%d geo_level=%d solver_threads=%d spmv_rows=%d", FVM_RHS_REV,
                FVM_GEO_LEVEL, FVM_SOLVER_THREADS, FVM_SPMV_ROWS);
  return FVM_OK;
}

int fvm_device_count(int* n) {
  FVM_CHECK(n, "fvm_device_count: null output");
  hipError_t e = hipGetDeviceCount(n);
  if (e != hipSuccess) {
    *n = 0;
    return fvm::hip_fail(e, "hipGetDeviceCount");
  }
  return FVM_OK;
}

int fvm_device_synchronize(void) {
  FVM_HIP(hipDeviceSynchronize());
  return FVM_OK;
}

int fvm_alloc(void** d_ptr, size_t bytes) {
  FVM_CHECK(d_ptr, "fvm_alloc: null output");
  *d_ptr = nullptr;
  FVM_HIP(fvm::dev_alloc(d_ptr, bytes));
  return FVM_OK;
}

int fvm_free(void* d_ptr) {
  if (!d_ptr) return FVM_OK;
  FVM_HIP(fvm::dev_free(d_ptr));
  return FVM_OK;
}

int fvm_memcpy_h2d(void* d_dst, const void* src, size_t bytes, fvm_stream s) {
  if (bytes == 0) return FVM_OK;
  FVM_CHECK(d_dst && src, "fvm_memcpy_h2d: null pointer");
  FVM_HIP(hipMemcpyAsync(d_dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)s));
  FVM_HIP(hipStreamSynchronize((hipStream_t)s));
  return FVM_OK;
}

int fvm_memcpy_d2h(void* dst, const void* d_src, size_t bytes, fvm_stream s) {
  if (bytes == 0) return FVM_OK;
  FVM_CHECK(dst && d_src, "fvm_memcpy_d2h: null pointer");
  FVM_HIP(hipMemcpyAsync(dst, d_src, bytes, hipMemcpyDeviceToHost, (hipStream_t)s));
  FVM_HIP(hipStreamSynchronize((hipStream_t)s));
  return FVM_OK;
}

int fvm_memcpy_d2d(void* d_dst, const void* d_src, size_t bytes, fvm_stream s) {
  if (bytes == 0) return FVM_OK;
  FVM_CHECK(d_dst && d_src, "fvm_memcpy_d2d: null pointer");
  FVM_HIP(hipMemcpyAsync(d_dst, d_src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)s));
  return FVM_OK;
}

int fvm_memset(void* d_dst, int value, size_t bytes, fvm_stream s) {
  if (bytes == 0) return FVM_OK;
  FVM_CHECK(d_dst, "fvm_memset: null pointer");
  FVM_HIP(hipMemsetAsync(d_dst, value, bytes, (hipStream_t)s));
  return FVM_OK;
}

int fvm_stream_create(fvm_stream* s) {
  FVM_CHECK(s, "fvm_stream_create: null output");
  hipStream_t h;
  FVM_HIP(hipStreamCreateWithFlags(&h, hipStreamNonBlocking));
  *s = h;
  return FVM_OK;
}

int fvm_stream_destroy(fvm_stream s) {
  if (!s) return FVM_OK;
  FVM_HIP(hipStreamDestroy((hipStream_t)s));
  return FVM_OK;
}

int fvm_stream_synchronize(fvm_stream s) {
  FVM_HIP(hipStreamSynchronize((hipStream_t)s));
  return FVM_OK;
}

int fvm_event_create(fvm_event* e) {
  FVM_CHECK(e, "fvm_event_create: null output");
  hipEvent_t h;
  FVM_HIP(hipEventCreate(&h));
  *e = h;
  return FVM_OK;
}

int fvm_event_destroy(fvm_event e) {
  if (!e) return FVM_OK;
  FVM_HIP(hipEventDestroy((hipEvent_t)e));
  return FVM_OK;
}

int fvm_event_record(fvm_event e, fvm_stream s) {
  FVM_CHECK(e, "fvm_event_record: null event");
  FVM_HIP(hipEventRecord((hipEvent_t)e, (hipStream_t)s));
  return FVM_OK;
}

int fvm_event_elapsed_ms(float* ms, fvm_event start, fvm_event stop) {
  FVM_CHECK(ms && start && stop, "fvm_event_elapsed_ms: null argument");
  FVM_HIP(hipEventSynchronize((hipEvent_t)stop));
  FVM_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
  return FVM_OK;
}

}  // extern "C"
