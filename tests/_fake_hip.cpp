// A HIP runtime without a GPU, for tests of libhk.so's host code: loaded with
// RTLD_GLOBAL before the library, its functions take the place of the ones the
// library imports.  "Device" memory is host memory and no kernel runs.
//
// What it checks is order.  Work on a stream is done when something waits for
// that stream, as late as the runtime may leave it: a copy from pinned memory
// reads its source then, and a memset of device memory (which the runtime may
// leave running on the null stream) writes then.  The counters are of the uses
// that a wait is missing for: a source changed or freed before its copy was
// done, and a launch on a non-blocking stream while a memset is in flight.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <functional>
#include <list>
#include <map>
#include <string>
#include <vector>

namespace {

struct Pending {
  hipStream_t stream;
  const char* src;             // pinned source, or null (a memset)
  std::vector<char> snapshot;  // what the source held when the copy was queued
  std::function<void()> run;
};

struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} call;

std::list<Pending> queue;
std::map<char*, size_t> pinned;
std::map<char*, size_t> device;
long early_sources = 0, early_launches = 0, fail_in = -1, fail_malloc_in = -1;
hipError_t last = hipSuccess;

hipError_t note(hipError_t err) {
  if (err != hipSuccess) last = err;
  return err;
}

bool inside(const std::map<char*, size_t>& m, const void* p) {
  auto it = m.upper_bound(const_cast<char*>(static_cast<const char*>(p)));
  if (it == m.begin()) return false;
  --it;
  return static_cast<const char*>(p) < it->first + it->second;
}

void finish(const std::function<bool(hipStream_t)>& which) {
  for (auto it = queue.begin(); it != queue.end();) {
    if (!which(it->stream)) {
      ++it;
      continue;
    }
    if (it->src && std::memcmp(it->src, it->snapshot.data(), it->snapshot.size())) ++early_sources;
    it->run();
    it = queue.erase(it);
  }
}
void finish_all() {
  finish([](hipStream_t) { return true; });
}
void finish_stream(hipStream_t s) {
  finish([s](hipStream_t q) { return q == s; });
}

}  // namespace

extern "C" {

long fake_early_sources() { return early_sources; }
long fake_early_launches() { return early_launches; }
// The launch after the next `n` fails; -1: none.
void fake_fail_launch(long n) { fail_in = n; }
// The hipMalloc after the next `n` fails; -1: none.
void fake_fail_malloc_after(long n) { fail_malloc_in = n; }
// Bytes of device memory in use.
long fake_device_bytes() {
  long n = 0;
  for (auto& d : device) n += (long)d.second;
  return n;
}

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char* block = static_cast<char*>(std::calloc(1, 4 << 20));
  return *p = block, hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  *p = nullptr;
  if (fail_malloc_in >= 0 && fail_malloc_in-- == 0) return note(hipErrorOutOfMemory);
  *p = std::calloc(1, n ? n : 1);
  device[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  finish_all();
  device.erase(static_cast<char*>(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(1, n ? n : 1);
  pinned[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  auto it = pinned.find(static_cast<char*>(p));
  for (auto& q : queue)
    if (it != pinned.end() && q.src >= it->first && q.src < it->first + it->second) ++early_sources;
  finish_all();
  pinned.erase(static_cast<char*>(p));
  std::free(p);
  return hipSuccess;
}

hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
  const char* from = static_cast<const char*>(src);
  Pending q{s, nullptr, {}, [=] { std::memmove(dst, from, n); }};
  if (inside(pinned, src)) {
    q.src = from;
    q.snapshot.assign(from, from + n);
  } else if (!inside(device, src)) {  // pageable: the runtime has its own copy when the call returns
    std::vector<char> own(from, from + n);
    q.run = [=] { std::memcpy(dst, own.data(), n); };
  }
  queue.push_back(std::move(q));
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* dst, size_t dp, const void* src, size_t sp, size_t w, size_t h, hipMemcpyKind,
                            hipStream_t s) {
  queue.push_back({s, nullptr, {}, [=] {
                     for (size_t r = 0; r < h; ++r)
                       std::memmove(static_cast<char*>(dst) + r * dp, static_cast<const char*>(src) + r * sp, w);
                   }});
  return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind) {
  finish_stream(nullptr);
  std::memmove(dst, src, n);
  return hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) {
  queue.push_back({nullptr, nullptr, {}, [=] { std::memset(p, v, n); }});
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) {
  queue.push_back({s, nullptr, {}, [=] { std::memset(p, v, n); }});
  return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  static long next = 0x1000;
  return *s = reinterpret_cast<hipStream_t>(next += 16), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return finish_stream(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return finish_stream(s), hipSuccess; }
hipError_t hipDeviceSynchronize() { return finish_all(), hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  call = {grid, block, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = call.grid, *block = call.block, *lds = call.lds, *s = call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t s) {
  if (s != nullptr)
    for (auto& q : queue)
      if (q.stream == nullptr) {
        ++early_launches;
        break;
      }
  if (fail_in >= 0 && fail_in-- == 0) return note(hipErrorLaunchFailure);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t err = last;
  last = hipSuccess;
  return err;
}
}
