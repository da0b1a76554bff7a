// Test-only stand-in for the HIP runtime, for tests of the library's host code
// on a machine without a GPU.  Loaded with global symbols before
// libthrml_hip.so, whose HIP calls then bind here.
//
//   - One device.  "Device" memory is host memory, reserved and not touched
//     until used, with a capacity that a test can set.
//   - One queue for all streams.  Copies and fills wait in it until something
//     synchronises; a copy that is still in it when a call returns would read or
//     write the caller's memory later (fake_pending_host counts those).
//   - Kernels do not run (state imports are taken as accepted).  Each launch is counted under the kernel's name; a
//     launch of no workgroup or of 2^32 threads or more is an error.
#define __HIP_PLATFORM_AMD__ 1
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Op {
  void *dst;
  const void *src;  // null: a fill with `value`
  size_t n;
  int value;
  bool host;        // reads or writes memory that is not the device's
};

std::mutex mu;
std::vector<Op> queue;
std::map<uintptr_t, size_t> blocks;
size_t capacity = ~(size_t)0, live = 0;
uint64_t n_malloc = 0, fail_at = 0;  // fail_at: the allocations from which on all fail
int cus = 256;
std::map<const void *, std::string> names;
std::map<std::string, uint64_t> launches;
void (*on_launch)() = nullptr;
thread_local hipError_t last = hipSuccess;
constexpr size_t BIG = 64u << 20;  // larger fills are left out

hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}

bool on_device(const void *p) {
  const auto it = blocks.upper_bound((uintptr_t)p);
  if (it == blocks.begin()) return false;
  const auto b = std::prev(it);
  return (uintptr_t)p < b->first + b->second;
}

void drain() {
  for (const Op &o : queue) {
    if (o.src) memcpy(o.dst, o.src, o.n);
    else if (o.n <= BIG) memset(o.dst, o.value, o.n);
  }
  queue.clear();
}

struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
thread_local Config config;

}  // namespace

extern "C" {

// ---- for the tests
void fake_reset() {
  capacity = ~(size_t)0;
  fail_at = 0;
  cus = 256;
  last = hipSuccess;
  on_launch = nullptr;
  launches.clear();
}
void fake_set_capacity(uint64_t bytes) { capacity = bytes; }
void fake_fail_malloc(uint64_t nth) { fail_at = nth ? n_malloc + nth : 0; }  // 1: from the next one on; 0: none
void fake_set_cus(int n) { cus = n; }
uint64_t fake_live_bytes() { return live; }
uint64_t fake_mallocs() { return n_malloc; }
uint64_t fake_pending_host() {
  std::lock_guard<std::mutex> lk(mu);
  uint64_t n = 0;
  for (const Op &o : queue) n += o.host;
  return n;
}
void fake_on_launch(void (*f)()) { on_launch = f; }
void fake_clear_launches() {
  std::lock_guard<std::mutex> lk(mu);
  launches.clear();
}
// "name count" per line; the length needed
uint64_t fake_launches(char *buf, uint64_t n) {
  std::lock_guard<std::mutex> lk(mu);
  std::string s;
  for (const auto &l : launches) s += l.first + " " + std::to_string(l.second) + "\n";
  if (buf && n > s.size()) memcpy(buf, s.c_str(), s.size() + 1);
  return s.size() + 1;
}

// ---- device, memory
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) { return ret(d == 0 ? hipSuccess : hipErrorInvalidDevice); }
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  memset(p, 0, sizeof *p);
  p->multiProcessorCount = cus;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) {
  return e == hipSuccess ? "no error" : e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  ++n_malloc;
  if ((fail_at && n_malloc >= fail_at) || live + n > capacity) return ret(hipErrorOutOfMemory);
  void *m = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (m == MAP_FAILED) return ret(hipErrorOutOfMemory);
  blocks[(uintptr_t)m] = n;
  live += n;
  *p = m;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  if (!p) return hipSuccess;
  const auto b = blocks.find((uintptr_t)p);
  if (b == blocks.end()) return ret(hipErrorInvalidValue);
  drain();
  live -= b->second;
  munmap(p, b->second);
  blocks.erase(b);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  queue.push_back(Op{dst, src, n, 0, !on_device(dst) || !on_device(src)});
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *dst, size_t dp, const void *src, size_t sp, size_t w, size_t h, hipMemcpyKind,
                            hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  for (size_t r = 0; r < h; ++r)
    queue.push_back(Op{(char *)dst + r * dp, (const char *)src + r * sp, w, 0, !on_device(dst) || !on_device(src)});
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int value, size_t n, hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  queue.push_back(Op{dst, nullptr, n, value, !on_device(dst)});
  return hipSuccess;
}

// ---- streams, events
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int) {
  *s = (hipStream_t) new char;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  delete (char *)s;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> lk(mu);
  drain();
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned int) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  *s = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t) new char;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (char *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
  *ms = 0.0f;
  return hipSuccess;
}

// ---- kernels
void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned int, void *, void *, void *,
                           void *, int *) {
  int st = 0;
  char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
  std::string s = d ? d : name;
  free(d);
  // "void thrml::kernel<2, unsigned char>(thrml::Args)" -> "kernel<2,unsigned_char>"
  s = s.substr(0, s.find('('));
  const size_t lt = s.find('<'), at = s.rfind("thrml::", lt);
  if (at != std::string::npos) s = s.substr(at + 7);
  std::string o;
  for (size_t i = 0; i < s.size(); ++i) {
    if (s[i] == ' ' && i && s[i - 1] == ',') continue;
    o += s[i] == ' ' ? '_' : s[i];
  }
  std::lock_guard<std::mutex> lk(mu);
  names[host] = o;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static void *mem = nullptr;
  if (!mem) {
    const hipError_t e = hipMalloc(&mem, 64u << 20);
    if (e != hipSuccess) return e;
  }
  *p = mem;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  config = Config{g, b, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = config.grid;
  *b = config.block;
  *lds = config.lds;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t) {
  {
    std::lock_guard<std::mutex> lk(mu);
    const uint64_t t = (uint64_t)g.x * b.x;
    if (t == 0 || t >= (1ull << 32)) return ret(hipErrorInvalidConfiguration);
    const std::string name = names.count(f) ? names[f] : "?";
    ++launches[name];
    // an import is accepted: its check leaves what this kernel writes
    if (name == "import_reset_kernel") queue.push_back(Op{*(void **)args[0], nullptr, 4, 0xff, false});
  }
  if (on_launch) on_launch();
  return hipSuccess;
}
}
