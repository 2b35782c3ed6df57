// A HIP runtime on the host for checks of the library's host code: linked into
// an executable beside libcsaw.so, its functions take the place of the real
// runtime's.  Device memory is host memory (zero until written, reserved and not
// committed), copies beyond kCopyMax are left out, kernels do nothing but be
// written down by name, except the ones that a check needs the results of
// (k_degree).  A check sets the device count, the memory a device has, and which
// call of a function fails.
#pragma once
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

struct FakeHip {
  static constexpr size_t kCopyMax = size_t(1) << 30;
  int device = 0;                        // the current one
  std::map<std::string, long> fail_in;   // fail_in[f] = k: the k-th call of f from now on fails
  size_t limit = SIZE_MAX, used = 0;     // device memory, of all devices together
  struct Alloc {
    size_t bytes;
    int device;
  };
  std::map<void*, Alloc> mem;
  std::map<const void*, std::string> kernel;
  std::vector<std::string> log;  // kernels launched, and what waits
  std::vector<size_t> allocs;    // sizes asked of hipMalloc
  float ms = 1.0f;               // next hipEventElapsedTime, and what each takes off it
  float ms_step = 0.0f;
  uintptr_t handles = 0;

  bool fails(const char* f) {
    auto it = fail_in.find(f);
    return it != fail_in.end() && it->second > 0 && --it->second == 0;
  }
  void note(const std::string& s) { log.push_back(s); }
  bool logged(const std::string& part) const {
    for (const std::string& s : log)
      if (s.find(part) != std::string::npos) return true;
    return false;
  }
  template <class H>
  H handle() {
    return reinterpret_cast<H>(++handles * 16);
  }
};

inline FakeHip& fake() {
  static FakeHip* f = new FakeHip;
  return *f;
}

extern "C" {
struct FakeCall {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
static FakeCall g_call;

void** __hipRegisterFatBinary(const void*) {
  static void* x;
  return &x;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  fake().kernel[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_call = {grid, block, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_call.grid;
  *block = g_call.block;
  *lds = g_call.lds;
  *s = g_call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t) {
  const std::string& name = fake().kernel[f];
  fake().note(name + " grid " + std::to_string(grid.x));
  if (name.find("k_degree") != std::string::npos) {
    const int64_t* off = *(const int64_t**)args[0];
    const int64_t V = *(int64_t*)args[1];
    int32_t* deg = *(int32_t**)args[2];
    unsigned long long* mx = *(unsigned long long**)args[3];
    for (int64_t v = 0; v < V; ++v) {
      deg[v] = (int32_t)(off[v + 1] - off[v]);
      if ((unsigned long long)deg[v] > *mx) *mx = (unsigned long long)deg[v];
    }
  }
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = fake().device;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  fake().device = d;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  FakeHip& f = fake();
  if (f.fails("hipMalloc as unsupported")) return hipErrorStreamCaptureUnsupported;
  if (f.fails("hipMalloc") || n > f.limit - f.used) return hipErrorOutOfMemory;
  void* q = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (q == MAP_FAILED) return hipErrorOutOfMemory;
  f.mem[q] = {n, f.device};
  f.used += n;
  f.allocs.push_back(n);
  *p = q;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  FakeHip& f = fake();
  auto it = f.mem.find(p);
  if (it == f.mem.end()) return p ? hipErrorInvalidValue : hipSuccess;
  f.note("free on " + std::to_string(it->second.device));
  f.used -= it->second.bytes;
  munmap(p, it->second.bytes);
  f.mem.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  if (fake().fails("hipMemcpy")) return hipErrorUnknown;
  if (n <= FakeHip::kCopyMax) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (fake().fails("hipMemcpyAsync")) return hipErrorUnknown;
  if (n <= FakeHip::kCopyMax) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  if (n <= FakeHip::kCopyMax) memset(d, v, n);
  return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
  FakeHip& f = fake();
  f.note("wait for device " + std::to_string(f.device));
  return f.fails("hipDeviceSynchronize") ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  fake().note("wait for stream");
  return fake().fails("hipStreamSynchronize") ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  if (fake().fails("hipStreamCreateWithFlags")) return hipErrorOutOfMemory;
  *s = fake().handle<hipStream_t>();
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) { return e ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventCreate(hipEvent_t* e) {
  if (fake().fails("hipEventCreate")) return hipErrorOutOfMemory;
  *e = fake().handle<hipEvent_t>();
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  if (fake().fails("hipEventCreateWithFlags")) return hipErrorOutOfMemory;
  *e = fake().handle<hipEvent_t>();
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { return e ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = fake().ms;
  fake().ms -= fake().ms_step;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char scratch[64];
  *p = scratch;
  return hipSuccess;
}
}
