// A HIP runtime for one GPU in host memory, linked into a test program ahead of
// the real one: what libnoptjk.so does on the host (allocations, routes, launch
// shapes, error paths) then runs without a GPU. Device memory is zeroed host
// memory, copies and clears move bytes, kernels are recorded and not run.
#include "fake_hip.hpp"

#include <cstdlib>
#include <cstring>
#include <map>

namespace fake {
std::map<void*, size_t> blocks;
std::map<const void*, std::string>& kernels() {  // filled while the library loads, before this file's globals
  static std::map<const void*, std::string> m;
  return m;
}
std::vector<Launch> launches;
size_t live = 0;
int mallocs = 0, fail_at = 0, pinned = 0, pinned_live = 0;
float elapsed = 1e6f;
}  // namespace fake

using fake::Dim3;

namespace {
constexpr int kOk = 0, kInvalidValue = 1, kOutOfMemory = 2;
struct {
  Dim3 grid, block;
  size_t shared;
  void* stream;
} config;

int copy(void* d, const void* s, size_t n) {
  if (!n) return kOk;
  if (!d || !s) return kInvalidValue;
  std::memcpy(d, s, n);
  return kOk;
}
}  // namespace

extern "C" {
int hipGetDeviceCount(int* n) { return *n = 1, kOk; }
int hipSetDevice(int d) { return d == 0 ? kOk : kInvalidValue; }
int hipDeviceGetAttribute(int* v, int, int) { return *v = 256, kOk; }  // the library asks for the compute units
int hipDeviceSynchronize() { return kOk; }
int hipGetLastError() { return kOk; }
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }

int hipMalloc(void** p, size_t bytes) {
  if (++fake::mallocs == fake::fail_at) return kOutOfMemory;
  *p = std::calloc(bytes ? bytes : 1, 1);
  fake::blocks[*p] = bytes;
  fake::live += bytes;
  return kOk;
}
int hipFree(void* p) {
  if (!p) return kOk;
  const auto it = fake::blocks.find(p);
  if (it == fake::blocks.end()) std::abort();
  fake::live -= it->second;
  fake::blocks.erase(it);
  std::free(p);
  return kOk;
}
int hipHostMalloc(void** p, size_t bytes, unsigned) {
  ++fake::pinned;
  ++fake::pinned_live;
  return *p = std::calloc(bytes, 1), kOk;
}
int hipHostFree(void* p) {
  --fake::pinned_live;
  return std::free(p), kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int) { return copy(d, s, n); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { return copy(d, s, n); }
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void*) {
  int rc = kOk;
  for (size_t r = 0; r < h && !rc; ++r) rc = copy((char*)d + r * dp, (const char*)s + r * sp, w);
  return rc;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  if (!d) return kInvalidValue;
  // large buffers are zero already (no kernel writes): their pages stay untouched
  if (v || n < ((size_t)1 << 20)) std::memset(d, v, n);
  return kOk;
}

int hipStreamCreateWithFlags(void** s, unsigned) { return *s = std::malloc(1), kOk; }
int hipStreamDestroy(void* s) { return std::free(s), kOk; }
int hipStreamSynchronize(void*) { return kOk; }
int hipStreamWaitEvent(void*, void*, unsigned) { return kOk; }
int hipEventCreate(void** e) { return *e = std::malloc(1), kOk; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = std::malloc(1), kOk; }
int hipEventDestroy(void* e) { return std::free(e), kOk; }
int hipEventRecord(void*, void*) { return kOk; }
int hipEventSynchronize(void*) { return kOk; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = fake::elapsed -= 1.f, kOk; }  // ever faster

int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
  config = {grid, block, shared, stream};
  return kOk;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return kOk;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void**, size_t, void* stream) {
  fake::launches.push_back({fake::kernels()[f], grid, stream});
  return kOk;
}
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, Dim3*, Dim3*,
                           int*) {
  fake::kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
}
