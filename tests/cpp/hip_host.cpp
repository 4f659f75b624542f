// The HIP runtime calls that libgbr.so makes, over host memory: device and
// pinned memory are malloc, copies are memcpy, kernels do not run.  Loaded
// before libgbr.so (RTLD_GLOBAL), it takes the place of the real runtime, so
// that the library's host code runs without a GPU, every launch can be looked
// at and an allocation can be made to fail (tests/hip_host.py).
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

enum { kSuccess = 0, kInvalidValue = 1, kOutOfMemory = 2 };
enum { kUnregistered = 0, kHost = 1, kDevice = 2 };  // hipMemoryType

struct Block {
  size_t size;
  int type;
};

std::map<uintptr_t, Block> g_blocks;
std::map<const void*, std::string> g_kernels;
std::map<std::string, int64_t> g_calls;
std::map<std::string, int64_t> g_fail;  // calls left until the named one fails (0: the next)
int64_t g_device_limit = -1, g_device_used = 0;
int g_last_error = kSuccess;
void (*g_hook)(const char* kernel, const uint32_t* grid, void** args) = nullptr;

struct Dim3 {
  uint32_t x, y, z;
};
struct {
  Dim3 grid, block;
  size_t shared;
  void* stream;
} g_config;

bool fails(const char* name) {
  ++g_calls[name];
  auto it = g_fail.find(name);
  if (it == g_fail.end()) return false;
  if (it->second-- > 0) return false;
  g_fail.erase(it);
  return true;
}

int allocate(const char* call, void** p, size_t n, int type) {
  *p = nullptr;
  const bool full = type == kDevice && g_device_limit >= 0 && g_device_used + (int64_t)n > g_device_limit;
  void* m = fails(call) || full ? nullptr : calloc(1, n ? n : 1);
  if (!m) return g_last_error = kOutOfMemory;
  g_blocks[(uintptr_t)m] = {n, type};
  if (type == kDevice) g_device_used += (int64_t)n;
  *p = m;
  return kSuccess;
}

int release(void* p) {
  if (!p) return kSuccess;
  auto it = g_blocks.find((uintptr_t)p);
  if (it == g_blocks.end()) return kInvalidValue;
  if (it->second.type == kDevice) g_device_used -= (int64_t)it->second.size;
  g_blocks.erase(it);
  free(p);
  return kSuccess;
}

// the block that holds p, or null
const std::pair<const uintptr_t, Block>* find(const void* p) {
  auto it = g_blocks.upper_bound((uintptr_t)p);
  if (it == g_blocks.begin()) return nullptr;
  --it;
  return (uintptr_t)p < it->first + it->second.size ? &*it : nullptr;
}

}  // namespace

extern "C" {

// ---- for the tests ---------------------------------------------------------
void hip_host_hook(void (*hook)(const char*, const uint32_t*, void**)) { g_hook = hook; }
void hip_host_fail(const char* call, int64_t after) { g_fail[call] = after; }
int64_t hip_host_calls(const char* call) { return g_calls[call]; }
void hip_host_memory(int64_t device_limit) { g_device_limit = device_limit; }
int64_t hip_host_used() { return g_device_used; }
int64_t hip_host_blocks() { return (int64_t)g_blocks.size(); }

// ---- modules -----------------------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  g_kernels[f] = name;
}
std::map<const void*, size_t>& variables() {
  static std::map<const void*, size_t> v;
  return v;
}
void __hipRegisterVar(void**, void* var, char*, const char*, int, size_t size, int, int) { variables()[var] = size; }
int hipGetSymbolAddress(void** p, const void* var) {
  static std::map<const void*, void*> at;
  if (!at.count(var)) at[var] = calloc(1, variables()[var]);
  *p = at[var];
  return kSuccess;
}

// ---- launches ----------------------------------------------------------------
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
  g_config = {grid, block, shared, stream};
  return kSuccess;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = g_config.grid;
  *block = g_config.block;
  *shared = g_config.shared;
  *stream = g_config.stream;
  return kSuccess;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void** args, size_t, void*) {
  if (fails("hipLaunchKernel")) return kInvalidValue;
  const uint32_t g[3] = {grid.x, grid.y, grid.z};
  if (g_hook) g_hook(g_kernels[f].c_str(), g, args);
  return kSuccess;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  *n = 4;
  return kSuccess;
}

// ---- devices, streams, events, graphs ------------------------------------------
int hipGetDeviceCount(int* n) {
  *n = 1;
  return kSuccess;
}
int hipGetDevice(int* d) {
  *d = 0;
  return kSuccess;
}
int hipSetDevice(int) { return kSuccess; }
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return kSuccess;
}
int hipGetLastError() {
  const int e = g_last_error;
  g_last_error = kSuccess;
  return e;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : e ? "error" : "no error"; }
int hipMemGetInfo(size_t* free_bytes, size_t* total) {
  *total = (size_t)(g_device_limit < 0 ? 64ll << 30 : g_device_limit);
  *free_bytes = *total - (size_t)g_device_used;
  return kSuccess;
}
static char g_handle;
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = &g_handle;
  return kSuccess;
}
int hipStreamDestroy(void*) { return kSuccess; }
int hipStreamSynchronize(void*) {
  ++g_calls["hipStreamSynchronize"];
  return kSuccess;
}
int hipStreamBeginCapture(void*, int) { return kSuccess; }
int hipStreamEndCapture(void*, void** graph) {
  *graph = &g_handle;
  return kSuccess;
}
int hipGraphInstantiate(void** exec, void*, void*, char*, size_t) {
  *exec = &g_handle;
  return kSuccess;
}
int hipGraphLaunch(void*, void*) { return kSuccess; }
int hipGraphDestroy(void*) { return kSuccess; }
int hipGraphExecDestroy(void*) { return kSuccess; }
int hipEventCreate(void** e) {
  *e = new char;
  return kSuccess;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
  delete static_cast<char*>(e);
  return kSuccess;
}
// (the hook sees events too: the call's name, and the event as its argument)
int hipEventRecord(void* e, void*) {
  const uint32_t none[3] = {};
  if (g_hook) g_hook("hipEventRecord", none, &e);
  return kSuccess;
}
int hipEventSynchronize(void* e) {
  const uint32_t none[3] = {};
  if (g_hook) g_hook("hipEventSynchronize", none, &e);
  return kSuccess;
}
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 1.0f;
  return kSuccess;
}

// ---- memory --------------------------------------------------------------------
int hipMalloc(void** p, size_t n) { return allocate("hipMalloc", p, n, kDevice); }
int hipFree(void* p) { return release(p); }
int hipHostMalloc(void** p, size_t n, unsigned) { return allocate("hipHostMalloc", p, n, kHost); }
int hipHostFree(void* p) { return release(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) {
  memcpy(d, s, n);
  return kSuccess;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  ++g_calls["hipMemcpyAsync"];
  memcpy(d, s, n);
  return kSuccess;
}
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void*) {
  ++g_calls["hipMemcpy2DAsync"];
  for (size_t y = 0; y < h; ++y) memcpy((char*)d + y * dp, (const char*)s + y * sp, w);
  return kSuccess;
}
int hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return kSuccess;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }
int hipMemsetD32Async(void* d, int v, size_t n, void*) {
  for (size_t i = 0; i < n; ++i) ((int*)d)[i] = v;
  return kSuccess;
}

struct PointerAttributes {  // hipPointerAttribute_t
  int type, device;
  void *device_pointer, *host_pointer;
  int managed;
  unsigned flags;
};
int hipPointerGetAttributes(PointerAttributes* a, const void* p) {
  memset(a, 0, sizeof *a);
  a->device = -2;
  if (const auto* b = find(p)) {
    a->type = b->second.type;
    a->device = 0;
    a->device_pointer = const_cast<void*>(p);
    a->host_pointer = b->second.type == kHost ? const_cast<void*>(p) : nullptr;
  }
  return kSuccess;
}

}  // extern "C"
