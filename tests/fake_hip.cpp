// Host stand-in for the HIP runtime: "device" memory is host memory, copies are
// memcpy, kernels do not run but are recorded by name.  Loaded before
// libculbm.so it takes the place of the runtime's symbols, so the host side of
// the C ABI (routes, memory accounting, error paths) runs without a GPU.
#include <dirent.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include <vector>

namespace {

constexpr int kOk = 0, kOutOfMemory = 2, kInvalidValue = 1, kInvalidDevice = 101;

std::map<void*, size_t> g_held;
size_t g_bytes = 0, g_limit = size_t(1) << 40;
std::map<const void*, std::string> g_names;
std::string g_log;  // names of the kernels launched, one a line
std::vector<uint32_t> g_grids;
long g_copies = 0, g_largest = 0;  // device-to-host copies
int g_threads = 0;                 // most threads seen while one was waited for
char* g_known = nullptr;           // a range that hipPointerGetAttributes knows
size_t g_known_bytes = 0;

struct Dim3 {
  uint32_t x, y, z;
};

}  // namespace

extern "C" {
long fake_new_left = -1;  // allocations until one fails (-1: none does); -1 again afterwards
}

void* operator new(size_t n) {
  if (fake_new_left >= 0 && fake_new_left-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {
// The stand-in's own allocations never fail.
struct Immune {
  long left = fake_new_left;
  Immune() { fake_new_left = -1; }
  ~Immune() { fake_new_left = left; }
};
}  // namespace

extern "C" {

// ---- control
void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_bytes() { return g_bytes; }
const char* fake_log() { return g_log.c_str(); }
long fake_grid(long k) { return k < long(g_grids.size()) ? long(g_grids[size_t(k)]) : -1; }
long fake_copies() { return g_copies; }
long fake_largest() { return g_largest; }
int fake_threads() { return g_threads; }
void fake_fail_new(long after) { fake_new_left = after; }
void fake_known(void* p, size_t bytes) {
  g_known = static_cast<char*>(p);
  g_known_bytes = bytes;
}
void fake_clear() {
  g_log.clear();
  g_grids.clear();
  g_copies = g_largest = 0;
  g_threads = 0;
}

// ---- modules and launches
void** __hipRegisterFatBinary(const void*) {
  static void* h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3, size_t, void*) {
  Immune immune;
  g_grids.push_back(grid.x);
  return kOk;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
  *grid = *block = {1, 1, 1};
  *shared = 0;
  *stream = nullptr;
  return kOk;
}
int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t, void*) {
  Immune immune;
  g_log += g_names.count(f) ? g_names[f] : std::string("?");
  g_log += '\n';
  return kOk;
}

// ---- memory
int hipMalloc(void** p, size_t n) {
  if (g_bytes + n > g_limit) return kOutOfMemory;
  *p = std::calloc(n ? n : 1, 1);
  if (!*p) return kOutOfMemory;
  Immune immune;
  g_held[*p] = n;
  g_bytes += n;
  return kOk;
}
int hipFree(void* p) {
  const auto it = g_held.find(p);
  if (it == g_held.end()) return p ? kInvalidValue : kOk;
  g_bytes -= it->second;
  g_held.erase(it);
  std::free(p);
  return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return *p ? kOk : kOutOfMemory;
}
int hipHostFree(void* p) {
  std::free(p);
  return kOk;
}
int hipMemGetInfo(size_t* fr, size_t* total) {
  *fr = g_limit > g_bytes ? g_limit - g_bytes : 0;
  *total = g_limit;
  return kOk;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) {
  if (kind == 2) {
    ++g_copies;
    if (long(n) > g_largest) g_largest = long(n);
  }
  std::memcpy(d, s, n);
  return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) { return hipMemcpyAsync(d, s, n, kind, nullptr); }
// Any type but "unregistered" (0) for the known range; an error for the rest, as
// the runtime gives for memory it has not seen.
int hipPointerGetAttributes(void* attr, const void* p) {
  const char* c = static_cast<const char*>(p);
  if (!g_known || c < g_known || c >= g_known + g_known_bytes) return kInvalidValue;
  *static_cast<int*>(attr) = 1;  // the first member: hipMemoryTypeHost
  return kOk;
}
int hipGetSymbolAddress(void** p, const void*) {
  static double scratch[8192];
  *p = scratch;
  return kOk;
}

// ---- devices, streams, events, graphs
int hipGetDeviceCount(int* n) {
  *n = 1;
  return kOk;
}
int hipSetDevice(int) { return kOk; }
int hipGetDevicePropertiesR0600(void*, int) { return kInvalidDevice; }  // the library then assumes 256 CUs
int hipDeviceSynchronize() { return kOk; }
int hipGetLastError() { return kOk; }
const char* hipGetErrorString(int) { return "error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = reinterpret_cast<void*>(8);
  return kOk;
}
int hipStreamDestroy(void*) { return kOk; }
int hipStreamSynchronize(void*) { return kOk; }
int hipEventCreate(void** e) {
  *e = reinterpret_cast<void*>(8);
  return kOk;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) { return kOk; }
int hipEventRecord(void*, void*) { return kOk; }
int hipEventSynchronize(void*) {
  int n = 0;
  if (DIR* d = opendir("/proc/self/task")) {
    while (const dirent* e = readdir(d)) n += e->d_name[0] != '.';
    closedir(d);
  }
  if (n > g_threads) g_threads = n;
  return kOk;
}
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 1.0f;
  return kOk;
}
int hipStreamBeginCapture(void*, int) { return kOk; }
int hipStreamEndCapture(void*, void** g) { return hipEventCreate(g); }
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) { return hipEventCreate(e); }
int hipGraphLaunch(void*, void*) { return kOk; }
int hipGraphDestroy(void*) { return kOk; }
int hipGraphExecDestroy(void*) { return kOk; }

}  // extern "C"
