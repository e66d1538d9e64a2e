// A stand-in for the HIP runtime that runs no kernel and writes down the calls
// that mpm_amd's host code makes: loaded with RTLD_GLOBAL before libmpmx.so in
// a process of its own, it takes the place of libamdhip64. Device memory is host
// memory; launches, graphs and events are names in the log (hip_record_log).
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
// never destroyed: the library's own teardown still calls in here
std::string& g_log = *new std::string;
std::map<const void*, std::string>& g_names = *new std::map<const void*, std::string>;
std::map<void*, size_t>& g_size = *new std::map<void*, size_t>;
size_t g_device = 0, g_pinned = 0;  // bytes held now
int g_current = 0;                  // of two devices
bool g_capturing = false;
int g_handles = 0;

void note(const std::string& s) { g_log += s + "\n"; }
// Whether [p, p + n) lies in one allocation, or in none at all (host memory).
bool in_bounds(const void* p, size_t n) {
  auto it = g_size.upper_bound(const_cast<void*>(p));
  if (it == g_size.begin()) return true;
  --it;
  const char *a = static_cast<char*>(it->first), *q = static_cast<const char*>(p);
  return q >= a + it->second || q + n <= a + it->second;
}
void* handle() { return reinterpret_cast<void*>(static_cast<uintptr_t>(16 * ++g_handles)); }
}  // namespace

struct Dim3 {
  uint32_t x, y, z;
};

extern "C" {
const char* hip_record_log() { return g_log.c_str(); }
void hip_record_clear() { g_log.clear(); }
size_t hip_record_device_bytes() { return g_device; }
size_t hip_record_pinned_bytes() { return g_pinned; }

void** __hipRegisterFatBinary(const void*) {
  static void* one = nullptr;
  return &one;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*,
                           void*, void*, void*, int*) {
  g_names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* shared, void** stream) {
  *g = *b = Dim3{1, 1, 1};
  *shared = 0;
  *stream = nullptr;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t, void*) {
  note((g_capturing ? "captured " : "launch ") + g_names[f] +
       (g_current ? " on the other device" : ""));
  return 0;
}

int hipMalloc(void** p, size_t n) {
  *p = std::calloc(n ? n : 1, 1);
  g_size[*p] = n;
  g_device += n;
  note("malloc " + std::to_string(n) + (g_current ? " on the other device" : ""));
  return *p ? 0 : 2;
}
int hipFree(void* p) {
  g_device -= g_size[p];
  g_size.erase(p);
  std::free(p);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(n ? n : 1, 1);
  g_size[*p] = n;
  g_pinned += n;
  note("pinned " + std::to_string(n));
  return *p ? 0 : 2;
}
int hipHostFree(void* p) {
  g_pinned -= g_size[p];
  g_size.erase(p);
  std::free(p);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) {
  if (!in_bounds(d, n) || !in_bounds(s, n)) {
    note("out_of_bounds copy of " + std::to_string(n));
    return 1;
  }
  std::memcpy(d, s, n);
  if (kind == 2) note("to_host " + std::to_string(n));
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  if (!in_bounds(d, n)) {
    note("out_of_bounds set of " + std::to_string(n));
    return 1;
  }
  std::memset(d, v, n);
  return 0;
}
int hipGetSymbolAddress(void** p, const void*) {
  *p = handle();  // never dereferenced: no kernel runs
  return 0;
}

int hipEventCreate(void** e) {
  *e = handle();
  return 0;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void* e, void*) {
  note("event " + std::to_string(reinterpret_cast<uintptr_t>(e)));
  return 0;
}
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 1.f;
  return 0;
}
int hipGetDevice(int* d) {
  *d = g_current;
  return 0;
}
int hipSetDevice(int d) {
  g_current = d;
  return 0;
}
int hipGetDeviceCount(int* n) {
  *n = 2;
  return 0;
}
const char* hipGetErrorString(int) { return "recorded"; }
int hipGetLastError() { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) {
  *s = handle();
  return 0;
}
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamBeginCapture(void*, int) {
  g_capturing = true;
  note("begin_capture");
  return 0;
}
int hipStreamEndCapture(void*, void** g) {
  g_capturing = false;
  *g = handle();
  return 0;
}
int hipGraphInstantiate(void** e, void*, void*, char*, size_t) {
  note("instantiate");
  *e = handle();
  return 0;
}
int hipGraphLaunch(void*, void*) {
  note("graph");
  return 0;
}
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }
}
