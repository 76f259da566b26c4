// A HIP runtime that runs nothing: device memory is host memory, launches and attribute settings are
// printed.  Loaded globally ahead of libpowspec_amd.so it takes the place of the real one, so that the
// host code can be followed on any machine, with any number of devices.
#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct Dim3 { uint32_t x, y, z; };
thread_local int device = 0;
thread_local Dim3 grid, block;
thread_local size_t shared;
thread_local void* stream;
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
const char* name(const void* f) { return names()[f].c_str(); }
}  // namespace

extern "C" {
void fake_set_device(int d) { device = d; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* dev, unsigned, void*, void*, void*, void*, int*) {
  names()[host] = dev;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t s, void* st) {
  grid = g, block = b, shared = s, stream = st;
  return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* s, void** st) {
  *g = grid, *b = block, *s = shared, *st = stream;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3, Dim3, void**, size_t s, void*) {
  printf("launch %d %zu %s\n", device, s, name(f));
  return 0;
}
int hipFuncSetAttribute(const void* f, int, int v) {
  printf("attribute %d %d %s\n", device, v, name(f));
  return 0;
}
int hipGetDevice(int* d) { *d = device; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return 0; }
int hipMalloc(void** p, size_t n) { *p = malloc(n); return 0; }
int hipFree(void* p) { free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); return 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void*, const void*, size_t, int, void*) { return 0; }
int hipGetSymbolAddress(void** p, const void*) { static char c[1]; *p = c; return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "fake"; }
int hipEventCreate(void** e) { *e = malloc(1); return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = malloc(1); return 0; }
int hipEventDestroy(void* e) { free(e); return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipStreamIsCapturing(void*, int* s) { *s = 0; return 0; }
}
