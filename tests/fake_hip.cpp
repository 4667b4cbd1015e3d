// A HIP runtime that launches nothing, for tests of libqlin's host side on the CPU: the
// symbols that the library imports, recording the kernels launched and the kernels whose
// occupancy was asked for, by their device names.  Loaded with RTLD_GLOBAL before the
// library (tests/dispatch.py), so that its calls come here.
#include <cstddef>
#include <cstdio>
#include <map>
#include <string>

struct dim3 {
  unsigned x, y, z;
};

namespace {
std::map<const void*, std::string>& names() {
  static auto* m = new std::map<const void*, std::string>;
  return *m;
}
std::string& log() {
  static auto* s = new std::string;
  return *s;
}
struct {
  dim3 grid, block;
  size_t lds;
  void* stream;
} config;
}  // namespace

extern "C" {

const char* fake_log() { return log().c_str(); }
void fake_clear() { log().clear(); }

void** __hipRegisterFatBinary(const void*) {
  static void* handle[1];
  return handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  names()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void* stream) {
  config = {grid, block, lds, stream};
  return 0;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, void** stream) {
  *grid = config.grid, *block = config.block, *lds = config.lds, *stream = config.stream;
  return 0;
}
int hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, void*) {
  char t[96];
  snprintf(t, sizeof t, " %u %u %u\n", grid.x, grid.y, block.x);
  log() += "launch " + names()[f] + t;
  return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int, size_t) {
  log() += "occupancy " + names()[f] + "\n";
  *n = 3;
  return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
  *v = 256;
  return 0;
}
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipFuncSetAttribute(const void*, int, int) { return 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "fake"; }
int hipGetSymbolAddress(void** p, const void*) {
  *p = (void*)0x700000000000;
  return 0;
}
int hipMemcpyAsync(void*, const void*, size_t, int, void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }

}  // extern "C"
