// A stand-in for the HIP runtime that runs nothing and writes down what a library asks it to launch (tests/test_launches.py loads
// it in front of libet_hip.so, so that no device is needed).
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string> names;
std::map<const void*, int> raised;
std::string lines;
struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} pushed;
void* slot[1];
char symbol[1];
int cus() {
  const char* n = std::getenv("RECORDER_CUS");
  return n ? std::atoi(n) : 256;
}
}  // namespace

extern "C" {
// one line per launch: kernel, workgroups, dynamic LDS, the size raised for the kernel on this device (0: none)
const char* recorded_launches() { return lines.c_str(); }
void forget_launches() { lines.clear(); }

void** __hipRegisterFatBinary(const void*) { return slot; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, void*, void*, void*, void*, int*) {
  names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
  pushed = {grid, block, lds, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
  *grid = pushed.grid, *block = pushed.block, *lds = pushed.lds, *stream = pushed.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t lds, hipStream_t) {
  char line[64];
  std::snprintf(line, sizeof line, " %u %zu %d\n", grid.x * grid.y * grid.z, lds, raised.count(f) ? raised[f] : 0);
  lines += names[f] + line;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute attr, int value) {
  if (attr == hipFuncAttributeMaxDynamicSharedMemorySize) raised[f] = value;
  return value <= 160 * 1024 ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = cus(), hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {       // (the header gives it its versioned name)
  std::memset(p, 0, sizeof *p);
  std::strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = cus();
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = symbol, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "recorder"; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { return *s = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
}
