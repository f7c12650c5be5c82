// The HIP calls of a standalone GEMV plan and of a context's forward passes on
// host memory, for tests of the host side without a GPU: loaded with
// RTLD_GLOBAL before libcis2amd.so, its definitions take the place of the
// runtime's.  Device memory starts as all ones (a NaN in every word); a GEMV
// launch records whether its input holds such a word and stores
// y[m] = x[0] + m; the model's kernels are counted by name and compute nothing.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

namespace {
std::map<const void*, std::string> names;
std::map<void*, size_t> live;
std::map<std::string, int> launched;
size_t device_most = SIZE_MAX;
int pinned_left = 1 << 30, undefined_inputs = 0, launches = 0, allocations = 0;
dim3 cfg_grid, cfg_block;

hipError_t take(void** p, size_t n) {
  ++allocations;
  *p = malloc(n);
  memset(*p, 0xFF, n);
  live[*p] = n;
  return hipSuccess;
}
hipError_t give(void* p) {
  if (p && !live.erase(p)) return hipErrorInvalidValue;
  free(p);
  return hipSuccess;
}
template <typename T>
T arg(void** args, int i) {
  return *static_cast<T*>(args[i]);
}
void gemv(const float* x, float* y, uint32_t M, uint32_t K, uint32_t n) {
  ++launches;
  for (uint32_t i = 0; i < n; ++i) {
    bool bad = false;
    for (uint32_t k = 0; k < K; ++k) {
      uint32_t w;
      memcpy(&w, x + (size_t)i * K + k, 4);
      bad = bad || w == 0xFFFFFFFFu;
    }
    undefined_inputs += bad;
    for (uint32_t m = 0; m < M; ++m) y[(size_t)i * M + m] = x[(size_t)i * K] + (float)m;
  }
}
}  // namespace

extern "C" {
void stub_allow_pinned(int n) { pinned_left = n; }
int stub_undefined_inputs() { return undefined_inputs; }
int stub_launches() { return launches; }
int stub_allocations() { return allocations; }
// device allocations of more than `most` bytes are refused
void stub_device_most(size_t most) { device_most = most; }
// launches of kernels whose name holds `part`
int stub_launched(const char* part) {
  int n = 0;
  for (const auto& l : launched)
    if (l.first.find(part) != std::string::npos) n += l.second;
  return n;
}
int stub_live() { return (int)live.size(); }

void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  names[fn] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
  cfg_grid = g;
  cfg_block = b;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = cfg_grid;
  *b = cfg_block;
  *s = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3, void** a, size_t, hipStream_t) {
  const std::string& n = names[fn];
  ++launched[n];
  if (n.find("k_gemv_blk") != std::string::npos)
    gemv(arg<const float*>(a, 1), arg<float*>(a, 2), arg<uint32_t>(a, 3), arg<uint32_t>(a, 4), 1);
  else if (n.find("k_gemv_many") != std::string::npos)
    gemv(arg<const float*>(a, 4), arg<float*>(a, 5), arg<uint32_t>(a, 6), arg<uint32_t>(a, 7),
         grid.y);
  else if (n.find("k_copy16") != std::string::npos)
    memcpy(arg<void*>(a, 1), arg<const void*>(a, 0), arg<uint64_t>(a, 2) * 16);
  else if (n.find("k_fpenv_probe") != std::string::npos)
    memset(arg<void*>(a, 1), 0, 8);  // subnormals are flushed
  else if (n.find("k_take_word") != std::string::npos) {
    *arg<uint32_t*>(a, 1) = *arg<uint32_t*>(a, 0);
    *arg<uint32_t*>(a, 0) = 0;
  }
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  return *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024, hipSuccess;
}
hipError_t hipDeviceGetPCIBusId(char* s, int n, int) { return strncpy(s, "stub", n), hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
  return *n = 1, hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static char symbol[64];
  return *p = symbol, hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
  return n <= device_most ? take(p, n) : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  return pinned_left-- > 0 ? take(p, n) : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  return memset(d, v, n), hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}
