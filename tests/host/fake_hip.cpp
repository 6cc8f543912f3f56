// The HIP runtime entry points that librtx.so calls, on host memory: allocations are
// malloc within a settable limit, copies are memcpy, kernels do not run.  Loaded with
// RTLD_GLOBAL before librtx.so it takes the place of libamdhip64, so that what the
// library allocates and how it takes a failed allocation can be tested without a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

namespace {
std::mutex g_lock;
std::map<void*, size_t> g_blocks;
size_t g_live = 0, g_peak = 0, g_limit = ~(size_t)0, g_largest = 0;
long g_launches = 0;
struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
thread_local Call g_call;

hipError_t take(void** p, size_t n) {
  std::lock_guard<std::mutex> hold(g_lock);
  *p = nullptr;
  if (g_live > g_limit || n > g_limit - g_live) return hipErrorOutOfMemory;
  *p = calloc(1, n ? n : 1);
  if (!*p) return hipErrorOutOfMemory;
  g_blocks[*p] = n;
  g_live += n;
  if (g_live > g_peak) g_peak = g_live;
  if (n > g_largest) g_largest = n;
  return hipSuccess;
}
}  // namespace

extern "C" {

void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_live() { return g_live; }
size_t fake_largest() { return g_largest; }
void fake_reset() { g_largest = 0, g_peak = g_live, g_launches = 0; }
size_t fake_peak() { return g_peak; }
long fake_launches() { return g_launches; }

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
  memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->maxSharedMemoryPerMultiProcessor = 160 << 10;
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> hold(g_lock);
  auto it = g_blocks.find(p);
  if (!p) return hipSuccess;
  if (it == g_blocks.end()) return hipErrorInvalidValue;
  g_live -= it->second;
  g_blocks.erase(it);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(calloc(1, 8)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(calloc(1, 8)), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 4, hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  static void* area = calloc(1, 256u << 20);
  return *p = area, hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_call = Call{grid, block, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_call.grid, *block = g_call.block, *lds = g_call.lds, *s = g_call.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3, void**, size_t, hipStream_t) {
  if (grid.x == 0 || grid.y == 0 || grid.z == 0) return hipErrorInvalidConfiguration;
  std::lock_guard<std::mutex> hold(g_lock);
  g_launches++;
  return hipSuccess;
}

}  // extern "C"
