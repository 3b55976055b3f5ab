// The HIP calls libptx_hip.so makes, answered from host memory: device memory
// with a limit, streams and events that have always finished, and kernels that
// do not run but are listed with their grids.  A check program that includes
// this header and links the library takes these in place of the runtime's, so
// the library's host code runs without a GPU (1 device, 256 CUs).
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace host_runtime {

struct Launch {
   std::string kernel;
   uint32_t grid;
};

struct State {
   std::mutex mu;
   std::map<void *, size_t> device;            // live device allocations
   size_t used = 0, limit = SIZE_MAX;
   uint32_t allocations = 0, copies = 0;        // made so far
   int blocks_per_cu = 4;                      // every kernel's occupancy
   std::map<const void *, std::string> names;  // kernels by host function
   std::vector<Launch> launches;
   hipError_t last = hipSuccess;
   dim3 grid;
};
inline State &state() {
   static State s;
   return s;
}

inline hipError_t result(hipError_t e) {
   if (e != hipSuccess) state().last = e;
   return e;
}
inline hipError_t take(void **p, size_t bytes) {
   State &s = state();
   std::lock_guard<std::mutex> lock(s.mu);
   *p = nullptr;
   if (bytes > s.limit - std::min(s.limit, s.used)) return result(hipErrorOutOfMemory);
   *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
   s.device[*p] = bytes;
   s.used += bytes;
   s.allocations++;
   return hipSuccess;
}
inline hipError_t give(void *p) {
   State &s = state();
   std::lock_guard<std::mutex> lock(s.mu);
   if (!p) return hipSuccess;
   const auto it = s.device.find(p);
   if (it == s.device.end()) return result(hipErrorInvalidValue);
   s.used -= it->second;
   s.device.erase(it);
   std::free(p);
   return hipSuccess;
}
template <class T>
hipError_t handle(T *p) {
   *p = reinterpret_cast<T>(uintptr_t(0x1000));
   return hipSuccess;
}

}  // namespace host_runtime

extern "C" {
using namespace host_runtime;

void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(uintptr_t(0x1000)); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
   state().names[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3, size_t, hipStream_t) {
   state().grid = grid;
   return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
   *grid = state().grid;
   *block = dim3(256);
   *shared = 0;
   *stream = nullptr;
   return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t) {
   State &s = state();
   std::lock_guard<std::mutex> lock(s.mu);
   s.launches.push_back(Launch{s.names[f], grid.x});
   return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
   *n = state().blocks_per_cu;
   return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
   static char *scratch = static_cast<char *>(std::aligned_alloc(256, size_t(64) << 20));
   *p = scratch;
   return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
   *n = 1;
   return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
   std::memset(p, 0, sizeof(*p));
   std::strcpy(p->gcnArchName, "gfx950");
   p->multiProcessorCount = 256;
   return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "host runtime"; }
hipError_t hipGetLastError(void) {
   const hipError_t e = state().last;
   state().last = hipSuccess;
   return e;
}
hipError_t hipMemGetInfo(size_t *unused, size_t *all) {
   *all = state().limit;
   *unused = state().limit - std::min(state().limit, state().used);
   return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return take(p, n); }
hipError_t hipMallocFromPoolAsync(void **p, size_t n, hipMemPool_t, hipStream_t) { return take(p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
   *p = std::malloc(n);
   return hipSuccess;
}
hipError_t hipHostFree(void *p) {
   std::free(p);
   return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
   state().copies++;
   std::memcpy(d, s, n);
   return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
   std::memcpy(d, s, n);
   return hipSuccess;
}
hipError_t hipMemPoolCreate(hipMemPool_t *p, const hipMemPoolProps *) { return handle(p); }
hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *g, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(g); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
   *ms = 1.f;
   return hipSuccess;
}

}  // extern "C"
