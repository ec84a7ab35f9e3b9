// fake_hip.cpp -- the HIP runtime calls of libbrawl_hip.so without a device,
// for tests of its host code: device memory is host memory, kernels do nothing
// (each launch goes to a callback, which can make it fail), and every stream
// knows whether work on it has been waited for.  Loaded with RTLD_GLOBAL before
// the library, so that the library's calls come here.
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <set>

namespace {
struct Event {
  hipStream_t after = nullptr;
};
std::set<void *> busy;                             // streams with work not waited for
std::map<void *, std::set<void *>> waits;          // streams that a stream's work comes after
int streams = 0, freed_busy = 0, pinned_made = 0, pinned_held = 0, syncs = 0;
int (*on_launch)(const void *, int, int, long long, void *) = nullptr;

void done(void *s) {
  busy.erase(s);
  const std::set<void *> before = waits[s];
  waits.erase(s);
  for (void *b : before) done(b);
}
}  // namespace

extern "C" {

void fake_on_launch(int (*f)(const void *, int, int, long long, void *)) { on_launch = f; }
int fake_busy() { return (int)busy.size(); }
int fake_freed_busy() { return freed_busy; }
int fake_pinned_made() { return pinned_made; }
int fake_pinned_held() { return pinned_held; }
int fake_syncs() { return syncs; }

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "made to fail"; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
  *p = calloc(1, n ? n : 1);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
  if (!busy.empty()) ++freed_busy;
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  ++pinned_made;
  ++pinned_held;
  return hipMalloc(p, n);
}
hipError_t hipHostFree(void *p) {
  --pinned_held;
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  busy.insert(st);
  return memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
  busy.insert(st);
  return memset(d, v, n), hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = (hipStream_t)(size_t)++streams;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  ++syncs;
  done(s);
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t) new Event, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (Event *)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return ((Event *)e)->after = s, hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return done(((Event *)e)->after), hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  void *after = ((Event *)e)->after;
  if (after != s && busy.count(after)) waits[s].insert(after);
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { return *n = 2, hipSuccess; }
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **, size_t lds, hipStream_t s) {
  const int rc = on_launch ? on_launch(fn, (int)grid.x, (int)block.x, (long long)lds, s) : 0;
  if (rc) return hipErrorLaunchFailure;
  busy.insert(s);
  return hipSuccess;
}

}  // extern "C"
