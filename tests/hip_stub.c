/* The HIP entry points that libfvm_gpu.so imports, on host memory and without a
 * device: allocations come from a budget, copies are memcpy, kernels do nothing.
 * For tests of the library's host side (what it allocates, in which order, and
 * how often it waits); nothing is computed.  Built and loaded by
 * tests/test_host_side.py, in a process of its own. */
#include <stdlib.h>
#include <string.h>

#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

static size_t used, budget = (size_t)-1;
static long waits, launches, copies;
static struct {
  char *p;
  size_t n;
} pinned[256]; /* live hipHostMalloc blocks */

size_t stub_used(void) { return used; }
void stub_budget(size_t bytes) { budget = bytes; }
long stub_waits(void) { return waits; }
long stub_launches(void) { return launches; }
long stub_copies(void) { return copies; }

hipError_t hipMalloc(void **p, size_t n) {
  if (n > budget || used > budget - n) return hipErrorOutOfMemory;
  size_t *q = (size_t *)calloc(1, n + 64);
  if (!q) return hipErrorOutOfMemory;
  q[0] = n;
  used += n;
  *p = q + 8;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  size_t *q = (size_t *)p - 8;
  used -= q[0];
  free(q);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) {
  int i = 0;
  while (i < 256 && pinned[i].p) i++;
  if (i == 256 || !(*p = calloc(1, n))) return hipErrorOutOfMemory;
  pinned[i].p = *p;
  pinned[i].n = n;
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  for (int i = 0; i < 256; i++)
    if (pinned[i].p == p) pinned[i].p = 0;
  free(p);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  memset(a, 0, sizeof *a);
  a->type = hipMemoryTypeUnregistered;
  for (int i = 0; i < 256; i++)
    if (pinned[i].p && (char *)p >= pinned[i].p && (char *)p < pinned[i].p + pinned[i].n) a->type = hipMemoryTypeHost;
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  __atomic_add_fetch(&copies, 1, __ATOMIC_RELAXED);
  return hipMemcpy(d, s, n, k);
}
hipError_t hipMemset(void *d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) { return hipMemset(d, v, n); }
hipError_t hipStreamSynchronize(hipStream_t st) {
  __atomic_add_fetch(&waits, 1, __ATOMIC_RELAXED);
  return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *st) {
  *st = (hipStream_t)1;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned f) { return hipStreamCreate(st); }
hipError_t hipStreamDestroy(hipStream_t st) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = (hipEvent_t)1;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
  *ms = 0.0f;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t st) { return 0; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) { /* hipGetDevicePropertiesR0600 */
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute a, int v) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *s) {
  static char symbol[64];
  *p = symbol;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t shared, hipStream_t st) {
  __atomic_add_fetch(&launches, 1, __ATOMIC_RELAXED);
  return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t st) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *st) {
  memset(g, 0, sizeof *g);
  memset(b, 0, sizeof *b);
  *shared = 0;
  *st = 0;
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *d) {
  static void *h;
  return &h;
}
void __hipRegisterFunction(void **m, const void *f, char *df, const char *n, unsigned l, void *a, void *b, void *c, void *d,
                           int *w) {}
void __hipRegisterVar(void **m, void *v, char *hv, char *dv, int e, size_t n, int c, int g) {}
void __hipUnregisterFatBinary(void **m) {}
