/* A stand-in for the HIP runtime, for tests of the library's host code without
 * a GPU: device memory is host memory, kernels do nothing, and every access
 * the host makes to an allocation is checked against its size. Loaded with
 * RTLD_GLOBAL before the library, whose calls then resolve to it. Entry
 * points of the runtime that the library does not call are not here. */
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#define MAX_BLOCKS 4096
static struct {
  char *p;
  size_t n;
} block[MAX_BLOCKS];
static int fail_in = -1;   /* allocations until one fails; -1: none does */
static int overruns;       /* accesses past their allocation */
static int queued;         /* launches and copies not waited for */
static hipError_t last;    /* the error hipGetLastError reports */

/* The n-th allocation from now fails (0: the next; -1: none); returns what is
 * left of the previous setting, -1 if that one has failed. */
int standin_fail_allocation(int n) {
  const int left = fail_in;
  fail_in = n;
  return left;
}
int standin_overruns(void) { return overruns; }
int standin_queued(void) { return queued; }
int standin_live(void) {
  int n = 0;
  for (int k = 0; k < MAX_BLOCKS; k++) n += block[k].p != NULL;
  return n;
}

/* Whether [p, p + n) is host memory or within one allocation. An allocation
 * is followed by 64 bytes of its own, so that an access just past its end is
 * seen and harms nothing. */
static int inside(const void *q, size_t n) {
  const char *p = (const char *)q;
  for (int k = 0; k < MAX_BLOCKS; k++)
    if (block[k].p && p >= block[k].p && p < block[k].p + block[k].n + 64) {
      if (p + n <= block[k].p + block[k].n) return 1;
      overruns++;
      return 0;
    }
  return 1;
}

static hipError_t take(void **out, size_t n) {
  *out = NULL;
  if (fail_in >= 0 && fail_in-- == 0) return last = hipErrorOutOfMemory;
  for (int k = 0; k < MAX_BLOCKS; k++)
    if (!block[k].p) {
      block[k].p = (char *)malloc(n + 64);
      if (!block[k].p) return hipErrorOutOfMemory;
      memset(block[k].p, 0xA5, n + 64);
      block[k].n = n;
      *out = block[k].p;
      return hipSuccess;
    }
  return hipErrorOutOfMemory;
}
static hipError_t give(void *p) {
  if (!p) return hipSuccess;
  for (int k = 0; k < MAX_BLOCKS; k++)
    if (block[k].p == (char *)p) {
      free(p);
      block[k].p = NULL;
      return hipSuccess;
    }
  return hipErrorInvalidValue;
}

hipError_t hipMalloc(void **p, size_t n) { return take(p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) {
  (void)flags;
  return take(p, n);
}
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemset(void *p, int v, size_t n) {
  if (inside(p, n)) memset(p, v, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t s) {
  (void)s;
  queued++;
  return hipMemset(p, v, n);
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
  (void)k;
  if (!d || !s) return hipErrorInvalidValue;
  if (inside(d, n) & inside(s, n)) memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
  (void)st;
  queued++;
  return hipMemcpy(d, s, n, k);
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t l, hipStream_t s) {
  (void)f, (void)g, (void)b, (void)a, (void)l, (void)s;
  queued++;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  (void)s;
  queued = 0;
  return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d) { /* (a macro: the name with the version) */
  (void)d;
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  (void)d;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "success" : "error"; }

static int handle; /* what every stream, event and module is */
#define HANDLE(type) ((type)&handle)
hipError_t hipStreamCreate(hipStream_t *s) {
  *s = HANDLE(hipStream_t);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
  (void)s;
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) {
  (void)s, (void)e, (void)f;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = HANDLE(hipEvent_t);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) {
  (void)f;
  return hipEventCreate(e);
}
hipError_t hipEventDestroy(hipEvent_t e) {
  (void)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  (void)e, (void)s;
  return hipSuccess;
}

/* What the compiler's launch and registration code calls. */
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
  (void)g, (void)b, (void)l, (void)s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s) {
  g->x = g->y = g->z = b->x = b->y = b->z = 1;
  *l = 0;
  *s = HANDLE(hipStream_t);
  return hipSuccess;
}
void **__hipRegisterFatBinary(const void *data) {
  (void)data;
  return HANDLE(void **);
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *hf, char *df, const char *dn, unsigned n, void *a, void *b, void *c,
                           void *d, int *e) {
  (void)m, (void)hf, (void)df, (void)dn, (void)n, (void)a, (void)b, (void)c, (void)d, (void)e;
}
void __hipRegisterVar(void **m, void *v, char *hv, char *dv, int ext, size_t n, int c, int g) {
  (void)m, (void)v, (void)hv, (void)dv, (void)ext, (void)n, (void)c, (void)g;
}
