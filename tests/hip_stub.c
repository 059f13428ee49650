/* A HIP runtime without a GPU, for tests of the host code: device memory is
 * host memory, kernels are only counted.  Preloaded before libimdg.so
 * (LD_PRELOAD) in a process of its own.  It knows which device was current at
 * each allocation and launch, can refuse memory beyond a limit, and can give
 * the launches of one block size a time of their own. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

#define NDEV 2
#define MAXTHR 2048

static __thread int current = 0;
static __thread hipError_t last_error = hipSuccess;   /* until it is read */

/* --- what the tests read and set ------------------------------------------ */
static size_t live = 0, peak = 0, limit = (size_t)1 << 46;
static long wrong_device = 0;        /* launches on another device's stream */
static long mallocs[NDEV];           /* allocations per current device */
static long launches[MAXTHR + 1];    /* launches per block size */
static double ms_of[MAXTHR + 1];     /* their time, 0: 1 ms */
static double clock_ms = 0.0;
static void *pinned = NULL;          /* the last pinned block, and where it */
static const void *pinned_from = NULL;   /* was last filled from */

size_t stub_live(void) { return live; }
size_t stub_peak(void) { return peak; }
void stub_reset_peak(void) { peak = live; }
void stub_limit(size_t bytes) { limit = bytes; }
long stub_wrong_device(void) { return wrong_device; }
long stub_mallocs(int dev) { return mallocs[dev]; }
long stub_launches(int threads) { return launches[threads]; }
void stub_reset_launches(void) { memset(launches, 0, sizeof launches); }
void stub_time(int threads, double ms) { ms_of[threads] = ms; }
void *stub_pinned_from(void) { return (void *)pinned_from; }

/* --- devices --------------------------------------------------------------- */
hipError_t hipGetDeviceCount(int *n) { *n = NDEV; return hipSuccess; }
hipError_t hipSetDevice(int d) {
  if (d < 0 || d >= NDEV) return hipErrorInvalidDevice;
  current = d;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t attr, int dev) {
  (void)dev;
  *v = attr == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) {
  return e == hipErrorOutOfMemory ? "out of memory" : "stub";
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}

/* --- memory: 64 bytes in front of each block hold its size ------------------ */
hipError_t hipMalloc(void **p, size_t n) {
  *p = NULL;
  char *b = n > limit || live > limit - n ? NULL : calloc(1, n + 64);
  if (!b) return last_error = hipErrorOutOfMemory;
  *(size_t *)b = n;
  live += n;
  if (live > peak) peak = live;
  mallocs[current]++;
  *p = b + 64;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  char *b = (char *)p - 64;
  live -= *(size_t *)b;
  free(b);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned int flags) {
  (void)flags;
  *p = pinned = calloc(1, n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind kind) {
  (void)kind;
  memmove(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n,
                          hipMemcpyKind kind, hipStream_t st) {
  (void)st;
  if (d == pinned) pinned_from = s;
  return hipMemcpy(d, s, n, kind);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
  if (st && *(int *)st != current) wrong_device++;   /* a fill is a launch */
  memset(d, v, n);
  return hipSuccess;
}

/* --- streams (a stream is the number of its device), events, launches ------- */
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int flags) {
  (void)flags;
  int *q = malloc(sizeof *q);
  *q = current;
  *s = (hipStream_t)q;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
  (void)s;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
  *e = calloc(1, sizeof(double));
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  (void)s;
  *(double *)e = clock_ms;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
  *ms = (float)(*(double *)b - *(double *)a);
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **args,
                           size_t lds, hipStream_t s) {
  (void)fn, (void)grid, (void)args, (void)lds;
  if (s && *(int *)s != current) wrong_device++;
  if (block.x > MAXTHR) return hipErrorInvalidConfiguration;
  launches[block.x]++;
  clock_ms += ms_of[block.x] > 0.0 ? ms_of[block.x] : 1.0;
  return hipSuccess;
}
static __thread struct {
  dim3 g, b;
  size_t lds;
  hipStream_t s;
} conf;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds,
                                      hipStream_t s) {
  conf.g = g, conf.b = b, conf.lds = lds, conf.s = s;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds,
                                     hipStream_t *s) {
  *g = conf.g, *b = conf.b, *lds = conf.lds, *s = conf.s;
  return hipSuccess;
}
hipError_t hipFuncGetAttributes(struct hipFuncAttributes *a, const void *fn) {
  (void)fn;
  memset(a, 0, sizeof *a);
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *fn, hipFuncAttribute attr, int v) {
  (void)fn, (void)attr, (void)v;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *fn,
                                                        int threads,
                                                        size_t lds) {
  (void)fn;
  *n = lds ? 1 : 2048 / threads;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) {
  (void)p, (void)s;
  return hipErrorNotSupported;
}

/* --- graphs: none ------------------------------------------------------------ */
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) {
  (void)s, (void)m;
  return hipErrorNotSupported;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
  (void)s, (void)g;
  return hipErrorNotSupported;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g,
                               hipGraphNode_t *n, char *b, size_t z) {
  (void)e, (void)g, (void)n, (void)b, (void)z;
  return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s) {
  (void)e, (void)s;
  return hipErrorNotSupported;
}
hipError_t hipGraphDestroy(hipGraph_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  (void)e;
  return hipSuccess;
}

/* --- registration of the library's kernels ----------------------------------- */
void **__hipRegisterFatBinary(const void *d) {
  static void *none = NULL;
  (void)d;
  return &none;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev,
                           const char *name, unsigned int lim, void *t,
                           void *b, void *bd, void *gd, int *ws) {
  (void)m, (void)host, (void)dev, (void)name, (void)lim, (void)t, (void)b;
  (void)bd, (void)gd, (void)ws;
}
void __hipRegisterVar(void **m, void *v, char *hv, char *dv, int ext,
                      size_t size, int constant, int global) {
  (void)m, (void)v, (void)hv, (void)dv, (void)ext, (void)size;
  (void)constant, (void)global;
}
