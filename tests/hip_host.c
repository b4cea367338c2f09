/* The HIP runtime on the host, as far as the transfers, saves and allocations
 * of libsac_amd.so use it: device memory is host memory, every stream runs at
 * once, k_rows (state rows to and from a flat buffer) is carried out, other
 * kernels do nothing.  Loaded before the library (tests/hip_host.py), so that
 * its failure paths can be run without a GPU.  Each hip_host_* variable sets a
 * failure or counts what happened. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <pthread.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

typedef int hipError_t;
typedef struct { uint32_t x, y, z; } dim3;
enum { OK = 0, INVALID = 1, NOMEM = 2, NOT_READY = 600, LAUNCH = 719 };

/* failures */
int hip_host_fail_malloc = 0;       /* the n-th hipMalloc from now on fails, once */
int hip_host_fail_event = 0;        /* the n-th event creation from now on fails, once */
int hip_host_fail_pinned = 0;       /* 1: every hipHostMalloc fails; 2: on other threads only */
int hip_host_fail_launch = 0;       /* launches fail: 1 on other threads, 2 on the first thread */
int hip_host_fail_new = 0;          /* the n-th operator new from now on throws, once */
/* what happened */
int hip_host_null_stores = 0;       /* kernels that would have used a null pointer */
int hip_host_freed_used = 0;        /* ensemble kernels given memory that was freed */
size_t hip_host_pinned_most = 0;    /* largest pinned allocation */
size_t hip_host_pinned_now = 0;     /* pinned bytes, now and at most */
size_t hip_host_pinned_peak = 0;
int hip_host_threads = 0;           /* launches on other threads than the first */

static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;
static __thread hipError_t last_error = OK;
static __thread int device = 0;
static pthread_t first;
__attribute__((constructor)) static void init(void) { first = pthread_self(); }
static int other(void) { return !pthread_equal(pthread_self(), first); }
static hipError_t err(hipError_t e) {
  if (e != OK) last_error = e;
  return e;
}
static int counted(int *n) { /* the call that brings *n to 0 */
  pthread_mutex_lock(&lock);
  const int hit = *n > 0 && --*n == 0;
  pthread_mutex_unlock(&lock);
  return hit;
}

/* ---- operator new of the library ---- */
void *_Znwm(size_t n) {
  if (counted(&hip_host_fail_new)) {
    void (*bad)(void) = (void (*)(void))dlsym(RTLD_DEFAULT, "_ZSt17__throw_bad_allocv");
    if (bad) bad();
    abort();
  }
  return malloc(n ? n : 1);
}

/* ---- errors and devices ---- */
hipError_t hipGetLastError(void) {
  const hipError_t e = last_error;
  last_error = OK;
  return e;
}
const char *hipGetErrorString(hipError_t e) {
  return e == OK ? "no error" : e == NOMEM ? "out of memory" : "failed";
}
hipError_t hipGetDeviceCount(int *n) { return *n = 2, OK; }
hipError_t hipGetDevice(int *d) { return *d = device, OK; }
hipError_t hipSetDevice(int d) { return device = d, OK; }
hipError_t hipDeviceSynchronize(void) { return OK; }

/* ---- memory ---- */
hipError_t hipMalloc(void **p, size_t n) {
  if (counted(&hip_host_fail_malloc)) return *p = NULL, err(NOMEM);
  return *p = calloc(1, n ? n : 1), OK;
}
static void *freed[4096]; /* kept, so that no allocation gets the address again */
static int nfreed = 0;
hipError_t hipFree(void *p) {
  pthread_mutex_lock(&lock);
  if (p && nfreed < 4096) freed[nfreed++] = p;
  else free(p);
  pthread_mutex_unlock(&lock);
  return OK;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) {
  (void)flags;
  if (hip_host_fail_pinned == 1 || (hip_host_fail_pinned == 2 && other())) return *p = NULL, err(NOMEM);
  size_t *b = malloc(n + 64);
  *b = n;
  pthread_mutex_lock(&lock);
  if (n > hip_host_pinned_most) hip_host_pinned_most = n;
  hip_host_pinned_now += n;
  if (hip_host_pinned_now > hip_host_pinned_peak) hip_host_pinned_peak = hip_host_pinned_now;
  pthread_mutex_unlock(&lock);
  return *p = (char *)b + 64, OK;
}
hipError_t hipHostFree(void *p) {
  if (!p) return OK;
  size_t *b = (size_t *)((char *)p - 64);
  pthread_mutex_lock(&lock);
  hip_host_pinned_now -= *b;
  pthread_mutex_unlock(&lock);
  return free(b), OK;
}
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), OK; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, int kind) {
  (void)kind;
  if (!d || !s) return err(INVALID);
  return memcpy(d, s, n), OK;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
  (void)st;
  return hipMemcpy(d, s, n, kind);
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h,
                            int kind, void *st) {
  (void)kind, (void)st;
  if (!d || !s || w > dp || w > sp) return err(INVALID);
  for (size_t i = 0; i < h; i++) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
  return OK;
}

/* ---- streams and events ---- */
hipError_t hipStreamCreate(void **s) { return *s = malloc(1), OK; }
hipError_t hipStreamCreateWithFlags(void **s, unsigned f) { return (void)f, *s = malloc(1), OK; }
hipError_t hipStreamDestroy(void *s) { return free(s), OK; }
hipError_t hipStreamSynchronize(void *s) { return (void)s, OK; }
hipError_t hipStreamWaitEvent(void *s, void *e, unsigned f) { return (void)s, (void)e, (void)f, OK; }
hipError_t hipEventCreateWithFlags(void **e, unsigned f) {
  (void)f;
  if (counted(&hip_host_fail_event)) return *e = NULL, err(NOMEM);
  return *e = malloc(1), OK;
}
hipError_t hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(void *e) { return free(e), OK; }
hipError_t hipEventRecord(void *e, void *s) { return (void)s, e ? OK : err(INVALID); }
hipError_t hipEventSynchronize(void *e) { return e ? OK : err(INVALID); }
hipError_t hipEventQuery(void *e) { return e ? OK : err(INVALID); }
hipError_t hipEventElapsedTime(float *ms, void *a, void *b) { return (void)a, (void)b, *ms = 0, OK; }

/* ---- kernels ---- */
static struct { const void *host; char name[256]; } kernels[512];
static int nkernels = 0;
void **__hipRegisterFatBinary(const void *d) {
  static void *m;
  return (void)d, &m;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t n, int c, int g) {
  (void)m, (void)v, (void)h, (void)d, (void)e, (void)n, (void)c, (void)g;
}
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned l,
                           void *t, void *b, void *bd, void *gd, int *ws) {
  (void)m, (void)dev, (void)l, (void)t, (void)b, (void)bd, (void)gd, (void)ws;
  if (nkernels < 512) {
    kernels[nkernels].host = host;
    strncpy(kernels[nkernels++].name, name, 255);
  }
}
static __thread struct { dim3 g, b; size_t sh; void *st; } call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void *st) {
  return call.g = g, call.b = b, call.sh = sh, call.st = st, OK;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, void **st) {
  return *g = call.g, *b = call.b, *sh = call.sh, *st = call.st, OK;
}

/* k_rows<T, OUT>(T *dev, T *flat, n, x0, R0, G0, rows, pitch, fs) */
static void rows(void **a, size_t esz, int out) {
  char *dev = *(char **)a[0], *flat = *(char **)a[1];
  const unsigned n = *(unsigned *)a[2], x0 = *(unsigned *)a[3], R0 = *(unsigned *)a[4],
                 G0 = *(unsigned *)a[5], nr = *(unsigned *)a[6];
  const long long pitch = *(long long *)a[7], fs = *(long long *)a[8];
  if (!dev || !flat) {
    hip_host_null_stores++;
    return;
  }
  for (unsigned i = 0; i < n; i++) {
    const unsigned r = (x0 + i) / G0, x = x0 + i - r * G0, R = R0 + r, f = R / nr;
    char *p = dev + esz * ((long long)f * fs + (long long)(R - f * nr) * pitch + x);
    if (out) memcpy(flat + esz * (size_t)i, p, esz);
    else memcpy(p, flat + esz * (size_t)i, esz);
  }
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t sh, void *st) {
  (void)g, (void)b, (void)sh, (void)st;
  if (other()) {
    pthread_mutex_lock(&lock);
    hip_host_threads++;
    pthread_mutex_unlock(&lock);
  }
  if (hip_host_fail_launch && hip_host_fail_launch == (other() ? 1 : 2)) return err(LAUNCH);
  if (hip_host_fail_launch) usleep(5000); /* the failing threads get chunks too */
  for (int k = 0; k < nkernels; k++)
    if (kernels[k].host == f) {
      const char *t = strstr(kernels[k].name, "k_rowsI");
      if (t) rows(args, t[7] == 'm' ? 8 : 4, strncmp(t + 8, "Lb1", 3) == 0);
      /* the pointers of sac::batch::Args, which is longer than this */
      if (strstr(kernels[k].name, "sac5batch") && strstr(kernels[k].name, "NS0_4ArgsE"))
        for (int w = 0; w < 25; w++)
          for (int j = 0; j < nfreed; j++)
            hip_host_freed_used += ((void **)args[0])[w] == freed[j];
      return OK;
    }
  return err(INVALID);
}

/* ---- not used in these tests ---- */
hipError_t hipGetSymbolAddress(void **p, const void *s) { return (void)s, *p = NULL, err(INVALID); }
hipError_t hipGraphDestroy(void *g) { return (void)g, OK; }
hipError_t hipGraphExecDestroy(void *g) { return (void)g, OK; }
hipError_t hipGraphInstantiate(void **g, void *h, void *e, char *l, size_t n) {
  return (void)g, (void)h, (void)e, (void)l, (void)n, err(INVALID);
}
hipError_t hipGraphLaunch(void *g, void *s) { return (void)g, (void)s, err(INVALID); }
hipError_t hipStreamBeginCapture(void *s, int m) { return (void)s, (void)m, err(INVALID); }
hipError_t hipStreamEndCapture(void *s, void **g) { return (void)s, (void)g, err(INVALID); }
