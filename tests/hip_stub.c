/* hip_stub.c -- a stand-in for the HIP runtime that the C ABI library links,
 * for tests of its host code without a GPU: memory is the host's, kernels do
 * nothing, and the test counts calls, makes them fail or holds them.  Built
 * with the runtime's soname, so that a library loaded after it takes it. */
#include <pthread.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, FAIL = 719 };

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static pthread_cond_t cv = PTHREAD_COND_INITIALIZER;

/* what the test reads and sets */
int stub_allocs, stub_frees;           /* device and host */
int stub_host_allocs, stub_host_frees; /* of these, the host's */
int stub_launches;
int stub_fail_launch; /* launches fail */
int stub_fail_sync;   /* stream synchronisations fail */
int stub_hold;        /* a stream synchronisation returns once this many are under way */
static int launch_error, held;

static int get(void **p, size_t n, int host) {
  *p = calloc(1, n ? n : 1);
  pthread_mutex_lock(&mu);
  stub_allocs++;
  stub_host_allocs += host;
  pthread_mutex_unlock(&mu);
  return OK;
}
static int put(void *p, int host) {
  free(p);
  pthread_mutex_lock(&mu);
  stub_frees++;
  stub_host_frees += host;
  pthread_mutex_unlock(&mu);
  return OK;
}
int hipMalloc(void **p, size_t n) { return get(p, n, 0); }
int hipFree(void *p) { return put(p, 0); }
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  (void)flags;
  return get(p, n, 1);
}
int hipHostFree(void *p) { return put(p, 1); }

int hipLaunchKernel() {
  pthread_mutex_lock(&mu);
  stub_launches++;
  if (stub_fail_launch) launch_error = FAIL;
  pthread_mutex_unlock(&mu);
  return stub_fail_launch ? FAIL : OK;
}
int hipGetLastError(void) {
  const int e = launch_error;
  launch_error = OK;
  return e;
}
int hipStreamSynchronize(void *s) {
  (void)s;
  if (stub_fail_sync) return FAIL;
  pthread_mutex_lock(&mu);
  held++;
  pthread_cond_broadcast(&cv);
  while (held < stub_hold) pthread_cond_wait(&cv, &mu);
  pthread_mutex_unlock(&mu);
  return OK;
}
void stub_reset_hold(int n) {
  held = 0;
  stub_hold = n;
}

int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) {
  (void)kind, (void)st;
  memcpy(d, s, n);
  return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return hipMemcpyAsync(d, s, n, kind, 0); }
int hipMemset(void *d, int v, size_t n) {
  memset(d, v, n);
  return OK;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) {
  (void)st;
  return hipMemset(d, v, n);
}
int hipGetSymbolAddress(void **p, const void *symbol) {
  static char area[8 << 20];
  (void)symbol;
  *p = area;
  return OK;
}
int hipGetDevice(int *d) {
  *d = 0;
  return OK;
}
int hipGetDeviceCount(int *n) {
  *n = 1;
  return OK;
}
int hipDeviceGetAttribute(int *v, int a, int d) {
  (void)a, (void)d;
  *v = 256;
  return OK;
}
int hipDeviceSynchronize(void) { return OK; }
const char *hipGetErrorString(int e) { return e ? "stub failure" : "no error"; }
int hipEventCreate(void **e) {
  *e = 0;
  return OK;
}
int hipEventCreateWithFlags(void **e, unsigned f) {
  (void)f;
  *e = 0;
  return OK;
}
int hipEventDestroy() { return OK; }
int hipEventElapsedTime(float *ms) {
  *ms = 1;
  return OK;
}
int hipEventRecord() { return OK; }
int hipEventSynchronize() { return OK; }
int hipGraphAddKernelNode() { return FAIL; }
int hipGraphCreate() { return FAIL; }
int hipGraphDestroy() { return FAIL; }
int hipGraphExecDestroy() { return FAIL; }
int hipGraphInstantiate() { return FAIL; }
int hipGraphLaunch() { return FAIL; }
/* what the compiler emits around kernels */
int __hipPushCallConfiguration() { return OK; }
int __hipPopCallConfiguration(void *grid, void *block, size_t *shared, void **stream) {
  memset(grid, 0, 12);
  memset(block, 0, 12);
  *shared = 0;
  *stream = 0;
  return OK;
}
void **__hipRegisterFatBinary() {
  static void *handle;
  return &handle;
}
void __hipRegisterFunction() {}
void __hipRegisterVar() {}
void __hipUnregisterFatBinary() {}
