// A HIP runtime without a device, preloaded over libamdhip64 (tests/test_failed_calls.py):
// device and pinned memory come from calloc, copies are memcpy, kernels are logged
// by name and do nothing. fake_fail(n) makes the n-th call from then on that can
// fail, and the one after it (an allocation is tried twice), return
// hipErrorOutOfMemory (2).
#include <stddef.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3_;

static long fail_at = 0, failing = 0;  // 0: off
static long live = 0;     // allocations, streams and events not given back
static char log_[1 << 20];
static size_t log_n = 0;

void fake_fail(long nth) { fail_at = nth; failing = 0; }
long fake_armed(void) { return fail_at; }
long fake_live(void) { return live; }
void fake_log_clear(void) { log_[log_n = 0] = 0; }
const char *fake_log(void) { return log_; }

static int fails(void) {
  if (fail_at > 0 && --fail_at == 0) failing = 2;
  return failing > 0 && failing-- > 0;
}
static int make(void **p, size_t n) {
  *p = NULL;
  if (fails()) return 2;
  *p = calloc(1, n ? n : 1);
  live++;
  return 0;
}
static int drop(void *p) {
  if (p) live--;
  free(p);
  return 0;
}

// kernels by the host stub's address
static const void *fn_host[4096];
static char fn_name[4096][128];
static int fn_n = 0;
void **__hipRegisterFatBinary(const void *d) { (void)d; static void *m; return &m; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned lim, void *a, void *b,
                           void *c, void *d, int *w) {
  (void)m; (void)dev; (void)lim; (void)a; (void)b; (void)c; (void)d; (void)w;
  if (fn_n == 4096) return;
  fn_host[fn_n] = host;
  snprintf(fn_name[fn_n++], sizeof fn_name[0], "%s", name);
}
static size_t var_size;
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t size, int c, int g) {
  (void)m; (void)v; (void)h; (void)d; (void)e; (void)c; (void)g;
  if (size > var_size) var_size = size;
}

static struct { dim3_ g, b; size_t s; void *st; } cfg;
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t s, void *st) {
  cfg.g = g; cfg.b = b; cfg.s = s; cfg.st = st;
  return 0;
}
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *s, void **st) {
  *g = cfg.g; *b = cfg.b; *s = cfg.s; *st = cfg.st;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **args, size_t s, void *st) {
  (void)g; (void)b; (void)args; (void)s; (void)st;
  for (int i = 0; i < fn_n; i++)
    if (fn_host[i] == f && log_n + 130 < sizeof log_) log_n += (size_t)sprintf(log_ + log_n, "%s\n", fn_name[i]);
  return 0;
}

int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { return e ? "out of memory (fake)" : "no error"; }
int hipDeviceSynchronize(void) { return 0; }
int hipFuncGetAttributes(void *a, const void *f) { (void)a; (void)f; return 0; }
int hipGetSymbolAddress(void **p, const void *s) {
  static void *var;
  (void)s;
  if (!var) var = calloc(1, var_size);
  *p = var;
  return 0;
}

int hipMalloc(void **p, size_t n) { return make(p, n); }
int hipFree(void *p) { return drop(p); }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return make(p, n); }
int hipHostFree(void *p) { return drop(p); }
int hipHostGetDevicePointer(void **d, void *h, unsigned f) {
  (void)f;
  *d = NULL;
  if (fails()) return 2;
  *d = h;
  return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; return make(s, 1); }
int hipStreamDestroy(void *s) { return drop(s); }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return 0; }
int hipEventCreate(void **e) { return make(e, 1); }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return make(e, 1); }
int hipEventDestroy(void *e) { return drop(e); }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *t, void *a, void *b) { (void)a; (void)b; *t = 0; return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) {
  (void)k; (void)st;
  memcpy(d, s, n);
  return 0;
}
