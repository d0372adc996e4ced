/* A stand-in for the HIP runtime, so that the host side of liblbm_hip.so runs
 * on the CPU: device memory is host memory, kernels do not run (the two that
 * the host reads results of are played), launches are recorded, and a test can
 * make an allocation or the launch of one kernel fail. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;

/* controls and records, read and set by the test */
int si_fail_malloc = -1;       /* the n-th hipMalloc from now fails (0: the next) */
char si_fail_launch[64] = "";  /* launches of kernels with this in their name fail ... */
int si_fail_after = 0;         /* ... after this many */
int si_retire = 0;             /* domains that the next graph launch retires */
int si_capturing = 0;
#define RECORDS 4096
int si_launches = 0;
char si_name[RECORDS][64];
unsigned char si_args[RECORDS][512];  /* the first argument of a launch */
unsigned char si_args2[RECORDS][64]; /* and the second of k_poisson_multi */

static struct { const void *f; char name[64]; } kernels[4096];
static int nkernels;
static int last_error;
static struct { dim3_t g, b; size_t shmem; void *s; } config[16];
static int depth;
static int *active;
static int ndom;

int hipMalloc(void **p, size_t n) {
  if (si_fail_malloc >= 0 && si_fail_malloc-- == 0) { *p = 0; return last_error = 2; }
  *p = calloc(n ? n : 1, 1);
  return *p ? 0 : (last_error = 2);
}
int hipFree(void *p) { free(p); return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(n, 1); return *p ? 0 : 2; }
int hipHostFree(void *p) { free(p); return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)st; return hipMemcpy(d, s, n, k); }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); return 0; }
int hipMemsetAsync(void *p, int v, size_t n, void *st) { (void)st; return hipMemset(p, v, n); }
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int e) { return e ? "made to fail" : "no error"; }
static __thread int device;
int hipGetDevice(int *d) { *d = device; return 0; }
int hipSetDevice(int d) { device = d; return 0; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = calloc(1, 256); return 0; }
/* streams and events hold their device */
static int *on_device(void) { int *p = malloc(sizeof(int)); *p = device; return p; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = on_device(); return 0; }
int hipStreamGetDevice(void *s, int *d) { *d = *(int *)s; return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; si_capturing = 1; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; si_capturing = 0; *g = malloc(1); return 0; }
int hipGraphInstantiate(void **e, void *g, void **n, char *l, size_t z) { (void)g; (void)n; (void)l; (void)z; *e = malloc(1); return 0; }
int hipGraphDestroy(void *g) { free(g); return 0; }
int hipGraphExecDestroy(void *e) { free(e); return 0; }
int hipGraphLaunch(void *e, void *s) {
  (void)e;
  (void)s;
  for (int d = 0; active && d < ndom && si_retire > 0; ++d)
    if (active[d]) { active[d] = 0; --si_retire; }
  return 0;
}
int hipEventCreate(void **e) { *e = on_device(); return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return hipEventCreate(e); }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *s) { return *(int *)e == *(int *)s ? 0 : (last_error = 400); }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *t, void *a, void *b) { (void)a; (void)b; *t = 1.0f; return 0; }

void **__hipRegisterFatBinary(const void *d) { (void)d; static void *m; return &m; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterFunction(void **m, const void *f, char *df, const char *name, unsigned l, void *a, void *b, void *c, void *d, int *w) {
  (void)m; (void)df; (void)l; (void)a; (void)b; (void)c; (void)d; (void)w;
  kernels[nkernels].f = f;
  strncpy(kernels[nkernels++].name, name, 63);
}
void __hipRegisterVar(void **m, void *v, char *h, char *n, int e, size_t z, int c, int g) {
  (void)m; (void)v; (void)h; (void)n; (void)e; (void)z; (void)c; (void)g;
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t shmem, void *s) {
  config[depth].g = g; config[depth].b = b; config[depth].shmem = shmem; config[depth++].s = s;
  return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *shmem, void **s) {
  --depth;
  *g = config[depth].g; *b = config[depth].b; *shmem = config[depth].shmem; *s = config[depth].s;
  return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t shmem, void *s) {
  (void)g; (void)b; (void)shmem; (void)s;
  const char *name = "";
  for (int k = 0; k < nkernels; ++k)
    if (kernels[k].f == f) name = kernels[k].name;
  if (si_fail_launch[0] && strstr(name, si_fail_launch) && si_fail_after-- <= 0) return last_error = 1;
  if (strstr(name, "k_fill_int")) {
    int *p = *(int **)args[0], n = *(int *)args[1], v = *(int *)args[2];
    for (int i = 0; i < n; ++i) p[i] = v;
  }
  if (strstr(name, "k_domain_finalize")) {
    ndom = *(int *)args[1];
    active = *(int **)args[4];
  }
  if (si_launches < RECORDS) {
    strcpy(si_name[si_launches], name);
    if (strstr(name, "k_multi")) memcpy(si_args[si_launches], args[0], 216);
    if (strstr(name, "k_poisson_multi")) memcpy(si_args2[si_launches], args[1], 40);
  }
  ++si_launches;
  return 0;
}
