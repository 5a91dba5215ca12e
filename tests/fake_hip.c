/* A HIP runtime without a device, for the host side of the library: loaded
 * with RTLD_GLOBAL before libh3dmg.so, its functions are the ones the library
 * calls.  Device memory is host memory, kernels do nothing, and a
 * host-to-device copy happens when its stream is next waited for, as a device
 * may do it: a source that changed in between (freed, or gone out of scope)
 * is counted by fake_late_sources(). */
#include <stdlib.h>
#include <string.h>

typedef struct {
  void *dst;
  const void *src;
  size_t n;
  unsigned char *was;
} Copy;
static Copy pending[4096];
static int npending, late;
static size_t room = (size_t)1 << 40; /* bytes hipMalloc still gives */

int fake_late_sources(void) { return late; }
void fake_set_room(size_t bytes) { room = bytes; }
size_t fake_room(void) { return room; }

static void finish(void) {
  for (int q = 0; q < npending; ++q) {
    Copy *c = &pending[q];
    late += memcmp(c->was, c->src, c->n) != 0;
    memcpy(c->dst, c->was, c->n);
    free(c->was);
  }
  npending = 0;
}

int hipMalloc(void **p, size_t n) { /* its size lies before the memory */
  size_t *q = n > room ? NULL : calloc(n + 64, 1);
  if (!q) return 2; /* hipErrorOutOfMemory */
  room -= *q = n;
  *p = q + 8;
  return 0;
}
int hipFree(void *p) {
  finish();
  if (p) room += *((size_t *)p - 8), free((size_t *)p - 8);
  return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned f) {
  (void)f;
  return (*p = calloc(n, 1)) ? 0 : 2;
}
int hipHostFree(void *p) {
  finish();
  free(p);
  return 0;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned f) {
  (void)f;
  *d = h;
  return 0;
}
int hipMemcpyAsync(void *dst, const void *src, size_t n, int kind, void *s) {
  (void)s;
  if (kind != 1 || npending == 4096) { /* not hipMemcpyHostToDevice */
    finish();
    memmove(dst, src, n);
    return 0;
  }
  Copy c = {dst, src, n, malloc(n ? n : 1)};
  memcpy(c.was, src, n);
  pending[npending++] = c;
  return 0;
}
int hipMemcpy(void *dst, const void *src, size_t n, int kind) {
  (void)kind;
  finish();
  memmove(dst, src, n);
  return 0;
}
int hipMemsetAsync(void *p, int v, size_t n, void *s) {
  (void)s;
  finish();
  memset(p, v, n);
  return 0;
}
int hipStreamSynchronize(void *s) { (void)s; finish(); return 0; }
int hipDeviceSynchronize(void) { finish(); return 0; }
int hipEventSynchronize(void *e) { (void)e; finish(); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = malloc(1); return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = malloc(1); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = malloc(1); return 0; }
int hipGraphInstantiate(void **x, void *g, void *n, char *l, size_t b) {
  (void)g; (void)n; (void)l; (void)b;
  *x = malloc(1);
  return 0;
}
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; return 0; }
int hipGraphExecDestroy(void *x) { free(x); return 0; }
int hipGraphDestroy(void *g) { free(g); return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 160 * 1024; return 0; }
int hipFuncSetAttribute(const void *f, int a, int v) { (void)f; (void)a; (void)v; return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { return e ? "out of memory" : "no error"; }
int hipGetSymbolAddress(void **p, const void *s) { *p = (void *)s; return 0; }
int hipLaunchKernel(const void *f, ...) { (void)f; return 0; }
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void) { return 0; }
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipRegisterFunction(void) {}
void __hipRegisterVar(void) {}
void __hipUnregisterFatBinary(void **h) { (void)h; }
