/* The HIP calls of libcathy_gpu.so on host memory, for tests without a GPU
 * (LD_PRELOAD): allocations and copies work, launches do nothing.
 * hip_stub_fail(k) lets the k-th allocation from now fail (0: the next);
 * hip_stub_live() counts the device allocations held, hip_stub_copies(p) the
 * copies made to p. */
#include <stdlib.h>
#include <string.h>

static int fail_at = -1, live = 0;
void hip_stub_fail(int k) { fail_at = k; }
int hip_stub_live(void) { return live; }

static void *copied[4096];
static int ncopied = 0;
int hip_stub_copies(void *p) {
  int c = 0;
  for (int i = 0; i < ncopied && i < 4096; ++i) c += copied[i] == p;
  return c;
}

int hipMalloc(void **p, size_t n) {
  if (fail_at >= 0 && fail_at-- == 0) { *p = 0; return 2; /* hipErrorOutOfMemory */ }
  *p = calloc(n ? n : 1, 1);
  ++live;
  return *p ? 0 : 2;
}
int hipFree(void *p) { if (p) { --live; free(p); } return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(n ? n : 1, 1); return 0; }
int hipHostFree(void *p) { free(p); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) {
  (void)k; (void)st;
  if (n && (!d || !s)) return 1; /* hipErrorInvalidValue */
  copied[ncopied++ % 4096] = d;
  memcpy(d, s, n);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; if (n && !d) return 1; memset(d, v, n); return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = (void *)1; return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) { (void)s; return 0; }
int hipEventCreate(void **e) { *e = (void *)1; return 0; }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0.f; return 0; }
int hipGetLastError(void) { return 0; }
int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetDeviceCount(int *c) { *c = 1; return 0; }
typedef struct { unsigned x, y, z; } grid3;
int hipLaunchKernel(const void *f, grid3 g, grid3 b, void **a, size_t sm, void *s) {
  (void)f; (void)g; (void)b; (void)a; (void)sm; (void)s;
  return 0;
}
