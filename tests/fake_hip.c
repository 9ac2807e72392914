/* A HIP runtime for tests on the CPU: device memory is host memory, kernels do nothing.  Loaded with RTLD_GLOBAL before
 * libdrx.so, it takes the calls that drx_locate makes; fake_* set which of them fails and what they saw. */
#include <stdlib.h>
#include <string.h>

int fake_fail_malloc = -1, fake_fail_launch = -1;   /* index of the call that fails */
int fake_mallocs = 0, fake_launches = 0, fake_copies = 0, fake_first_copy = 0;
long fake_live = 0;                                 /* bytes of device memory held */
unsigned fake_grid = 0;                             /* blocks of the last launch */
static int last_error = 0;

static int failed (int e) { return last_error = e; }

int hipGetDevice (int *d) { *d = 0; return 0; }
int hipDeviceGetAttribute (int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetLastError (void) { const int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString (int e) { return e == 2 ? "out of memory" : e ? "launch failure" : "no error"; }
int hipMallocAsync (void **p, size_t n, void *st)
{
  (void)st;
  if (fake_mallocs++ == fake_fail_malloc) return failed (2);
  size_t *m = (size_t *)calloc (1, n + 64);
  m[0] = n;
  fake_live += (long)n;
  *p = (char *)m + 64;
  return 0;
}
int hipFreeAsync (void *p, void *st)
{
  (void)st;
  size_t *m = (size_t *)((char *)p - 64);
  fake_live -= (long)m[0];
  free (m);
  return 0;
}
int hipHostMalloc (void **p, size_t n, unsigned f) { (void)f; *p = calloc (1, n); return 0; }
int hipThreadExchangeStreamCaptureMode (int *m) { (void)m; return 0; }
int hipStreamSynchronize (void *st) { (void)st; return 0; }
int hipMemcpyAsync (void *d, const void *s, size_t n, int k, void *st)
{
  (void)k; (void)st;
  memcpy (d, s, n);
  if (fake_copies++ == 0 && n == 4) *(int *)d = fake_first_copy;
  return 0;
}
typedef struct { unsigned x, y, z; } dim3;
int __hipPushCallConfiguration (dim3 g, dim3 b, size_t s, void *st)
{
  (void)b; (void)s; (void)st;
  fake_grid = g.x;
  return 0;
}
int __hipPopCallConfiguration (dim3 *g, dim3 *b, size_t *s, void **st)
{
  g->x = g->y = g->z = b->x = b->y = b->z = 1;
  *s = 0;
  *st = 0;
  return 0;
}
int hipLaunchKernel (const void *f, dim3 g, dim3 b, void **a, size_t s, void *st)
{
  (void)f; (void)g; (void)b; (void)a; (void)s; (void)st;
  return fake_launches++ == fake_fail_launch ? failed (719) : 0;
}
