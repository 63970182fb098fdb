/* A HIP runtime without a GPU, for tests of the host code's failure paths on
 * the CPU: loaded globally ahead of libse2w_hip.so, it takes the place of the
 * runtime's entry points.  Device memory is an address that nobody reads, a
 * kernel launch does nothing, an upload moves nothing and a download fills its
 * destination with a byte.  One allocation of a given size can be made to
 * fail. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2, MAX = 4096 };

static struct { void *p; size_t n; int pinned; } live[MAX];
static size_t fail_size[2], next_address = (size_t)1 << 44;
static int fill_byte, downloads, launches, slow;
static char handle;

/* kind 0: device, 1: pinned host */
void fake_fail_next(int kind, size_t bytes) { fail_size[kind] = bytes; }
void fake_fill(int byte) { fill_byte = byte; }
void fake_slow(int n) { slow = n; }  /* the next n times between events are twice as long */
int fake_downloads(void) { return downloads; }
int fake_launches(void) { return launches; }
size_t fake_live(int kind)
{
  size_t s = 0;
  for (int i = 0; i < MAX; i++) if (live[i].p && live[i].pinned == kind) s += live[i].n;
  return s;
}

static int take(void **p, size_t n, int kind)
{
  if (fail_size[kind] && fail_size[kind] == n) { fail_size[kind] = 0; return OUT_OF_MEMORY; }
  *p = kind ? calloc(1, n ? n : 1) : (void *)next_address;
  if (!*p) return OUT_OF_MEMORY;
  if (!kind) next_address += (n + 4095) / 4096 * 4096;
  for (int i = 0; i < MAX; i++)
    if (!live[i].p) { live[i].p = *p; live[i].n = n; live[i].pinned = kind; return OK; }
  abort();
}

static int give(void *p, int kind)
{
  for (int i = 0; i < MAX; i++)
    if (live[i].p == p && p) {
      if (live[i].pinned != kind) abort();
      live[i].p = NULL;
      if (kind) free(p);
      return OK;
    }
  return p ? 1 : OK;
}

int hipMalloc(void **p, size_t n) { return take(p, n, 0); }
int hipFree(void *p) { return give(p, 0); }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; return take(p, n, 1); }
int hipHostFree(void *p) { return give(p, 1); }

int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st)
{
  (void)s; (void)st;
  if (kind == 2) { memset(d, fill_byte, n); downloads++; }
  return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return hipMemcpyAsync(d, s, n, kind, NULL); }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)d; (void)v; (void)n; (void)st; return OK; }

int hipSetDevice(int d) { (void)d; return OK; }
int hipGetLastError(void) { return OK; }
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "error"; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = (void *)((size_t)1 << 43); return OK; }

int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = &handle; return OK; }
int hipStreamDestroy(void *s) { (void)s; return OK; }
int hipStreamSynchronize(void *s) { (void)s; return OK; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { (void)s; (void)e; (void)f; return OK; }
int hipEventCreate(void **e) { *e = &handle; return OK; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = &handle; return OK; }
int hipEventDestroy(void *e) { (void)e; return OK; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return OK; }
int hipEventSynchronize(void *e) { (void)e; return OK; }
int hipEventElapsedTime(float *ms, void *a, void *b)
{
  (void)a; (void)b;
  *ms = slow > 0 ? 2.0f : 1.0f;
  slow -= slow > 0;
  return OK;
}

int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return OK; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = &handle; return OK; }
int hipGraphInstantiate(void **x, void *g, void *n, char *b, size_t z)
{
  (void)g; (void)n; (void)b; (void)z;
  *x = &handle;
  return OK;
}
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; return OK; }
int hipGraphDestroy(void *g) { (void)g; return OK; }
int hipGraphExecDestroy(void *x) { (void)x; return OK; }

typedef struct { uint32_t x, y, z; } dim3_t;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t sh, void *s) { (void)g; (void)b; (void)sh; (void)s; return OK; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *sh, void **s)
{
  g->x = g->y = g->z = b->x = b->y = b->z = 1;
  *sh = 0;
  *s = NULL;
  return OK;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t sh, void *s)
{
  (void)f; (void)g; (void)b; (void)a; (void)sh; (void)s;
  launches++;
  return OK;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int t, size_t sh)
{
  (void)f; (void)t; (void)sh;
  *n = 1;
  return OK;
}
