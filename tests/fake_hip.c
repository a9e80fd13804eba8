/* A HIP runtime for the host paths around the kernels, without a device:
 * memory comes from calloc, kernels do not run, and the calls that may fail
 * fail when told to.  Loaded before the library, its functions take the
 * runtime's place.  It counts what a call left behind: allocations, streams
 * with copies from or to pageable memory (the caller's, mostly) that nobody
 * waited for, copies through NULL, and bytes moved.
 * Interfaces: the HIP runtime API's public signatures. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, NO_MEMORY = 2 };
typedef struct {
  int queued;
} stream_t;

static long countdown, failed, live, nulls, h2d, launches, calls, bytes;
static stream_t *streams[64];
static int nstreams;
static struct {
  char *p;
  size_t n;
} pinned[256];

static int fails(void) {
  calls++;
  if (countdown > 0 && --countdown == 0) {
    failed = 1;
    return 1;
  }
  return 0;
}

/* the k-th call from now that may fail does (0: none) */
void fake_fail_at(long k) {
  countdown = k;
  failed = 0;
}
long fake_failed(void) { return failed; }
long fake_live(void) { return live; }
long fake_nulls(void) { return nulls; }
long fake_launches(void) { return launches; }
long fake_calls(void) { return calls; }
long fake_h2d_bytes(void) { return h2d; }
long fake_device_bytes(void) { return bytes; } /* allocated so far */
long fake_queued(void) {
  long q = 0;
  for (int k = 0; k < nstreams; k++)
    q += streams[k] && streams[k]->queued;
  return q;
}

static int make(void **p, size_t n) {
  if (fails())
    return NO_MEMORY;
  *p = calloc(n ? n : 1, 1);
  live++;
  return OK;
}
static int drop(void *p) {
  if (p) {
    free(p);
    live--;
  }
  return OK;
}
static int copy(void *d, const void *s, size_t n, int kind, stream_t *st) {
  if (fails())
    return NO_MEMORY;
  if (!d || !s) {
    nulls += n > 0;
    return OK;
  }
  if (kind == 1)
    h2d += (long)n;
  memcpy(d, s, n);
  const char *host = kind == 1 ? s : d;
  for (int k = 0; k < 256; k++)
    if (pinned[k].p && host >= pinned[k].p && host < pinned[k].p + pinned[k].n)
      return OK;
  if (st && (kind == 1 || kind == 2))
    st->queued = 1;
  return OK;
}

int hipGetDeviceCount(int *n) { return *n = 1, OK; }
int hipSetDevice(int d) { return (void)d, OK; }
int hipDeviceGetAttribute(int *v, int a, int d) { return (void)a, (void)d, *v = 4, OK; }
int hipGetLastError(void) { return fails() ? NO_MEMORY : OK; } /* a launch that failed */
const char *hipGetErrorString(int e) { return e ? "told to fail" : "no error"; }
int hipMalloc(void **p, size_t n) { return *p = NULL, bytes += (long)n, make(p, n); }
int hipFree(void *p) { return drop(p); }
int hipHostMalloc(void **p, size_t n, unsigned f) {
  (void)f;
  *p = NULL;
  int rc = make(p, n);
  for (int k = 0; k < 256 && !rc; k++)
    if (!pinned[k].p) {
      pinned[k].p = *p;
      pinned[k].n = n;
      break;
    }
  return rc;
}
int hipHostFree(void *p) {
  for (int k = 0; k < 256; k++)
    if (p && pinned[k].p == p)
      pinned[k].p = NULL;
  return drop(p);
}
int hipGetSymbolAddress(void **p, const void *s) {
  static char scratch[1 << 20];
  return (void)s, *p = scratch, OK;
}
int hipMemset(void *p, int v, size_t n) { return memset(p, v, n), OK; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) { return copy(d, s, n, kind, NULL); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) { return copy(d, s, n, kind, st); }
int hipLaunchKernel(const void *f, ...) {
  (void)f;
  launches++;
  return OK;
}
int hipStreamCreateWithFlags(void **s, unsigned f) {
  (void)f;
  int rc = make(s, sizeof(stream_t));
  if (!rc && nstreams < 64)
    streams[nstreams++] = *s;
  return rc;
}
int hipStreamDestroy(void *s) {
  for (int k = 0; k < nstreams; k++)
    if (streams[k] == s)
      streams[k] = NULL;
  return drop(s);
}
int hipStreamSynchronize(void *s) {
  if (s)
    ((stream_t *)s)->queued = 0;
  return OK;
}
int hipStreamWaitEvent(void *s, void *e, unsigned f) { return (void)s, (void)f, nulls += !e, fails() ? NO_MEMORY : OK; }
int hipEventCreate(void **e) { return make(e, 8); }
int hipEventCreateWithFlags(void **e, unsigned f) { return (void)f, make(e, 8); }
int hipEventDestroy(void *e) { return drop(e); }
int hipEventRecord(void *e, void *s) { return (void)s, nulls += !e, fails() ? NO_MEMORY : OK; }
int hipEventSynchronize(void *e) { return (void)e, OK; }
int hipEventElapsedTime(float *ms, void *a, void *b) { return (void)a, (void)b, *ms = 1.f, OK; }
