/* A stand-in for the HIP runtime on the CPU, for tests of the library's host code: allocations are untouched address
 * space, copies and fills do nothing (what comes to the host is zeros), launches are counted, and one of them or the pinned
 * allocations can be made to fail. No kernel runs, so no result means anything. A 256-CU device that holds fake_per_cu workgroups of any kernel a
 * CU. Loaded with RTLD_GLOBAL before the library, whose HIP calls then land here. */
#define _GNU_SOURCE
#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

typedef struct { uint32_t x, y, z; } dim3;
typedef void* stream_t;
enum { OK = 0, INVALID = 1, NOMEM = 2 };

int fake_fail_host_malloc, fake_fail_launch = -1 /* the launch to fail, counted from 0 */, fake_per_cu = 1;
int fake_launches, fake_copies, fake_streams, fake_mallocs;
int fake_pending;      /* launches and asynchronous copies since the last synchronization of their stream (any stream) */
int fake_freed_busy;   /* pinned buffers freed with some pending */
static int pending_of[64], last_error;
static struct { dim3 g, b; size_t shared; stream_t s; } call;

static int slot(stream_t s) { return (int)((uintptr_t)s % 64); }
static void queued(stream_t s) { pending_of[slot(s)]++, fake_pending++; }
static int map(void** p, size_t n) {
  *p = mmap(NULL, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return *p == MAP_FAILED ? NOMEM : OK;
}

int hipGetDeviceCount(int* n) { return *n = 1, OK; }
int hipGetDevice(int* d) { return *d = 0, OK; }
int hipDeviceGetAttribute(int* v, int attr, int dev) { return (void)attr, (void)dev, *v = 256, OK; }
int hipFuncSetAttribute(const void* f, int attr, int v) { return (void)f, (void)attr, (void)v, OK; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int threads, size_t lds) {
  return (void)f, (void)threads, (void)lds, *n = fake_per_cu, OK;
}
int hipGetSymbolAddress(void** p, const void* symbol) { return (void)symbol, map(p, 8 << 20); }
int hipMalloc(void** p, size_t n) { return fake_mallocs++, map(p, n); }
int hipFree(void* p) { return (void)p, OK; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  return (void)flags, fake_fail_host_malloc ? (last_error = NOMEM) : map(p, n);
}
int hipHostFree(void* p) { return (void)p, fake_freed_busy += fake_pending != 0, OK; }
int hipStreamCreateWithFlags(stream_t* s, unsigned flags) {
  return (void)flags, *s = (stream_t)(uintptr_t)(++fake_streams), OK;
}
int hipStreamDestroy(stream_t s) { return (void)s, OK; }
int hipStreamSynchronize(stream_t s) { return fake_pending -= pending_of[slot(s)], pending_of[slot(s)] = 0, OK; }
int hipMemcpy(void* d, const void* s, size_t n, int kind) {
  if (kind == 2 /* to the host */) memset(d, 0, n);
  return (void)s, fake_copies++, OK;
}
int hipMemcpyAsync(void* d, const void* src, size_t n, int kind, stream_t s) {
  return queued(s), hipMemcpy(d, src, n, kind);
}
int hipMemsetAsync(void* d, int v, size_t n, stream_t s) { return (void)d, (void)v, (void)n, queued(s), OK; }
int hipMemsetD32Async(void* d, int v, size_t n, stream_t s) { return (void)d, (void)v, (void)n, queued(s), OK; }
int hipEventCreate(void** e) { return *e = NULL, OK; }
int hipEventDestroy(void* e) { return (void)e, OK; }
int hipEventRecord(void* e, stream_t s) { return (void)e, (void)s, OK; }
int hipEventSynchronize(void* e) { return (void)e, OK; }
int hipEventElapsedTime(float* ms, void* a, void* b) { return (void)a, (void)b, *ms = 0, OK; }
int hipGetLastError(void) {
  const int e = last_error;
  return last_error = OK, e;
}
const char* hipGetErrorString(int e) { return e == NOMEM ? "out of memory" : e ? "invalid" : "no error"; }
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, stream_t s) {
  return call.g = g, call.b = b, call.shared = shared, call.s = s, OK;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, stream_t* s) {
  return *g = call.g, *b = call.b, *shared = call.shared, *s = call.s, OK;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t shared, stream_t s) {
  (void)f, (void)args;
  if (fake_launches++ == fake_fail_launch) return last_error = INVALID;
  if (shared > 160 * 1024 || !g.x || !g.y || !g.z || b.x * b.y * b.z > 1024) return last_error = INVALID;
  return queued(s), OK;
}
