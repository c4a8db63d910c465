/* Stands in for the HIP runtime's memory calls on a machine without a GPU: a
 * device of 256 CUs with shim_set_free() bytes of memory, which is host memory
 * here.  For tests of what the library allocates, what it does when that does not
 * fit, and how it copies; nothing is launched.  Test infrastructure. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

static size_t free_bytes = (size_t)1 << 62, in_use;

void shim_set_free(size_t n) { free_bytes = n; }
size_t shim_in_use(void) { return in_use; }

hipError_t hipMalloc(void **p, size_t n) {
    if (n > free_bytes) return hipErrorOutOfMemory;
    size_t *q = malloc(n + 64);
    if (!q) return hipErrorOutOfMemory;
    q[0] = n;
    free_bytes -= n;
    in_use += n;
    *p = (char *)q + 64;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    size_t *q = (size_t *)((char *)p - 64);
    free_bytes += q[0];
    in_use -= q[0];
    free(q);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return (void)k, memcpy(d, s, n), hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int d) {
    (void)d;
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return *s = NULL, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return (void)s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return (void)s, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }

/* Copies, events and launches for downloads: copies are made at once, kernels do
 * nothing (loaded fields are then the fields read back). */
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)st;
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t st) { return (void)st, hipMemset(p, v, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { return (void)f, *p = malloc(n), *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipSetDevice(int d) { return (void)d, hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { return (void)f, *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return (void)e, (void)s, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return (void)e, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    (void)p;
    memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    (void)s;
    return *st = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, hipStream_t s) {
    (void)f, (void)g, (void)b, (void)args, (void)lds, (void)s;
    return hipSuccess;
}

/* In a program of its own: a new thread first runs after shim_set_thread_delay() ms, as one
 * does that gets no CPU. */
static int delay_ms;
static int started;
void shim_set_thread_delay(int ms) { delay_ms = ms; }
int shim_threads_started(void) { return __atomic_load_n(&started, __ATOMIC_SEQ_CST); }

struct start {
    void *(*fn)(void *);
    void *arg;
    int ms;
};
static void *late(void *p) {
    struct start s = *(struct start *)p;
    free(p);
    usleep((useconds_t)s.ms * 1000);
    return s.fn(s.arg);
}
int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*fn)(void *), void *arg) {
    int (*real)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    *(void **)&real = dlsym(RTLD_NEXT, "pthread_create");
    if (!delay_ms) return real(t, a, fn, arg);
    struct start *s = malloc(sizeof *s);
    s->fn = fn, s->arg = arg, s->ms = delay_ms;
    __atomic_add_fetch(&started, 1, __ATOMIC_SEQ_CST);
    return real(t, a, late, s);
}
