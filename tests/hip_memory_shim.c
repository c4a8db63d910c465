/* Stands in for the HIP runtime's memory calls on a machine without a GPU: a
 * device of 256 CUs with shim_set_free() bytes of memory, which is host memory
 * here.  For tests of what the library allocates and what it does when that does
 * not fit; nothing is launched.  Test infrastructure. */
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

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
