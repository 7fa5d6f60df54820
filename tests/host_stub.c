/* The HIP runtime and the kernel launchers under openfish_host.c, for tests on the CPU of what the host code asks of them: two devices,
 * "device" memory from malloc, kernels that do nothing.  Errors are kept as the runtime keeps them: the last one stays until
 * hipGetLastError takes it, calls that succeed leave it, and a launcher returns it (hipErrorNotReady is an answer, not kept). */
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

int stub_null_busy[2];  /* whether the null stream of a device has work left */
int stub_null_joins;    /* events recorded on a null stream */
int stub_launches;
static int device;
static hipError_t last;

static hipError_t said(hipError_t e) {
    if (e != hipSuccess && e != hipErrorNotReady) last = e;
    return e;
}

hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return said(hipErrorInvalidDevice);
    device = d;
    return hipSuccess;
}
void stub_fail(void) { (void)said(hipErrorInvalidConfiguration); } /* a caller's own call that failed, its error not looked at */
hipError_t hipGetLastError(void) {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipPeekAtLastError(void) { return last; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorInvalidConfiguration ? "invalid configuration" : e == hipErrorInvalidHandle ? "invalid handle" : "error"; }

/* a stream or an event remembers its device: one past its number, as a pointer that is never followed */
static void *of_device(int d) { return (void *)(size_t)(d + 1); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int flags) { (void)flags; *s = (hipStream_t)of_device(device); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { return said(s == NULL && stub_null_busy[device] ? hipErrorNotReady : hipSuccess); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int flags) { (void)s; (void)e; (void)flags; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)of_device(device); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if ((void *)e != (s ? (void *)s : of_device(device))) return said(hipErrorInvalidHandle); /* an event and a stream of two devices */
    if (s == NULL) ++stub_null_joins;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 0.0f; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = aligned_alloc(256, (n + 255) / 256 * 256); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned int flags) { (void)flags; *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned int flags) { (void)flags; *d = h; return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { (void)k; (void)st; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemGetInfo(size_t *free_b, size_t *total) { *free_b = *total = 0; return hipSuccess; }

static int launched(void) {
    ++stub_launches;
    return (int)hipGetLastError();
}
int ofk_meet(int *mark, int waits, void *stream) {
    (void)stream;
    if (!waits) mark[1] = 1;
    return launched();
}
/* the others take no notice of their arguments (kernels.h is left out: these are not its declarations) */
#define LAUNCHER(name) int name(void) { return launched(); }
LAUNCHER(ofk_bwd_scan)
LAUNCHER(ofk_fwd_scan)
LAUNCHER(ofk_fwd_post_scan)
LAUNCHER(ofk_posterior_rows)
LAUNCHER(ofk_scan_posterior)
LAUNCHER(ofk_beam_search)
LAUNCHER(ofk_beam_search_forward)
LAUNCHER(ofk_beam_search_static)
LAUNCHER(ofk_beam_search_static_prepare)
LAUNCHER(ofk_beam_search_static_ready)
LAUNCHER(ofk_path_sums)
LAUNCHER(ofk_sequence)
LAUNCHER(ofk_copy)
LAUNCHER(ofk_rotary_emb)
LAUNCHER(ofk_probe_hw_math)
