/* The HIP runtime and the kernel launchers under openfish_host.c, for tests on the CPU of what the host code asks of them: two devices,
 * "device" memory from malloc, kernels that do nothing.  Errors are kept as the runtime keeps them: the last one stays until
 * hipGetLastError takes it, calls that succeed leave it, and a launcher returns it (hipErrorNotReady is an answer, not kept).
 * Time passes on the streams alone: a kernel takes its stream a millisecond, a marker nothing, and an event's time is its stream's. */
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#include "kernels.h"

int stub_null_busy[2];  /* whether the null stream of a device has work left */
int stub_null_joins;    /* events recorded on a null stream */
int stub_launches;
int stub_intruder; /* milliseconds of another thread's work that every other stream gets right behind a decode's first kernel */
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

typedef struct { int device; float now; } queue_t; /* a stream; of an event, its device and time */
static queue_t null_stream[2] = {{0, 0.0f}, {1, 0.0f}}, streams[64];
static int stream_count;
static queue_t *queue_of(hipStream_t s) { return s ? (queue_t *)s : &null_stream[device]; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned int flags) {
    (void)flags;
    if (stream_count == 64) return said(hipErrorOutOfMemory);
    streams[stream_count].device = device;
    *s = (hipStream_t)&streams[stream_count++];
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { return said(s == NULL && stub_null_busy[device] ? hipErrorNotReady : hipSuccess); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int flags) {
    (void)flags;
    if (((queue_t *)e)->now > queue_of(s)->now) queue_of(s)->now = ((queue_t *)e)->now;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) {
    queue_t *q = calloc(1, sizeof *q);
    q->device = device;
    *e = (hipEvent_t)q;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (((queue_t *)e)->device != queue_of(s)->device) return said(hipErrorInvalidHandle); /* an event and a stream of two devices */
    if (s == NULL) ++stub_null_joins;
    ((queue_t *)e)->now = queue_of(s)->now;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) { *ms = ((queue_t *)b)->now - ((queue_t *)a)->now; return hipSuccess; }
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

static int launched(void *stream, void *done) {
    ++stub_launches;
    queue_of(stream)->now += 1.0f;
    if (done) ((queue_t *)done)->now = queue_of(stream)->now;
    return (int)hipGetLastError();
}
static int launched_first(void *stream, void *done) { /* the kernel that a decode begins with */
    const int rc = launched(stream, done);
    for (int i = 0; i < stream_count; ++i)
        if (&streams[i] != stream) streams[i].now += (float)stub_intruder;
    return rc;
}
int ofk_meet(int *mark, int waits, void *stream) {
    if (!waits) mark[1] = 1;
    return launched(stream, NULL);
}
/* the others take no notice of their arguments */
#define KERNEL { return launched(stream, done); }
#define KERNEL_NO_EVENT { return launched(stream, NULL); }
int ofk_bwd_scan(const void *scores, float *bwd, int T, int N, int state_len, int columns, float stay, int mode, int spl,
                 void *stream, void *done) { return launched_first(stream, done); }
int ofk_scan_posterior(const void *scores, float *bwd, float *post, int T, int N, int state_len, int columns, float stay, int mode, int spl,
                       void *stream, void *done) { return launched_first(stream, done); }
int ofk_fwd_scan(const void *scores, float *fwd, int T, int N, int state_len, int columns, float stay, void *stream, void *done) KERNEL
int ofk_fwd_post_scan(const void *scores, const float *bwd, float *post, int T, int N, int state_len, int columns, float stay, int mode, int spl,
                      void *stream, void *done) KERNEL
int ofk_posterior_rows(const float *bwd, float *post, int T, int N, int state_len, void *stream, void *done) KERNEL
int ofk_beam_search(const void *scores, const float *bwd, ofk_beam_slot_t *beam, int32_t *states, uint8_t *moves, int T, int N, int state_len,
                    int columns, float log_beam_cut, float stay, const double *lse_table, int flags, void *stream, void *done) KERNEL
int ofk_beam_search_forward(const void *scores, const float *bwd, float *post, ofk_beam_slot_t *beam, int32_t *states, uint8_t *moves, int T,
                            int N, int state_len, int columns, float log_beam_cut, float stay, const double *lse_table, int flags,
                            void *stream, void *done) KERNEL
int ofk_path_sums(const float *post, float *sums, int T, int N, int state_len, void *stream, void *done) KERNEL
int ofk_sequence(const float *post, int32_t *states, const uint8_t *moves, float *qual_data, float *base_probs, float *total_probs,
                 char *sequence, char *qstring, int T, int N, int state_len, const ofk_phred_table_t *phred, const float *path_sums,
                 uint8_t *moves_out, void *stream, void *done) KERNEL
int ofk_beam_search_static(const void *scores, const float *bwd, int32_t *states, uint8_t *moves, int T, int N, int state_len, int columns,
                           float log_beam_cut, float stay, int flags, void *stream) KERNEL_NO_EVENT
int ofk_beam_search_static_prepare(const double *lse_table_host) { return 0; }
int ofk_beam_search_static_ready(void) { return 0; }
int ofk_copy(void *dst, const void *src, size_t bytes, void *stream) KERNEL_NO_EVENT
int ofk_rotary_emb(void *x, const float *sin_buf, const float *cos_buf, int batch, int seqlen, int nheads, int rotary_half, long stride_batch,
                   long stride_seq, long stride_head, void *stream) KERNEL_NO_EVENT
int ofk_probe_hw_math(void *scratch40, void *stream) KERNEL_NO_EVENT
