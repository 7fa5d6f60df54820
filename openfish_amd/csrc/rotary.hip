// In-place rotary embedding on half data with fp32 sin/cos tables, gfx950.
//
// For every (batch, seq, head, rot < rotary_half) the pair
//   x0 = x[batch*stride_batch + seq*stride_seq + head*stride_head + rot], x1 = x0's partner at +rotary_half
// becomes (x0*cos - x1*sin, x0*sin + x1*cos) with cos/sin taken at [seq][rot]
// (reference src/rotary_emb_hip.h:36-70, CPU twin src/nn_cpu.c:10-39).  Products and
// sums are separate fp32 operations (no fused multiply-add), the result is rounded
// to half once.  The op is pure streaming; what bounds it is how whole the pieces are
// that a wave asks memory for:
//   rows    rotary_half a power of two from 8 to 64: a wave's loads and stores are whole lines;
//   vec8    other multiples of 8, single and short batches: 8 pairs per thread with 128-bit loads and stores;
//   narrow  everything else: 4, 2 or 1 pairs per thread.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void rotary_vec8_kernel(_Float16 *__restrict__ x, const float *__restrict__ sin_buf,
                                                          const float *__restrict__ cos_buf, long total, int seqlen,
                                                          int nheads, int groups, int rotary_half, long stride_batch,
                                                          long stride_seq, long stride_head) {
    const long id = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= total) return;
    const int grp = (int)(id % groups);
    long rest = id / groups;
    const int head = (int)(rest % nheads);
    rest /= nheads;
    const int seq = (int)(rest % seqlen);
    const long batch = rest / seqlen;
    const int rot = grp * 8;

    _Float16 *p0 = x + batch * stride_batch + (long)seq * stride_seq + (long)head * stride_head + rot;
    _Float16 *p1 = p0 + rotary_half;
    const long tab = (long)seq * rotary_half + rot;
    const float4v c0 = *reinterpret_cast<const float4v *>(cos_buf + tab);
    const float4v c1 = *reinterpret_cast<const float4v *>(cos_buf + tab + 4);
    const float4v s0 = *reinterpret_cast<const float4v *>(sin_buf + tab);
    const float4v s1 = *reinterpret_cast<const float4v *>(sin_buf + tab + 4);
    const half8 a = *reinterpret_cast<const half8 *>(p0);
    const half8 b = *reinterpret_cast<const half8 *>(p1);
    half8 ra, rb;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float c = k < 4 ? c0[k & 3] : c1[k & 3];
        const float s = k < 4 ? s0[k & 3] : s1[k & 3];
        const float x0 = (float)a[k], x1 = (float)b[k];
        ra[k] = (_Float16)(x0 * c - x1 * s);
        rb[k] = (_Float16)(x0 * s + x1 * c);
    }
    *reinterpret_cast<half8 *>(p0) = ra;
    *reinterpret_cast<half8 *>(p1) = rb;
}

struct __attribute__((aligned(16))) Table8 {
    float v[8];
};

// A lane holds 16 consecutive bytes of a head, of its first halves or of its second, and gets the partners of its eight values
// from the lane that holds those: a wave asks for 1024 consecutive bytes where the pairs' own order gives pieces of
// 2 rotary_half bytes.  Two batches to a lane share the sines and cosines, which are twice what it reads of x, and keep as
// much in flight as a lane of rotary_vec8_kernel does.  500 x 833 x 8 heads of 64: 165 us -> 144 (5.9 TB/s; one batch to a
// lane 150, four 149); heads of 32, 500 x 400 x 8: 41 -> 36; 31 x 833 x 8 heads of 64: 13.1 -> 12.1;
// heads of 128, whose pieces are lines already: 144 -> 143.
__global__ __launch_bounds__(256) void rotary_rows_kernel(_Float16 *__restrict__ x, const float *__restrict__ sin_buf,
                                                          const float *__restrict__ cos_buf, unsigned per_batch, int batch,
                                                          unsigned nheads, int log_lanes, int rotary_half, long stride_batch,
                                                          long stride_seq, long stride_head) {
    typedef int int4v __attribute__((ext_vector_type(4)));
    const unsigned id = blockIdx.x * 256 + threadIdx.x;
    if (id >= per_batch) return;  // all lanes of a head or none
    const int lanes = 1 << log_lanes, mate = lanes >> 1;
    const unsigned row = id >> log_lanes, seq = row / nheads, head = row - seq * nheads;
    const int at = (int)(id & (unsigned)(lanes - 1));
    const bool first = at < mate;
    const long tab = (long)seq * rotary_half + (at & (mate - 1)) * 8;
    const Table8 c = *reinterpret_cast<const Table8 *>(cos_buf + tab), s = *reinterpret_cast<const Table8 *>(sin_buf + tab);
    _Float16 *const p = x + (long)seq * stride_seq + (long)head * stride_head + at * 8;
    auto turn = [&](const half8 &own) {
        int4v w = __builtin_bit_cast(int4v, own);
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = __shfl_xor(w[k], mate);
        const half8 other = __builtin_bit_cast(half8, w);
        half8 r;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float a = (float)own[k] * c.v[k], b = (float)other[k] * s.v[k];
            r[k] = (_Float16)(first ? a - b : b + a);
        }
        return r;
    };
    for (long b = 2 * (long)blockIdx.y; b < batch; b += 2 * (long)gridDim.y) {
        half8 *const p0 = reinterpret_cast<half8 *>(p + b * stride_batch);
        half8 *const p1 = reinterpret_cast<half8 *>(p + (b + 1) * stride_batch);
        const bool two = b + 1 < batch;
        const half8 own0 = *p0;
        half8 own1;
        if (two) own1 = *p1;
        *p0 = turn(own0);
        if (two) *p1 = turn(own1);
    }
}

template <typename T, int V>
using Run = T __attribute__((ext_vector_type(V)));

// V pairs per thread, indexes in 32 bits: a grid has fewer threads.  500 x 833 x 8 heads of 24 (V = 4): 137 us -> 62 against a pair
// per thread and 64-bit divisions; 100 x 833 x 8 of 12 (V = 2) 18 -> 11, of 6 (V = 1) 9.6 -> 8.7.
template <int V>
__global__ __launch_bounds__(256) void rotary_narrow_kernel(_Float16 *__restrict__ x, const float *__restrict__ sin_buf,
                                                            const float *__restrict__ cos_buf, unsigned total, unsigned seqlen,
                                                            unsigned nheads, unsigned groups, int rotary_half, long stride_batch,
                                                            long stride_seq, long stride_head) {
    typedef Run<_Float16, V> Half;
    typedef Run<float, V> Float;
    const unsigned id = blockIdx.x * 256 + threadIdx.x;
    if (id >= total) return;
    const unsigned at_head = id / groups, at_seq = at_head / nheads, batch = at_seq / seqlen;
    const unsigned rot = (id - at_head * groups) * V, head = at_head - at_seq * nheads, seq = at_seq - batch * seqlen;
    _Float16 *p0 = x + (long)batch * stride_batch + (long)seq * stride_seq + (long)head * stride_head + rot;
    _Float16 *p1 = p0 + rotary_half;
    const long tab = (long)seq * rotary_half + rot;
    const Float c = *reinterpret_cast<const Float *>(cos_buf + tab), s = *reinterpret_cast<const Float *>(sin_buf + tab);
    const Half a = *reinterpret_cast<const Half *>(p0), b = *reinterpret_cast<const Half *>(p1);
    Half ra, rb;
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const float x0 = (float)a[k], x1 = (float)b[k];
        ra[k] = (_Float16)(x0 * c[k] - x1 * s[k]);
        rb[k] = (_Float16)(x0 * s[k] + x1 * c[k]);
    }
    *reinterpret_cast<Half *>(p0) = ra;
    *reinterpret_cast<Half *>(p1) = rb;
}

template <int V>
int launch_narrow(_Float16 *x, const float *sin_buf, const float *cos_buf, int batch, int seqlen, int nheads, int rotary_half,
                  long stride_batch, long stride_seq, long stride_head, hipStream_t st) {
    const unsigned __int128 total = (unsigned __int128)((unsigned long)batch * (unsigned long)seqlen) *
                                    ((unsigned long)nheads * (unsigned long)(rotary_half / V));
    if (total > 0xffffff00u) return OFK_BAD_ARGS;  // a grid has less than 2^32 threads
    const unsigned n = (unsigned)total;
    hipLaunchKernelGGL((rotary_narrow_kernel<V>), dim3((n + 255) / 256), dim3(256), 0, st, x, sin_buf, cos_buf, n, (unsigned)seqlen,
                       (unsigned)nheads, (unsigned)(rotary_half / V), rotary_half, stride_batch, stride_seq, stride_head);
    return (int)hipGetLastError();
}

}  // namespace

extern "C" int ofk_rotary_emb(void *x, const float *sin_buf, const float *cos_buf, int batch, int seqlen,
                              int nheads, int rotary_half, long stride_batch, long stride_seq,
                              long stride_head, void *stream) {
    if (!x || !sin_buf || !cos_buf || batch < 0 || seqlen < 0 || nheads < 0 || rotary_half < 0) return OFK_BAD_ARGS;
    if (batch == 0 || seqlen == 0 || nheads == 0 || rotary_half == 0) return 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    _Float16 *const halves = static_cast<_Float16 *>(x);
    // how far apart and how aligned everything is: 2 V bytes of x and 4 V of the tables, up to the 16 of a load, for V pairs at once
    const unsigned long apart = (unsigned long)rotary_half | (unsigned long)stride_batch | (unsigned long)stride_seq | (unsigned long)stride_head;
    const uintptr_t data = reinterpret_cast<uintptr_t>(x), tables = reinterpret_cast<uintptr_t>(sin_buf) | reinterpret_cast<uintptr_t>(cos_buf);
    if (apart % 8 == 0 && data % 16 == 0 && tables % 16 == 0) {
        // Rows: heads of up to 128, batches for every lane to have two (3 x 1700 x 12 heads of 64: 5.2 us | 5.3), and batches whose last
        // workgroup's idle lanes are few beside the rest (500 x 1700 heads of 16, 14 workgroups for 3400 lanes a batch: 15.3 us | 13.2;
        // 70000 batches of 2 lanes 3.5 | 17.8).  Batches that fit the launch's own time take the same either way.  Larger heads gain
        // nothing in general: whole calls, us, vec8 | rows, heads of 256: 100 x 833 x 4 61.5 | 65.0, 500 x 833 71.8 | 74.4, 500 x 833 x 4 300 | 308,
        // 16 x 1700 x 12 63.9 | 63.1, 1000 x 833 174 | 161; heads of 512: 64 x 833 x 8 158.8 | 162.9, 500 x 833 175 | 160.
        const unsigned __int128 per_batch = (unsigned __int128)((unsigned long)seqlen * (unsigned long)nheads) * (unsigned)(rotary_half / 4);
        if (rotary_half >= 8 && rotary_half <= 64 && (rotary_half & (rotary_half - 1)) == 0 && batch >= 4 && per_batch >= 2048 && per_batch <= 0xffffff00u) {
            const unsigned n = (unsigned)per_batch;
            const long pairs = ((long)batch + 1) / 2;
            hipLaunchKernelGGL(rotary_rows_kernel, dim3((n + 255) / 256, (unsigned)(pairs < 65535 ? pairs : 65535)), dim3(256), 0, st,
                               halves, sin_buf, cos_buf, n, batch, (unsigned)nheads, __builtin_ctz((unsigned)rotary_half / 4),
                               rotary_half, stride_batch, stride_seq, stride_head);
            return (int)hipGetLastError();
        }
        const int groups = rotary_half / 8;
        const long total = (long)batch * seqlen * nheads * groups;
        const long blocks = (total + 255) / 256;
        if (blocks > 0x7fffffffL) return OFK_BAD_ARGS;
        hipLaunchKernelGGL(rotary_vec8_kernel, dim3((unsigned)blocks), dim3(256), 0, st, halves, sin_buf, cos_buf, total, seqlen, nheads,
                           groups, rotary_half, stride_batch, stride_seq, stride_head);
        return (int)hipGetLastError();
    }
    const auto narrow = apart % 4 == 0 && data % 8 == 0 && tables % 16 == 0 ? launch_narrow<4>
                        : apart % 2 == 0 && data % 4 == 0 && tables % 8 == 0 ? launch_narrow<2> : launch_narrow<1>;
    return narrow(halves, sin_buf, cos_buf, batch, seqlen, nheads, rotary_half, stride_batch, stride_seq, stride_head, st);
}
