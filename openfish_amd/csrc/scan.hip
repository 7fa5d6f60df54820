// Backward and forward log-space scans over the 4^state_len CRF states, gfx950.
//
// The k-mer transition graph has a quad structure: the four states {4q+j} share
// the four predecessors {q + b*S/4} and the 16 contiguous scores [16q, 16q+16)
// (element 4j+b is the transition pred b -> state 4q+j).  A lane owns SPL = 4, 2 or 1
// states of one quad:
//   forward : owns SPL consecutive states of the contiguous quad {4q+j}, needs the
//             strided quad of the previous vector (4 LDS reads); its own values
//             stay in registers;
//   backward: owns SPL consecutive members of the strided quad {r + c*S/4}, needs
//             the contiguous quad {4r+b} of the next vector (one 128-bit LDS read).
// Per time step a lane reads its 8*SPL bytes of fp16 scores (a wave reads whole
// rows, every cache line fully used), the state vector is exchanged through LDS
// and, when a chunk fits one wavefront, no block barrier is needed.  SPL is chosen
// at launch so that the batch fills the 1024 SIMDs of the device: few chunks are
// spread over more lanes.  Score rows (and bwd rows in the forward sweep) for the
// next DEPTH time steps are kept in flight in registers.
//
// Arithmetic follows the CPU path (reference src/decode_cpu.c:13-147): fp32
// sums of state value and score, max, exp of the fp32 differences, running sum
// in transition order, max + log(sum).  Three variants of that last step exist:
//   precise : exp and log in double, the running sum rounded to fp32 after every
//             term and one rounding of max + log(sum), i.e. the CPU path's own
//             sequence of roundings (fp64 FMA issues at the fp32 rate on gfx950);
//   fast    : v_exp_f32 / v_log_f32, within an ulp or two of the precise result;
//   two-tier: the fast value wherever it provably rounds like the precise one (its
//             distance to a rounding boundary exceeds a bound on its error, or the CPU
//             path's running sum lies between its two boundaries), the logarithm of that
//             sum for the rest.  Same bits as precise.
// State values reach several thousand, where one fp32 ulp is already 5e-4, and
// the posterior is exp(fwd + bwd - const): a last-bit difference in a scan shows
// up as a 5e-4 relative difference of a posterior.  Two-tier is the default for
// that reason; fast exists for measurements.
//
// Kernels: bwd_scan_kernel is the backward sweep; fwd_post_kernel and fwd_post_roles_kernel are the
// forward sweep with the posterior, for a decode that runs it beside the beam search (the third place
// for it, within the search's kernel, is in beam.hip); fwd_scan_kernel and posterior_rows_kernel are the same in two
// steps, for few chunks of 1024 states; scan_post_kernel runs both sweeps of a chunk in one
// workgroup, from both ends of the chunk towards the middle and on to the other end.  Which of them a
// decode uses is decided by its shape (openfish_host.c).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "lse5.h"
#include "kernels.h"
#include "queue.h"

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// fp16 scores per state and time step: the four transitions, or five with an unused blank first.
// The file is compiled once for each layout.
#ifndef OFK_COLS
#define OFK_COLS 4
#endif
constexpr int kCols = OFK_COLS;
constexpr int kLead = kCols - 4;
static_assert(kCols == 4 || kCols == 5, "scores have four or five columns");

template <bool MULTIWAVE>
__device__ __forceinline__ void chunk_sync() {
    if constexpr (MULTIWAVE) {
        // Only LDS traffic has to be ordered across the barrier.  __syncthreads() would also
        // wait for every global load and store in flight, i.e. drain the prefetch ring at
        // every time step.  The wait for this wave's own LDS writes is spelled out: the one that the
        // fence stands for is dropped by the compiler where a loop begins with the barrier and
        // nothing is under way when the loop is entered, although every trip round it ends with a write.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), the other counters unlimited
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    } else {
        // one wavefront per chunk: LDS operations of a wave complete in order, only the
        // compiler has to be kept from moving the reads above the writes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

template <int S, int SPL>
struct Shape {
    static constexpr int kLanes = S / SPL;                            // lanes per chunk
    // Workgroups are four wavefronts wherever a chunk needs fewer: the four waves of a
    // group land on the four SIMDs of a compute unit, while smaller groups were seen
    // to pile up on two of them.  Chunks sharing a group stay independent.
    static constexpr int kChunks = kLanes >= 256 ? 1 : 256 / kLanes;  // chunks per workgroup
    static constexpr int kThreads = kLanes >= 256 ? kLanes : 256;
    static constexpr bool kMultiWave = kLanes > 64;                   // a chunk spans several waves
    static constexpr int kGroup = kLanes >= 64 ? 64 : kLanes;         // chunk lanes inside one wave
    static constexpr int kChunkWaves = kLanes > 64 ? kLanes / 64 : 1;
    static constexpr int kQuarter = S / 4;
};

// The backward sweep keeps its state vector in LDS with the four quarters {c * S/4 ..} spaced
// S/4 + kPad floats apart: a lane stores r + c * S/4, and with S/4 a multiple of the 64 banks
// the lanes of a wave that differ only in c would all hit one bank.  16 floats of padding
// spread them over all banks; reads of the contiguous quad {4r + b} stay 16-byte aligned.
template <int S>
struct BwdVec {
    static constexpr int kQ = S / 4;
    static constexpr int kPad = kQ % 64 == 0 ? 16 : 0;
    static constexpr int kLen = S + 4 * kPad;
    static __device__ __forceinline__ int at(int r, int c) { return r + c * (kQ + kPad); }  // state r + c * S/4, r < S/4
    static __device__ __forceinline__ int of(int s) { return s + kPad * (s / kQ); }         // any state s
};

// The scores one lane needs for one time step, as loaded: fp16 pairs in 32-bit words.
// A state's scores are kCols consecutive fp16 values: the four transitions, after kLead
// values that the decoder never reads (the blank column of five-column scores).  With
// four columns a lane's window is contiguous and is fetched with vector loads; with five
// it is fetched straight from the caller's layout, 32 bits at a time where two wanted values
// are neighbours (from addresses that are only 2-byte aligned, which global loads accept), two
// bytes at a time elsewhere.
__device__ __forceinline__ uint32_t half_at(const _Float16 *p) { return *reinterpret_cast<const uint16_t *>(p); }
__device__ __forceinline__ uint32_t half_pair_at(const _Float16 *p) {
    if constexpr (kCols == 4) {
        return *reinterpret_cast<const uint32_t *>(p);
    } else {  // one 32-bit load from an address that is only 2-byte aligned
        uint32_t w;
        __builtin_memcpy(&w, p, 4);
        return w;
    }
}

// Backward: transition b of own state i is element kCols * b + i of the lane's window
// (word (4b + i) / 2 of w once packed).
template <int SPL>
struct BwdRow;
template <>
struct BwdRow<4> {
    uint32_t w[8];
    __device__ __forceinline__ void load(const _Float16 *p) {
        if constexpr (kCols == 4) {
            const uint4 x = reinterpret_cast<const uint4 *>(p)[0], y = reinterpret_cast<const uint4 *>(p)[1];
            w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
            w[4] = y.x; w[5] = y.y; w[6] = y.z; w[7] = y.w;
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                w[2 * b] = half_pair_at(p + kCols * b);
                w[2 * b + 1] = half_pair_at(p + kCols * b + 2);
            }
        }
    }
    template <int B, int I>
    __device__ __forceinline__ float add(float x) const {
        constexpr int e = 4 * B + I;
        return add_half<e % 2>(w[e / 2], x);
    }
};
template <>
struct BwdRow<2> {
    uint32_t v[4];
    __device__ __forceinline__ void load(const _Float16 *p) {
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = half_pair_at(p + kCols * b);
    }
    template <int B, int I>
    __device__ __forceinline__ float add(float x) const { return add_half<I>(v[B], x); }
};
template <>
struct BwdRow<1> {
    uint32_t v[4];  // one fp16 value each, in the low half
    __device__ __forceinline__ void load(const _Float16 *p) {
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = half_at(p + kCols * b);
    }
    template <int B, int I>
    __device__ __forceinline__ float add(float x) const { return add_half<0>(v[B], x); }
};

// Forward: transition b into own state i is element kCols * i + b of the lane's window
// (word (4i + b) / 2 of w once packed).
template <int SPL>
struct FwdRow {
    uint32_t w[2 * SPL];
    __device__ __forceinline__ void load(const _Float16 *p) {
        if constexpr (kCols == 4 && SPL == 4) {
            const uint4 x = reinterpret_cast<const uint4 *>(p)[0], y = reinterpret_cast<const uint4 *>(p)[1];
            w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
            w[4] = y.x; w[5] = y.y; w[6] = y.z; w[7] = y.w;
        } else if constexpr (kCols == 4 && SPL == 2) {
            const uint4 x = *reinterpret_cast<const uint4 *>(p);
            w[0] = x.x; w[1] = x.y; w[2] = x.z; w[3] = x.w;
        } else if constexpr (kCols == 4) {
            const uint2 x = *reinterpret_cast<const uint2 *>(p);
            w[0] = x.x; w[1] = x.y;
        } else {
#pragma unroll
            for (int i = 0; i < SPL; ++i) {
                w[2 * i] = half_pair_at(p + kCols * i);
                w[2 * i + 1] = half_pair_at(p + kCols * i + 2);
            }
        }
    }
    template <int I, int B>
    __device__ __forceinline__ float add(float x) const {
        constexpr int e = 4 * I + B;
        return add_half<e % 2>(w[e / 2], x);
    }
};

// SPL consecutive floats in global or shared memory
template <int SPL>
struct FloatRun {
    float v[SPL];
    __device__ __forceinline__ void load(const float *p) {
        if constexpr (SPL == 4) {
            const float4 x = *reinterpret_cast<const float4 *>(p);
            v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
        } else if constexpr (SPL == 2) {
            const float2 x = *reinterpret_cast<const float2 *>(p);
            v[0] = x.x; v[1] = x.y;
        } else {
            v[0] = *p;
        }
    }
    __device__ __forceinline__ void store(float *p) const {
        if constexpr (SPL == 4) *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
        else if constexpr (SPL == 2) *reinterpret_cast<float2 *>(p) = make_float2(v[0], v[1]);
        else *p = v[0];
    }
};

template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// `count` steps, DEPTH of them unrolled per trip: step(k, j, checked) with k = j % DEPTH a
// compile-time index; in unchecked trips j + DEPTH + SLACK < count holds for every step, i.e.
// every prefetch DEPTH steps ahead is in range (of a tensor with SLACK rows fewer than steps).
template <int DEPTH, int SLACK = 0, typename Step>
__device__ __forceinline__ void pipelined(int count, Step &&step) {
    int j0 = 0;
    for (; j0 + 2 * DEPTH + SLACK <= count; j0 += DEPTH)
        static_for<DEPTH>([&](auto k) { step(k, j0 + (int)k, std::false_type{}); });
    for (; j0 < count; j0 += DEPTH)
        static_for<DEPTH>([&](auto k) {
            if (j0 + (int)k < count) step(k, j0 + (int)k, std::true_type{});
        });
}

// The same in two kinds of trips: while early() holds, asked once a trip, steps get a true_type as their fourth argument.
template <int DEPTH, typename Early, typename Step>
__device__ __forceinline__ void pipelined_from_early(int count, Early &&early, Step &&step) {
    int j0 = 0;
    for (; j0 + 2 * DEPTH <= count && early(); j0 += DEPTH)
        static_for<DEPTH>([&](auto k) { step(k, j0 + (int)k, std::false_type{}, std::true_type{}); });
    for (; j0 + 2 * DEPTH <= count; j0 += DEPTH)
        static_for<DEPTH>([&](auto k) { step(k, j0 + (int)k, std::false_type{}, std::false_type{}); });
    for (; j0 < count && early(); j0 += DEPTH)
        static_for<DEPTH>([&](auto k) {
            if (j0 + (int)k < count) step(k, j0 + (int)k, std::true_type{}, std::true_type{});
        });
    for (; j0 < count; j0 += DEPTH)
        static_for<DEPTH>([&](auto k) {
            if (j0 + (int)k < count) step(k, j0 + (int)k, std::true_type{}, std::false_type{});
        });
}

// the five terms of one state of a lane, and of every one; the row's registers are free for the next load afterwards
template <int I, int SPL>
__device__ __forceinline__ void bwd_terms_of(float (&v)[5], const float (&a)[SPL], const float4 &nx, const BwdRow<SPL> &row, float stay) {
    v[0] = a[I] + stay;
    v[1] = row.template add<0, I>(nx.x);
    v[2] = row.template add<1, I>(nx.y);
    v[3] = row.template add<2, I>(nx.z);
    v[4] = row.template add<3, I>(nx.w);
}
template <int I, int SPL>
__device__ __forceinline__ void fwd_terms_of(float (&v)[5], const float (&f)[SPL], float p0, float p1, float p2, float p3,
                                             const FwdRow<SPL> &row, float stay) {
    v[0] = f[I] + stay;
    v[1] = row.template add<I, 0>(p0);
    v[2] = row.template add<I, 1>(p1);
    v[3] = row.template add<I, 2>(p2);
    v[4] = row.template add<I, 3>(p3);
}
template <int SPL>
__device__ __forceinline__ void bwd_terms(float (&v)[SPL][5], const float (&a)[SPL], const float4 &nx, const BwdRow<SPL> &row, float stay) {
    static_for<SPL>([&](auto i) { bwd_terms_of<i, SPL>(v[i], a, nx, row, stay); });
}
template <int SPL>
__device__ __forceinline__ void fwd_terms(float (&v)[SPL][5], const float (&f)[SPL], float p0, float p1, float p2, float p3,
                                          const FwdRow<SPL> &row, float stay) {
    static_for<SPL>([&](auto i) { fwd_terms_of<i, SPL>(v[i], f, p0, p1, p2, p3, row, stay); });
}

// the update of a step of the separate sweeps; EARLY: in the double arithmetic at once
template <int SPL, int MODE, bool EARLY, typename Publish, typename Beside>
__device__ __forceinline__ void update(float (&out)[SPL], const float (&v)[SPL][5], const LogArgs &logtab, Publish &&publish, Beside &&beside) {
    if constexpr (EARLY) lse5_all_double<SPL>(out, v, logtab, publish, beside);
    else lse5_all<SPL, MODE>(out, v, logtab, publish, beside);
}

// A step of the kernel that holds both sweeps and is capped at 128 registers.  Of four states to a lane the terms are
// not kept for a common second tier (as in the separate sweeps, which may use 256 registers): that spilled inside the
// loops.  One state after another needs no scratch with 256
// states, and with 1024 only between the phases.  Scans of 2048 chunks of 256 states, T = 1666: 6.87 ms all four
// together, 5.7 now (five columns 7.87, 6.05); 512 chunks of 1024 states 6.14, 5.45; with the batch spread over twice the
// lanes 5.65, 6.0 and 5.75.
// `publish` writes the new values to LDS (lse5_all says when; with four states to a lane once all of them are there).
template <int SPL, int MODE, typename Publish>
__device__ __forceinline__ void bwd_update(float (&a)[SPL], const float4 &nx, const BwdRow<SPL> &row, float stay, const LogArgs &logtab,
                                           Publish &&publish) {
    if constexpr (SPL < 4) {
        float v[SPL][5];
        bwd_terms(v, a, nx, row, stay);
        lse5_all<SPL, MODE>(a, v, logtab, publish, [](bool) {});
    } else {
        static_for<SPL>([&](auto i) {
            float v[1][5], out[1];
            bwd_terms_of<i, SPL>(v[0], a, nx, row, stay);
            lse5_all<1, MODE, true>(out, v, logtab, [] {}, [](bool) {});
            a[i] = out[0];
        });
        publish();
    }
}
template <int SPL, int MODE, typename Publish>
__device__ __forceinline__ void fwd_update(float (&f)[SPL], float p0, float p1, float p2, float p3, const FwdRow<SPL> &row, float stay,
                                           const LogArgs &logtab, Publish &&publish) {
    if constexpr (SPL < 4) {
        float v[SPL][5];
        fwd_terms(v, f, p0, p1, p2, p3, row, stay);
        lse5_all<SPL, MODE>(f, v, logtab, publish, [](bool) {});
    } else {
        static_for<SPL>([&](auto i) {
            float v[1][5], out[1];
            fwd_terms_of<i, SPL>(v[0], f, p0, p1, p2, p3, row, stay);
            lse5_all<1, MODE, true>(out, v, logtab, [] {}, [](bool) {});
            f[i] = out[0];
        });
        publish();
    }
}

// ---------------------------------------------------------------------------
// backward: bwd[n][t][s] for t = T..0
// ---------------------------------------------------------------------------
template <int S, int SPL, int DEPTH, int MODE, bool EARLY>  // EARLY: the first steps in double arithmetic, while values are small
__global__ __launch_bounds__((Shape<S, SPL>::kThreads)) void bwd_scan_kernel(
    const _Float16 *__restrict__ scores, float *__restrict__ bwd, int T, int N, float stay, uint32_t double_below, LogSeries series) {
    using Sh = Shape<S, SPL>;
    constexpr int L = Sh::kLanes;
    constexpr int Q = Sh::kQuarter;
    constexpr int H = 4 / SPL;  // lanes sharing one quad
    using Vec = BwdVec<S>;
    __shared__ __attribute__((aligned(16))) float vec[Sh::kChunks][2][Vec::kLen];
    __shared__ __attribute__((aligned(16))) ofa::LogCell logcells[MODE == OFK_SCAN_PRECISE ? 32 : 1], centred[ofa::kLogCentredCells];
    __shared__ __attribute__((aligned(16))) float tier_lanes[MODE == OFK_SCAN_TWO_TIER ? Sh::kThreads : 64];
    const int tid = threadIdx.x;
    const LogArgs logtab{MODE == OFK_SCAN_PRECISE ? logcells : nullptr, centred, series.c, series.e,
                         tier_lanes + (MODE == OFK_SCAN_TWO_TIER ? (tid & ~63) : 0)};

    fill_log_tables<MODE, Sh::kThreads>(logcells, centred);
    const int g = tid / L, l = tid % L;
    const int r = l / H, c0 = (l % H) * SPL;  // own states: r + (c0 + i) * Q
    int n = blockIdx.x * Sh::kChunks + g;
    if (n >= N) n = N - 1;

    // Rows are addressed by a base that is the same for the whole workgroup (scalar registers, stepped by
    // scalar additions) plus a 32-bit offset of the lane.  Lanes past the batch repeat its last chunk, stores included.
    const ptrdiff_t row_stride = (ptrdiff_t)N * kCols * S;  // fp16 elements between time steps
    const int first_chunk = blockIdx.x * Sh::kChunks;
    const unsigned g_eff = (unsigned)(n - first_chunk);
    const unsigned sc_lane = g_eff * kCols * S + 4 * kCols * r + kLead + c0;
    const unsigned st_lane = g_eff * (unsigned)(T + 1) * S + r + c0 * Q;
    const _Float16 *pre = scores + (size_t)first_chunk * kCols * S + (ptrdiff_t)(T - 1) * row_stride;  // next row to fetch
    float *orow = bwd + ((size_t)first_chunk * (size_t)(T + 1) + T) * S;                              // row stored last

    float a[SPL];
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        a[i] = 0.f;
        orow[st_lane + i * Q] = 0.f;
        vec[g][0][Vec::at(r, c0 + i)] = 0.f;
    }

    int buf = 0;
    __syncthreads();  // the log table is shared by the whole group

    // The chain of a step: LDS read, terms, estimate, LDS write (and the barrier).  The verdict on the estimates is formed
    // while the write is under way, the row's store and the loads ahead are issued while the verdict's mask is (lse5_all);
    // where a chunk is one wave, the next step's read is asked for as soon as the values are written.
    auto neighbours = [&](int b) { return *reinterpret_cast<const float4 *>(&vec[g][b][Vec::of(4 * r)]); };
    float4 nx;
    if constexpr (!Sh::kMultiWave) {
        chunk_sync<false>();
        nx = neighbours(0);
    }
    // one step; `load_ahead` fetches into the row's registers
    auto step = [&](BwdRow<SPL> &next, auto early, auto &&load_ahead) {
        constexpr bool kEarly = decltype(early)::value, kBehindRead = SPL == 1 && !kEarly;
        if constexpr (Sh::kMultiWave) {
            chunk_sync<true>();
            nx = neighbours(buf);
        }
        const BwdRow<SPL> row = next;
        if constexpr (kBehindRead) {
            __builtin_amdgcn_sched_barrier(0);
            load_ahead();
            __builtin_amdgcn_sched_barrier(0);
        }
        float v[SPL][5];
        bwd_terms(v, a, nx, row, stay);
        buf ^= 1;
        orow -= S;
        update<SPL, MODE, kEarly>(a, v, logtab, [&] {
#pragma unroll
            for (int i = 0; i < SPL; ++i) vec[g][buf][Vec::at(r, c0 + i)] = a[i];
            if constexpr (!Sh::kMultiWave) {
                chunk_sync<false>();
                nx = neighbours(buf);
            }
        }, [&](bool first) {
#pragma unroll
            for (int i = 0; i < SPL; ++i) orow[st_lane + i * Q] = a[i];
            if (!kBehindRead && first) load_ahead();
        });
    };
    // The first rows are fetched without a condition (of a chunk shorter than the ring the oldest row again):
    // were they not, the compiler, which counts loads in flight, would have to assume that a row's load may
    // be the latest one and let every trip round the loop below wait for all of them.
    auto first_rows = [&](auto &ring, auto depth, int left) {
        static_for<decltype(depth)::value>([&](auto k) {
            ring[k].load(pre + sc_lane);
            pre -= (int)k < left - 1 ? row_stride : 0;
        });
    };
    int done = 0;
    if constexpr (EARLY) {
        static_assert(MODE == OFK_SCAN_TWO_TIER && SPL == 1);
        // The early steps, in double arithmetic (double_below in the launcher).  They have a ring of their own and fill the one below anew: with one
        // ring for both the compiler kept every row twice, 164 registers instead of 120.
        constexpr int kRows = 8;
        BwdRow<SPL> ring[kRows];
        first_rows(ring, std::integral_constant<int, kRows>{}, T);
        auto trip = [&](auto checked) {
            static_for<kRows>([&](auto k) {
                const int j = done + (int)k;
                if (checked && j >= T) return;
                step(ring[k], std::true_type{}, [&] {
                    if (!checked || j + kRows < T) {
                        ring[k].load(pre + sc_lane);
                        pre -= row_stride;
                    }
                });
            });
            done += kRows;
        };
        while (done + 2 * kRows <= T && values_below(a[0], double_below)) trip(std::false_type{});
        while (done < T && values_below(a[0], double_below)) trip(std::true_type{});
        if (done >= T) return;
        pre = scores + (size_t)first_chunk * kCols * S + (ptrdiff_t)(T - 1 - done) * row_stride;
    }
    BwdRow<SPL> ring[DEPTH];
    first_rows(ring, std::integral_constant<int, DEPTH>{}, T - done);
    pipelined<DEPTH>(T - done, [&](auto k, int j, auto checked) {
        step(ring[k], std::false_type{}, [&] {
            if (!checked || done + j + DEPTH < T) {
                ring[k].load(pre + sc_lane);
                pre -= row_stride;
            }
        });
    });
}

// ---------------------------------------------------------------------------
// forward + posterior: post[n][t][s] = softmax_s(fwd[t][s] + bwd[n][t][s]), t = 0..T
// ---------------------------------------------------------------------------
template <int S, int SPL, int DEPTH, int MODE, bool EARLY>
__global__ __launch_bounds__((Shape<S, SPL>::kThreads)) void fwd_post_kernel(
    const _Float16 *__restrict__ scores, const float *__restrict__ bwd, float *__restrict__ post, int T,
    int N, float stay, uint32_t double_below, LogSeries series) {
    using Sh = Shape<S, SPL>;
    constexpr int L = Sh::kLanes;
    constexpr int Q = Sh::kQuarter;
    __shared__ __attribute__((aligned(16))) float vec[Sh::kChunks][2][S];
    __shared__ float part[2][Sh::kChunks][Sh::kChunkWaves];
    __shared__ __attribute__((aligned(16))) ofa::LogCell logcells[MODE == OFK_SCAN_PRECISE ? 32 : 1], centred[ofa::kLogCentredCells];
    __shared__ __attribute__((aligned(16))) float tier_lanes[MODE == OFK_SCAN_TWO_TIER ? Sh::kThreads : 64];
    const int tid = threadIdx.x;
    // this sweep runs beside the beam search, whose waves run at priority 3: trips through the second tier
    // at 1 leave that search alone (2048 chunks of 64 states: search 2.50 ms against 2.59 with 3 here)
    const LogArgs logtab{MODE == OFK_SCAN_PRECISE ? logcells : nullptr, centred, series.c, series.e,
                         tier_lanes + (MODE == OFK_SCAN_TWO_TIER ? (tid & ~63) : 0), 1};

    fill_log_tables<MODE, Sh::kThreads>(logcells, centred);
    const int g = tid / L, l = tid % L;
    const int s0 = SPL * l, q = s0 >> 2;  // own states s0 .. s0+SPL-1, all in quad q
    const int wave = l / 64;  // wave within the chunk
    int n = blockIdx.x * Sh::kChunks + g;
    if (n >= N) n = N - 1;

    // addresses as in bwd_scan_kernel; the first rows are fetched without a condition for the reason given there
    const ptrdiff_t row_stride = (ptrdiff_t)N * kCols * S;
    const int first_chunk = blockIdx.x * Sh::kChunks;
    const unsigned g_eff = (unsigned)(n - first_chunk);
    const unsigned sc_lane = g_eff * kCols * S + kCols * s0 + kLead;
    const unsigned st_lane = g_eff * (unsigned)(T + 1) * S + s0;
    const _Float16 *pre = scores + (size_t)first_chunk * kCols * S;
    const size_t blk_off = (size_t)first_chunk * (size_t)(T + 1) * S;
    const float *bpre = bwd + blk_off;
    float *prow = post + blk_off;

    FwdRow<SPL> ring[DEPTH];
    FloatRun<SPL> bring[DEPTH];
    static_for<DEPTH>([&](auto k) {
        ring[k].load(pre + sc_lane);
        bring[k].load(bpre + st_lane);
        pre += (int)k < T - 1 ? row_stride : 0;
        bpre += (int)k < T ? S : 0;
    });

    // Shift of the softmax exponent.  sum_s exp(fwd+bwd) is the same partition function at
    // every time step, and at t = 0 it lies within log(S) of max_s bwd[0][s]; that maximum,
    // lowered by 10 so that tiny posteriors stay normal numbers until the final product,
    // replaces the per-step maximum (the quotient does not depend on the shift).
    float shift;
    {
        float m = bring[0].v[0];
#pragma unroll
        for (int i = 1; i < SPL; ++i) m = fmaxf(m, bring[0].v[i]);
        m = group_max<Sh::kGroup>(m);
        if constexpr (Sh::kMultiWave) {
            if ((tid & 63) == 0) part[0][g][wave] = m;
            chunk_sync<true>();
            m = part[0][g][0];
#pragma unroll
            for (int w = 1; w < Sh::kChunkWaves; ++w) m = fmaxf(m, part[0][g][w]);
            chunk_sync<true>();
        }
        shift = m - 10.0f;
    }

    FloatRun<SPL> fv;  // the state vector
    float (&f)[SPL] = fv.v;
#pragma unroll
    for (int i = 0; i < SPL; ++i) f[i] = 0.f;
    int buf = 0;
    fv.store(&vec[g][0][s0]);
    __syncthreads();  // the log table is shared by the whole group

    // row j: its posterior; the state vector, written by the update before, becomes visible to the other lanes
    auto row = [&](const FloatRun<SPL> &bw) {
        FloatRun<SPL> e;
        float total = 0.f;
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            e.v[i] = __builtin_amdgcn_exp2f(((f[i] + bw.v[i]) - shift) * kLog2e);
            total += e.v[i];
        }
        total = group_sum<Sh::kGroup>(total);
        if constexpr (Sh::kMultiWave) {
            if ((tid & 63) == 0) part[buf][g][wave] = total;
        }
        chunk_sync<Sh::kMultiWave>();
        if constexpr (Sh::kMultiWave) {
            total = part[buf][g][0];
#pragma unroll
            for (int w = 1; w < Sh::kChunkWaves; ++w) total += part[buf][g][w];
        }
        const float inv = __builtin_amdgcn_rcpf(total);
#pragma unroll
        for (int i = 0; i < SPL; ++i) e.v[i] *= inv;
        e.store(prow + st_lane);
        prow += S;
    };
    auto step = [&](auto k, int j, auto checked, auto early) {
        row(bring[k]);
        const float p0 = vec[g][buf][q], p1 = vec[g][buf][q + Q];
        const float p2 = vec[g][buf][q + 2 * Q], p3 = vec[g][buf][q + 3 * Q];
        float v[SPL][5];
        fwd_terms(v, f, p0, p1, p2, p3, ring[k], stay);
        if (!checked || j + DEPTH < T) {
            ring[k].load(pre + sc_lane);
            pre += row_stride;
        }
        if (!checked || j + DEPTH <= T) {
            bring[k].load(bpre + st_lane);
            bpre += S;
        }
        buf ^= 1;
        update<SPL, MODE, decltype(early)::value>(f, v, logtab, [&] { fv.store(&vec[g][buf][s0]); }, [](bool) {});
    };
    if constexpr (EARLY)
        pipelined_from_early<DEPTH>(T, [&] { return values_below(f[0], double_below); }, step);
    else
        pipelined<DEPTH>(T, [&](auto k, int j, auto checked) { step(k, j, checked, std::false_type{}); });
    static_for<DEPTH>([&](auto k) {
        if (T % DEPTH == (int)k) row(bring[k]);
    });
}

// ---------------------------------------------------------------------------
// forward + posterior with the two jobs on different waves.
//
// fwd_post_kernel's lanes take the posterior of a row between two steps of the recursion: an
// exponential, a sum over the wave, a partial sum through LDS, a reciprocal and a store join the
// chain of dependent operations of every time step, which is what this sweep's duration is made
// of.  Here a chunk has twice the
// lanes: one half runs the recursion alone, the other half reads every row the first half
// publishes in LDS for its own exchange anyway, and forms that row's posterior one step behind.
// Every wave takes one block barrier per time step (plus one at the end and two for the shift).
// Same arithmetic, same results.  (Letting the second half also sum the finished row over every
// state's neighbours for the quality stage was measured and dropped: the extra LDS traffic slowed
// the recursion by more, 0.18 ms, than the sums save that stage, 0.09 ms.)
//
// Only two rows are in flight per stream: the kernel shares the memory with the beam search, whose rows
// lie the same N * C * 2 bytes apart, and both together run at the rate a copy reaches.  More rows in
// flight spread the accesses over more DRAM pages at once and slow both down (512 chunks of 256 states, this
// kernel / the search beside it: eight rows 1.52 / 2.09 ms, four 1.23 / 1.20, two 1.15 / 1.10).
// ---------------------------------------------------------------------------
constexpr int kRolesDepth = 2;

template <int S, int SPL, int DEPTH>
__global__ __launch_bounds__((2 * (S / SPL))) void fwd_post_roles_kernel(
    const _Float16 *__restrict__ scores, const float *__restrict__ bwd, float *__restrict__ post, int T,
    int N, float stay, uint32_t double_below, LogSeries series) {
    constexpr int L = S / SPL;  // lanes of either job
    constexpr int Q = S / 4;
    constexpr int RW = L / 64;  // waves of either job
    static_assert(L % 64 == 0 && RW > 1, "either job owns several whole waves");
    __shared__ __attribute__((aligned(16))) float vec[2][S];
    __shared__ float part[2][RW];
    __shared__ __attribute__((aligned(16))) ofa::LogCell centred[ofa::kLogCentredCells];
    __shared__ __attribute__((aligned(16))) float tier_lanes[L];
    const int tid = threadIdx.x;
    const int posterior = __builtin_amdgcn_readfirstlane(tid / L);
    const int l = tid % L, lane = tid & 63, wave = l / 64;
    // This kernel runs beside the beam search, whose waves run at priority 3, which trips through the second tier leave
    // alone.  The recursion, which is the chain, goes before the posterior (512 chunks of 256 states: 1.02 ms against 1.14
    // with both at 0, search beside it 1.09 against 1.11).
    const LogArgs logtab{nullptr, centred, series.c, series.e, tier_lanes + (l & ~63), 2, 1};
    if (!posterior) __builtin_amdgcn_s_setprio(1);
    fill_log_tables<OFK_SCAN_TWO_TIER, 2 * (S / SPL)>(nullptr, centred);
    const int s0 = SPL * l, q = s0 >> 2;  // own states s0 .. s0+SPL-1, all in quad q
    const int n = blockIdx.x;            // one chunk per workgroup
    const ptrdiff_t row_stride = (ptrdiff_t)N * kCols * S;
    auto barrier = [] { chunk_sync<true>(); };

    if (!posterior) {
        const _Float16 *pre = scores + (size_t)n * kCols * S;
        const unsigned sc_lane = kCols * s0 + kLead;
        FwdRow<SPL> ring[DEPTH];
        static_for<DEPTH>([&](auto k) {  // without a condition, as in bwd_scan_kernel
            ring[k].load(pre + sc_lane);
            pre += (int)k < T - 1 ? row_stride : 0;
        });
        FloatRun<SPL> fv;
        float (&f)[SPL] = fv.v;
#pragma unroll
        for (int i = 0; i < SPL; ++i) f[i] = 0.f;
        int buf = 0;
        fv.store(&vec[0][s0]);  // row 0
        barrier();  // the other half exchanges the maxima behind the shift
        barrier();
        __syncthreads();  // the log table
        auto step = [&](auto k, int j, auto checked, auto early) {
            barrier();
            const float p0 = vec[buf][q], p1 = vec[buf][q + Q];
            const float p2 = vec[buf][q + 2 * Q], p3 = vec[buf][q + 3 * Q];
            float v[SPL][5];
            fwd_terms(v, f, p0, p1, p2, p3, ring[k], stay);
            buf ^= 1;
            update<SPL, OFK_SCAN_TWO_TIER, decltype(early)::value>(f, v, logtab, [&] { fv.store(&vec[buf][s0]); }, [&](bool first) {  // row j + 1
                if (first && (!checked || j + DEPTH < T)) {
                    ring[k].load(pre + sc_lane);
                    pre += row_stride;
                }
            });
        };
        if constexpr (SPL == 1)
            pipelined_from_early<DEPTH>(T, [&] { return values_below(f[0], double_below); }, step);
        else
            pipelined<DEPTH>(T, [&](auto k, int j, auto checked) { step(k, j, checked, std::false_type{}); });
        barrier();
        barrier();  // the other half finishes row T
    } else {
        const float *bpre = bwd + (size_t)n * (size_t)(T + 1) * S;
        float *prow = post + (size_t)n * (size_t)(T + 1) * S;  // row finished next
        FloatRun<SPL> bring[DEPTH];
        static_for<DEPTH>([&](auto k) {
            bring[k].load(bpre + s0);
            bpre += (int)k < T ? S : 0;
        });
        // Shift of the softmax exponent, as in fwd_post_kernel: max_s bwd[0][s] - 10.
        float shift;
        {
            float m = bring[0].v[0];
#pragma unroll
            for (int i = 1; i < SPL; ++i) m = fmaxf(m, bring[0].v[i]);
            m = group_max<64>(m);
            if (lane == 0) part[0][wave] = m;
            barrier();
            m = part[0][0];
#pragma unroll
            for (int w = 1; w < RW; ++w) m = fmaxf(m, part[0][w]);
            barrier();
            shift = m - 10.0f;
        }
        __syncthreads();
        FloatRun<SPL> e;  // terms of the row before, waiting for the sum over the waves
        int buf = 0;
        auto finish_row = [&] {  // the row before the one in vec[buf]
            float total = part[buf ^ 1][0];
#pragma unroll
            for (int w = 1; w < RW; ++w) total += part[buf ^ 1][w];
            const float inv = __builtin_amdgcn_rcpf(total);
#pragma unroll
            for (int i = 0; i < SPL; ++i) e.v[i] *= inv;
            e.store(prow + s0);
            prow += S;
        };
        auto terms = [&](const FloatRun<SPL> &bw) {
            FloatRun<SPL> fv;
            fv.load(&vec[buf][s0]);
            float total = 0.f;
#pragma unroll
            for (int i = 0; i < SPL; ++i) {
                e.v[i] = __builtin_amdgcn_exp2f(((fv.v[i] + bw.v[i]) - shift) * kLog2e);
                total += e.v[i];
            }
            total = group_sum<64>(total);
            if (lane == 0) part[buf][wave] = total;
            buf ^= 1;
        };
        pipelined<DEPTH>(T + 1, [&](auto k, int j, auto checked) {
            barrier();  // row j is in vec[buf], the partial sums of row j - 1 in part[buf ^ 1]
            if ((int)k != 0 || j > 0) finish_row();
            terms(bring[k]);
            if (!checked || j + DEPTH <= T) {
                bring[k].load(bpre + s0);
                bpre += S;
            }
        });
        barrier();
        finish_row();
    }
}

// ---------------------------------------------------------------------------
// The forward recursion by itself, rows left in post[t], and the posterior of rows whose recursion is done: for
// batches of 1024 states that leave compute units idle.  A chunk's sweep is bound by what its one unit can issue, and nothing
// in the recursion waits for the backward one: on units of their own the two run at the same time, and what is left to do
// beside the search is a pass over rows that depends on no other row.  37 chunks, T = 833, ms: backward 0.67, then forward
// sweep with posterior 0.74 beside a search of 0.49 | both sweeps 0.68, then posteriors 0.14 beside a search of 0.49.
// ---------------------------------------------------------------------------
template <int S, int DEPTH>
__global__ __launch_bounds__(S) void fwd_scan_kernel(const _Float16 *__restrict__ scores, float *__restrict__ fwd, int T, int N,
                                                     float stay, uint32_t double_below, LogSeries series) {
    constexpr int Q = S / 4;
    static_assert(S > 64, "a state to a lane, and several waves");
    __shared__ __attribute__((aligned(16))) float vec[2][S];
    __shared__ __attribute__((aligned(16))) ofa::LogCell centred[ofa::kLogCentredCells];
    __shared__ __attribute__((aligned(16))) float tier_lanes[S];
    const int s = threadIdx.x, q = s >> 2;
    const LogArgs logtab{nullptr, centred, series.c, series.e, tier_lanes + (s & ~63)};
    fill_log_tables<OFK_SCAN_TWO_TIER, S>(nullptr, centred);
    const ptrdiff_t row_stride = (ptrdiff_t)N * kCols * S;
    const _Float16 *pre = scores + (size_t)blockIdx.x * kCols * S;
    float *frow = fwd + (size_t)blockIdx.x * (size_t)(T + 1) * S;
    const unsigned sc_lane = kCols * s + kLead;
    FwdRow<1> ring[DEPTH];
    static_for<DEPTH>([&](auto k) {  // without a condition, as in bwd_scan_kernel
        ring[k].load(pre + sc_lane);
        pre += (int)k < T - 1 ? row_stride : 0;
    });
    float f[1] = {0.f};
    int buf = 0;
    vec[0][s] = 0.f;
    frow[s] = 0.f;
    __syncthreads();  // the log table
    pipelined_from_early<DEPTH>(T, [&] { return values_below(f[0], double_below); }, [&](auto k, int j, auto checked, auto early) {
        chunk_sync<true>();
        const float p0 = vec[buf][q], p1 = vec[buf][q + Q], p2 = vec[buf][q + 2 * Q], p3 = vec[buf][q + 3 * Q];
        const FwdRow<1> row = ring[k];
        __builtin_amdgcn_sched_barrier(0);
        if (!checked || j + DEPTH < T) {
            ring[k].load(pre + sc_lane);
            pre += row_stride;
        }
        __builtin_amdgcn_sched_barrier(0);
        float v[1][5];
        fwd_terms(v, f, p0, p1, p2, p3, row, stay);
        buf ^= 1;
        frow += S;
        update<1, OFK_SCAN_TWO_TIER, decltype(early)::value>(f, v, logtab, [&] { vec[buf][s] = f[0]; }, [&](bool) { frow[s] = f[0]; });
    });
}

// post[n][t] holds fwd[t] and gets softmax(fwd[t] + bwd[n][t]): a wave takes a row, `parts` workgroups a chunk.  Sums in the order
// of fwd_post_roles_kernel with two states to a lane (pieces of 128 states, their totals one after another): the same bits.
template <int S>
__global__ __launch_bounds__(256) void posterior_rows_kernel(const float *__restrict__ bwd, float *__restrict__ post, int T, int parts) {
    constexpr int P = S / 128;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int n = blockIdx.x / parts, part = blockIdx.x % parts;
    const size_t first = (size_t)n * (size_t)(T + 1) * S + 2 * lane;
    const float *b0 = bwd + first;
    float *p0 = post + first;
    auto load = [&](const float *row, float2 (&x)[P]) {
#pragma unroll
        for (int k = 0; k < P; ++k) x[k] = *reinterpret_cast<const float2 *>(row + 128 * k);
    };
    float2 b[P], f[P], b_next[P], f_next[P];
    load(b0, b);  // the shift of the exponent, as in fwd_post_kernel: max_s bwd[0][s] - 10
    float top = fmaxf(b[0].x, b[0].y);
#pragma unroll
    for (int k = 1; k < P; ++k) top = fmaxf(top, fmaxf(b[k].x, b[k].y));
    const float shift = group_max<64>(top) - 10.0f;
    const int step = 4 * parts;
    int t = 4 * part + wave;
    if (t > T) return;
    load(b0 + (size_t)t * S, b_next);
    load(p0 + (size_t)t * S, f_next);
    for (; t <= T; t += step) {
#pragma unroll
        for (int k = 0; k < P; ++k) {
            b[k] = b_next[k];
            f[k] = f_next[k];
        }
        if (t + step <= T) {
            load(b0 + (size_t)(t + step) * S, b_next);
            load(p0 + (size_t)(t + step) * S, f_next);
        }
        float total = 0.f;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            f[k].x = __builtin_amdgcn_exp2f(((f[k].x + b[k].x) - shift) * kLog2e);
            f[k].y = __builtin_amdgcn_exp2f(((f[k].y + b[k].y) - shift) * kLog2e);
            const float piece = group_sum<64>(f[k].x + f[k].y);
            total = k == 0 ? piece : total + piece;
        }
        const float inv = __builtin_amdgcn_rcpf(total);
#pragma unroll
        for (int k = 0; k < P; ++k)
            *reinterpret_cast<float2 *>(p0 + (size_t)t * S + 128 * k) = make_float2(f[k].x * inv, f[k].y * inv);
    }
}

// ---------------------------------------------------------------------------
// Both sweeps in one kernel, meeting in the middle.
//
// The forward recursion does not depend on the backward one; only the posterior needs
// both.  A chunk is served by two groups of lanes of one workgroup, one per direction,
// which doubles the wavefronts in flight (the separate sweeps leave the device at one or
// two waves per SIMD at 512 chunks of 256 states, where every wave issues at half the rate
// the SIMD could take).
//   phase 1: the backward lanes run t = T-1 .. H and write bwd[t]; the forward lanes run
//            t = 0 .. H-1 and park fwd[t] in post[t];
//   middle : the partition function max_s(fwd[H][s] + bwd[H][s]) fixes the exponent shift
//            of the softmax (it is the same at every time step);
//   phase 2: the forward lanes run t = H .. T reading bwd[t] (written in phase 1), the
//            backward lanes run t = H-1 .. 0 reading the parked fwd[t]; both write the
//            posterior, the backward lanes over the parked values.
// HBM traffic: every score twice, bwd written once, half of it read once, post written once
// and half of it written and read once more as fwd: (T+1) S 4 bytes above the two separate
// sweeps.  One block barrier per time step serves both directions.
// ---------------------------------------------------------------------------
template <int S, int SPL>
struct FusedShape {
    static constexpr int kLanes = S / SPL;                 // lanes per direction and chunk
    static constexpr int kRoleWaves = kLanes / 64;         // whole waves: a wave has one direction
    static constexpr int kChunkThreads = 2 * kLanes;
    static constexpr int kChunks = kChunkThreads >= 512 ? 1 : 512 / kChunkThreads;
    static constexpr int kThreads = kChunks * kChunkThreads;
    static constexpr int kQuarter = S / 4;
    static_assert(kLanes % 64 == 0, "a direction owns whole wavefronts");
};

__device__ __forceinline__ void block_barrier_lds() { chunk_sync<true>(); }

template <int S, int SPL, int DEPTH, int MODE>
__global__ __launch_bounds__((FusedShape<S, SPL>::kThreads), 4) void scan_post_kernel(
    const _Float16 *__restrict__ scores, float *__restrict__ bwd, float *__restrict__ post, int T, int N, float stay,
    LogSeries series) {
    using Sh = FusedShape<S, SPL>;
    constexpr int L = Sh::kLanes;
    constexpr int Q = Sh::kQuarter;
    constexpr int RW = Sh::kRoleWaves;
    constexpr int H4 = 4 / SPL;  // backward lanes sharing one quad
    constexpr int kWarmup = 32;  // time steps of either sweep evaluated in double before the two tiers take over
    // Per time step the lanes of one direction exchange their state vector (and the partial sums of
    // the posterior's denominator) through LDS.  With several waves per direction that takes a
    // workgroup barrier, which both directions (and every chunk of the group) then share; when a
    // direction is a single wave (64 states), a time step only needs the wave's own LDS operations
    // kept in order, and the waves of a group run their steps without waiting for one another.  The
    // two directions of a chunk meet only in the middle, at block barriers that every wave reaches.
    auto step_sync = [] { chunk_sync<(RW > 1)>(); };
    using VecB = BwdVec<S>;
    __shared__ __attribute__((aligned(16))) float vecB[Sh::kChunks][2][VecB::kLen];
    __shared__ __attribute__((aligned(16))) float vecF[Sh::kChunks][2][S];
    __shared__ float part[Sh::kChunks][2][2][RW];  // [chunk][direction][parity][wave]
    __shared__ float shift_of[Sh::kChunks];
    __shared__ __attribute__((aligned(16))) ofa::LogCell logcells[32], centred[ofa::kLogCentredCells];
    __shared__ __attribute__((aligned(16))) float tier_lanes[MODE == OFK_SCAN_TWO_TIER ? Sh::kThreads : 64];
    const int tid = threadIdx.x;
    const LogArgs logtab{logcells, centred, series.c, series.e, tier_lanes + (MODE == OFK_SCAN_TWO_TIER ? (tid & ~63) : 0)};

    fill_log_tables<MODE, Sh::kThreads, MODE == OFK_SCAN_TWO_TIER>(logcells, centred);  // the first steps of either sweep take the always-double arithmetic
    const int g = tid / Sh::kChunkThreads, u = tid % Sh::kChunkThreads;
    const int forward = __builtin_amdgcn_readfirstlane(u / L);
    const int l = u % L, wave = l / 64;
    int n = blockIdx.x * Sh::kChunks + g;
    const bool live = Sh::kChunks == 1 || n < N;
    if (!live) n = N - 1;

    const int H = T / 2;  // forward: rows 0..H-1 in phase 1, H..T in phase 2
    // Addresses are a base that is the same for the whole workgroup (kept in scalar registers and
    // stepped from row to row by scalar additions) plus a 32-bit offset of the lane that never changes.
    const ptrdiff_t row_stride = (ptrdiff_t)N * kCols * S;  // fp16 elements between time steps
    const int first_chunk = blockIdx.x * Sh::kChunks;
    const unsigned g_eff = (unsigned)(n - first_chunk);  // chunk within the group (dead lanes repeat the last chunk)
    const _Float16 *const sc_blk = scores + (size_t)first_chunk * kCols * S;
    const size_t blk_off = (size_t)first_chunk * (size_t)(T + 1) * S;
    float *const bwd_blk = bwd + blk_off;
    float *const post_blk = post + blk_off;
    const unsigned chunk_rows = g_eff * (unsigned)(T + 1) * S;

    if (!forward) {
        // ------------------------------ backward lanes ------------------------------
        const int r = l / H4, c0 = (l % H4) * SPL;  // own states: r + (c0 + i) * Q
        const unsigned sc_lane = g_eff * kCols * S + 4 * kCols * r + kLead + c0;
        const unsigned st_lane = chunk_rows + r + c0 * Q;
        float a[SPL];
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            a[i] = 0.f;
            vecB[g][0][VecB::at(r, c0 + i)] = 0.f;
            if (live) bwd_blk[(size_t)T * S + st_lane + i * Q] = 0.f;
        }
        int buf = 0;
        BwdRow<SPL> ring[DEPTH];
        __syncthreads();  // log table, initial vectors

        // phase 1: t = T-1 .. H.  Values start at zero, where an ulp is far below the error bound of
        // the estimate: in two-tier mode the first kWarmup steps use the double arithmetic throughout.
        const int cnt1 = T - H;
        auto sweep1 = [&](auto mode, int first, int count) {
            constexpr int M = decltype(mode)::value;
            const _Float16 *pre = sc_blk + (ptrdiff_t)(T - 1 - first) * row_stride;  // next row to fetch
            float *orow = bwd_blk + (ptrdiff_t)(T - 1 - first) * S;
            static_for<DEPTH>([&](auto k) {
                if ((int)k < count) {
                    ring[k].load(pre + sc_lane);
                    pre -= row_stride;
                }
            });
            pipelined<DEPTH>(count, [&](auto k, int j, auto checked) {
                const BwdRow<SPL> row = ring[k];
                if (!checked || j + DEPTH < count) {
                    ring[k].load(pre + sc_lane);
                    pre -= row_stride;
                }
                step_sync();
                const float4 nx = *reinterpret_cast<const float4 *>(&vecB[g][buf][VecB::of(4 * r)]);
                buf ^= 1;
                bwd_update<SPL, M>(a, nx, row, stay, logtab, [&] {
#pragma unroll
                    for (int i = 0; i < SPL; ++i) vecB[g][buf][VecB::at(r, c0 + i)] = a[i];
                });
                if (live) {
#pragma unroll
                    for (int i = 0; i < SPL; ++i) orow[st_lane + i * Q] = a[i];
                }
                orow -= S;
            });
        };
        const int warm = MODE == OFK_SCAN_TWO_TIER ? (cnt1 < kWarmup ? cnt1 : kWarmup) : 0;
        if constexpr (MODE == OFK_SCAN_TWO_TIER) sweep1(std::integral_constant<int, OFK_SCAN_PRECISE>{}, 0, warm);
        sweep1(std::integral_constant<int, MODE>{}, warm, cnt1 - warm);
        // forward lanes may run one step fewer in phase 1: cnt1 - H is 0 or 1; they wait here
        // middle: bwd[H..T] visible to the forward lanes, fwd[0..H-1] to these; the shift
        __syncthreads();
        block_barrier_lds();  // the forward lanes exchange their partial maxima
        block_barrier_lds();  // ... and publish the shift
        const float shift = shift_of[g];

        // phase 2: t = H-1 .. 0, posterior of row t from the parked fwd[t]
        const int cnt2 = H;
        int pb = 0;
        float e_prev[SPL];
        {
            const _Float16 *pre = sc_blk + (ptrdiff_t)(H - 1) * row_stride;
            const float *fpre = post_blk + (ptrdiff_t)(H - 1) * S;  // next parked row to fetch
            float *orow = bwd_blk + (ptrdiff_t)(H - 1) * S;
            float *prow = post_blk + (ptrdiff_t)H * S;  // row of the posterior that is stored next (one step late)
            float fring[DEPTH][SPL];
            static_for<DEPTH>([&](auto k) {
                if ((int)k < cnt2) {
                    ring[k].load(pre + sc_lane);
#pragma unroll
                    for (int i = 0; i < SPL; ++i) fring[k][i] = fpre[st_lane + i * Q];
                    pre -= row_stride;
                    fpre -= S;
                }
            });
            pipelined<DEPTH>(cnt2, [&](auto k, int j, auto checked) {
                const BwdRow<SPL> row = ring[k];
                float fv[SPL];
#pragma unroll
                for (int i = 0; i < SPL; ++i) fv[i] = fring[k][i];
                if (!checked || j + DEPTH < cnt2) {
                    ring[k].load(pre + sc_lane);
#pragma unroll
                    for (int i = 0; i < SPL; ++i) fring[k][i] = fpre[st_lane + i * Q];
                    pre -= row_stride;
                    fpre -= S;
                }
                step_sync();
                if (j > 0) {  // posterior of the previous row: its total is complete now
                    float total = part[g][0][pb ^ 1][0];
#pragma unroll
                    for (int w = 1; w < RW; ++w) total += part[g][0][pb ^ 1][w];
                    const float inv = __builtin_amdgcn_rcpf(total);
                    if (live) {
#pragma unroll
                        for (int i = 0; i < SPL; ++i) prow[st_lane + i * Q] = e_prev[i] * inv;
                    }
                }
                prow -= S;
                const float4 nx = *reinterpret_cast<const float4 *>(&vecB[g][buf][VecB::of(4 * r)]);
                buf ^= 1;
                bwd_update<SPL, MODE>(a, nx, row, stay, logtab, [&] {
#pragma unroll
                    for (int i = 0; i < SPL; ++i) vecB[g][buf][VecB::at(r, c0 + i)] = a[i];
                });
                float total;
#pragma unroll
                for (int i = 0; i < SPL; ++i) {
                    e_prev[i] = __builtin_amdgcn_exp2f(((fv[i] + a[i]) - shift) * kLog2e);
                    total = i ? total + e_prev[i] : e_prev[i];
                }
                total = group_sum<64>(total);
                if ((tid & 63) == 0) part[g][0][pb][wave] = total;
                pb ^= 1;
                if (live) {
#pragma unroll
                    for (int i = 0; i < SPL; ++i) orow[st_lane + i * Q] = a[i];
                }
                orow -= S;
            });
        }
        step_sync();
        if (cnt2 > 0) {
            float total = part[g][0][pb ^ 1][0];
#pragma unroll
            for (int w = 1; w < RW; ++w) total += part[g][0][pb ^ 1][w];
            const float inv = __builtin_amdgcn_rcpf(total);
            if (live) {
#pragma unroll
                for (int i = 0; i < SPL; ++i) post_blk[st_lane + i * Q] = e_prev[i] * inv;  // row 0
            }
        }
        // the forward lanes take T - H + 1 barriers in phase 2, these took H + 1
        for (int x = H + 1; x < T - H + 1; ++x) step_sync();
    } else {
        // ------------------------------ forward lanes ------------------------------
        const int s0 = SPL * l, q = s0 >> 2;  // own states s0 .. s0+SPL-1, all in quad q
        const unsigned sc_lane = g_eff * kCols * S + kCols * s0 + kLead;
        const unsigned st_lane = chunk_rows + s0;
        float f[SPL];
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            f[i] = 0.f;
            vecF[g][0][s0 + i] = 0.f;
        }
        int buf = 0;
        auto hand_on = [&] {  // the state vector, to the other lanes
            FloatRun<SPL> mine;
#pragma unroll
            for (int i = 0; i < SPL; ++i) mine.v[i] = f[i];
            mine.store(&vecF[g][buf][s0]);
        };
        FwdRow<SPL> ring[DEPTH];
        __syncthreads();

        // phase 1: t = 0 .. H-1, fwd[t] parked in post[t]; warm-up as for the backward lanes
        const int cnt1 = H;
        auto sweep1 = [&](auto mode, int first, int count) {
            constexpr int M = decltype(mode)::value;
            const _Float16 *pre = sc_blk + (ptrdiff_t)first * row_stride;
            float *prow = post_blk + (size_t)first * S;
            static_for<DEPTH>([&](auto k) {
                if ((int)k < count) {
                    ring[k].load(pre + sc_lane);
                    pre += row_stride;
                }
            });
            pipelined<DEPTH>(count, [&](auto k, int j, auto checked) {
                const FwdRow<SPL> row = ring[k];
                if (!checked || j + DEPTH < count) {
                    ring[k].load(pre + sc_lane);
                    pre += row_stride;
                }
                if (live) {
                    FloatRun<SPL> mine;
#pragma unroll
                    for (int i = 0; i < SPL; ++i) mine.v[i] = f[i];
                    mine.store(prow + st_lane);
                }
                prow += S;
                step_sync();
                const float p0 = vecF[g][buf][q], p1 = vecF[g][buf][q + Q];
                const float p2 = vecF[g][buf][q + 2 * Q], p3 = vecF[g][buf][q + 3 * Q];
                buf ^= 1;
                fwd_update<SPL, M>(f, p0, p1, p2, p3, row, stay, logtab, hand_on);
            });
        };
        const int warm = MODE == OFK_SCAN_TWO_TIER ? (cnt1 < kWarmup ? cnt1 : kWarmup) : 0;
        if constexpr (MODE == OFK_SCAN_TWO_TIER) sweep1(std::integral_constant<int, OFK_SCAN_PRECISE>{}, 0, warm);
        sweep1(std::integral_constant<int, MODE>{}, warm, cnt1 - warm);
        for (int x = cnt1; x < T - H; ++x) step_sync();  // the backward lanes' extra step

        // middle: shift = max_s(fwd[H][s] + bwd[H][s]) - 10
        __syncthreads();
        {
            const int bbuf = (T - H) & 1;  // where the backward lanes left bwd[H]
            FloatRun<SPL> bh;
            bh.load(&vecB[g][bbuf][VecB::of(s0)]);
            float m = f[0] + bh.v[0];
#pragma unroll
            for (int i = 1; i < SPL; ++i) m = fmaxf(m, f[i] + bh.v[i]);
            m = group_max<64>(m);
            if ((tid & 63) == 0) part[g][1][0][wave] = m;
            block_barrier_lds();
            m = part[g][1][0][0];
#pragma unroll
            for (int w = 1; w < RW; ++w) m = fmaxf(m, part[g][1][0][w]);
            if (l == 0) shift_of[g] = m - 10.0f;
            block_barrier_lds();
        }
        const float shift = shift_of[g];

        // phase 2: rows t = H .. T
        const int cnt2 = T - H + 1;
        int pb = 1;  // parity 0 of part[][1] was used for the maximum just now
        {
            const _Float16 *pre = sc_blk + (ptrdiff_t)H * row_stride;
            const float *bpre = bwd_blk + (size_t)H * S;
            float *prow = post_blk + (size_t)H * S;
            FloatRun<SPL> bring[DEPTH];
            static_for<DEPTH>([&](auto k) {
                if ((int)k < cnt2 - 1) ring[k].load(pre + sc_lane);
                if ((int)k < cnt2) bring[k].load(bpre + st_lane);
                pre += row_stride;
                bpre += S;
            });
            pipelined<DEPTH, 1>(cnt2, [&](auto k, int j, auto checked) {
                const FwdRow<SPL> row = ring[k];
                const FloatRun<SPL> bw = bring[k];
                if (!checked || j + DEPTH < cnt2 - 1) ring[k].load(pre + sc_lane);
                if (!checked || j + DEPTH < cnt2) bring[k].load(bpre + st_lane);
                pre += row_stride;
                bpre += S;
                FloatRun<SPL> e;
                float total;
#pragma unroll
                for (int i = 0; i < SPL; ++i) {
                    e.v[i] = __builtin_amdgcn_exp2f(((f[i] + bw.v[i]) - shift) * kLog2e);
                    total = i ? total + e.v[i] : e.v[i];
                }
                total = group_sum<64>(total);
                if ((tid & 63) == 0) part[g][1][pb][wave] = total;
                step_sync();
                total = part[g][1][pb][0];
#pragma unroll
                for (int w = 1; w < RW; ++w) total += part[g][1][pb][w];
                pb ^= 1;
                const float inv = __builtin_amdgcn_rcpf(total);
#pragma unroll
                for (int i = 0; i < SPL; ++i) e.v[i] *= inv;
                if (live) e.store(prow + st_lane);
                prow += S;
                if (!checked || j + 1 < cnt2) {
                    const float p0 = vecF[g][buf][q], p1 = vecF[g][buf][q + Q];
                    const float p2 = vecF[g][buf][q + 2 * Q], p3 = vecF[g][buf][q + 3 * Q];
                    buf ^= 1;
                    fwd_update<SPL, MODE>(f, p0, p1, p2, p3, row, stay, logtab, hand_on);
                }
            });
        }
    }
}

const LogSeries kSeries = {OFA_LOG_SERIES, OFA_EXP_COEFS};

// The always-double and the hardware-only arithmetic exist for tests and measurements: they are
// built with the fewest states per lane only (the entry points below ask for nothing else).
template <int S>
constexpr int kPlainSpl = S >= 1024 ? 2 : 1;

// Rows that the backward sweep keeps in flight with one state to a lane and the default arithmetic: 8 (1024 states: 6) | 12 (8) | 16 (10) |
// 20 (12) rows, ms, T = 1666: 512 chunks of 64 states 0.432 | 0.414 | 0.399 | 0.393, 512 of 256 states 0.733 | 0.711 | 0.700 | 0.694, 256 of
// 1024 states 1.262 | 1.235 | 1.25 | 1.227; 20 take so many registers that 1000 chunks of 256 states find no room (T = 1000: 0.70, 0.88).
// Several states to a lane fill the machine with fewer rows (1024 chunks of 256 states: 1.26 with 5, 8 or 12).
#ifndef OFK_DEPTH_DEEP
#define OFK_DEPTH_DEEP 16
#endif
#ifndef OFK_DEPTH_DEEP_1024
#define OFK_DEPTH_DEEP_1024 8
#endif

// Where sixteen rows, 120 registers, cost more than they give, and eight, 88 to 90 registers, are kept instead: more than four waves for
// every SIMD of 256 compute units, which only states per lane that were asked for bring about.  256 states, one to a
// lane, T = 300, ms, 8 | 16 rows: 1024 chunks 0.249 | 0.251, 1100 0.296 | 0.347, 2048 0.468 | 0.487, 2100 0.515 | 0.553; 8192 of 64 0.443 | 0.454.
// Beside another decode's merged kernel of 256 states sixteen are no dearer: four of its waves on a SIMD, of 96 registers (104 before, when
// eight rows were 2 % ahead), leave room for a wave of either kind, and with five columns, 120 registers, for neither.  Two decodes in
// flight, ms, 8 | 16 rows, T = 1666: 385 chunks 2.893 | 2.901, 450 3.126 | 3.132, 512 3.298 | 3.313 (runs differ by 3 %), 640 5.018 | 5.023,
// 1024 7.348 | 7.354; T = 600: 395 1.244 | 1.244, 512 1.333 | 1.324; T = 1000: 800 4.261 | 4.255; five columns: 512 3.483 | 3.507, 1024 7.735 |
// 7.731, T = 1201 2.570 | 2.573, T = 600 1.389 | 1.388.
constexpr long kWavesOfDepth16 = 4096;
template <int S>
bool eight_rows(int N) {
    return (long)N * (S / 64) > kWavesOfDepth16;
}

// Up to which magnitude of its values a sweep with one state to a lane takes the double arithmetic for every update at once.  An ulp of small
// values is below or near the estimate's bound, most steps have several unsettled updates somewhere in a chunk, and the double arithmetic
// behind an estimate and its verdict takes longer than by itself.  Values grow by about four a step; below 0 | 256 | 512 | 1024 | 2048 |
// 4096, backward sweep, us: 5 chunks of 64 states, T = 512 154 | 142 | 137 | 133 | 139 | 140; 512 of them, T = 1666 386 | 376 | 369 | 369 |
// 378 | 422; 16 of 256 states, T = 1666 577 | 565 | 558 | 548 | 538 | 555; 200, T = 600 258 | 246 | 239 | 228 | 216 | 217.  Where waves
// share a SIMD the other waves' trips are hidden and instructions count: 400 of 256 states, T = 256 138 | 135 | 143 | 146; 37 of 1024, T = 833
// 662 | 652 | 659 | 678.  The forward sweeps beside a search lose less time to unsettled updates (16 of 256 states 599 | 592 | 588 | 584 | 590 | 628).
uint32_t double_below(int S, int N, bool backward) {
    constexpr uint32_t k256 = 0x43800000u, k1024 = 0x44800000u, k2048 = 0x45000000u;  // as floats
    if ((long)N * (S / 64) > 1024) return S == 256 && !backward ? 0u : k256;  // more than a wave for every SIMD, or sixteen waves to a chunk
    return S == 1024 ? k256 : S == 256 && backward ? k2048 : k1024;
}

// Where the kernels have these early steps.  What follows them in the same kernel is slower for it where waves share a SIMD.  Backward sweep of 256
// states, us, without | with: 300 chunks, T = 96 59 | 55, 200 109 | 107, 300 156 | 155, 500 243 | 246; 512, T = 96 67 | 63, 200 118 | 115, 300 172 |
// 172, 500 248 | 252, 1666 677 | 711, with five columns 695 | 732; of the other models the early steps are ahead at any size (1024 states, 160 chunks, T = 64
// 74 | 63, 833 661 | 655; 2048 of 64, T = 1000 357 | 350).  Forward sweep of 64 states beside a search: 1024 chunks, T = 300 184 | 175, T = 1666 733 |
// 685; 1500 234 | 315 and 1002 | 1324.  Whole calls of 2048 chunks 614 | 711 at T = 300, but 3116 | 3034 at T = 1666, where the slower sweep leaves more
// to the search beside it: the rule goes by chunks alone and gives that away.
bool early_backward(int S, int T, int N) { return S != 256 || N <= 256 || T <= 256; }
constexpr int kEarlyForwardChunks = 1024;

template <int S, int SPL, int DEPTH>
int launch_bwd(int mode, const void *scores, float *bwd, int T, int N, float stay, Queue st) {
    using Sh = Shape<S, SPL>;
    constexpr int kDeep = SPL > 1 ? DEPTH : S >= 1024 ? OFK_DEPTH_DEEP_1024 : OFK_DEPTH_DEEP;
    const dim3 grid((N + Sh::kChunks - 1) / Sh::kChunks), block(Sh::kThreads);
    const _Float16 *sc = static_cast<const _Float16 *>(scores);
    switch (mode) {
        case OFK_SCAN_TWO_TIER:
            if constexpr (SPL == 1 && S <= 256) {
                if (eight_rows<S>(N)) {
                    queue_kernel((bwd_scan_kernel<S, SPL, DEPTH, OFK_SCAN_TWO_TIER, false>), grid, block, 0, st, sc, bwd, T, N, stay, 0u, kSeries);
                    break;
                }
            }
            if constexpr (SPL == 1) {
                if (early_backward(S, T, N)) {
                    queue_kernel((bwd_scan_kernel<S, SPL, kDeep, OFK_SCAN_TWO_TIER, true>), grid, block, 0, st, sc, bwd, T, N, stay, double_below(S, N, true), kSeries);
                    break;
                }
            }
            queue_kernel((bwd_scan_kernel<S, SPL, kDeep, OFK_SCAN_TWO_TIER, false>), grid, block, 0, st, sc, bwd, T, N, stay, 0u, kSeries);
            break;
        case OFK_SCAN_PRECISE:
            if constexpr (SPL == kPlainSpl<S>)
                queue_kernel((bwd_scan_kernel<S, SPL, DEPTH, OFK_SCAN_PRECISE, false>), grid, block, 0, st, sc, bwd, T, N, stay, 0u, kSeries);
            else
                return OFK_BAD_ARGS;
            break;
        case OFK_SCAN_FAST:
            if constexpr (SPL == kPlainSpl<S>)
                queue_kernel((bwd_scan_kernel<S, SPL, DEPTH, OFK_SCAN_FAST, false>), grid, block, 0, st, sc, bwd, T, N, stay, 0u, kSeries);
            else
                return OFK_BAD_ARGS;
            break;
        default: return OFK_BAD_ARGS;
    }
    return (int)hipGetLastError();
}

template <int S, int SPL, int DEPTH>
int launch_fwd(int mode, const void *scores, const float *bwd, float *post, int T, int N, float stay, Queue st) {
    using Sh = Shape<S, SPL>;
    const dim3 grid((N + Sh::kChunks - 1) / Sh::kChunks), block(Sh::kThreads);
    const _Float16 *sc = static_cast<const _Float16 *>(scores);
    switch (mode) {
        case OFK_SCAN_TWO_TIER:
            // Recursion and posterior on separate waves, one chunk per group of twice the lanes: where a chunk
            // spans several waves, and while that leaves every SIMD at most four of them (measured, 256 states:
            // 512 chunks 1.17 ms against 1.41 ms beside the beam search, 1024 chunks 3.5 against 3.1)
            if constexpr (Sh::kMultiWave && 2 * Sh::kLanes <= 1024) {
                if ((long)N * (2 * Sh::kLanes / 64) <= 4096) {
                    queue_kernel((fwd_post_roles_kernel<S, SPL, kRolesDepth>), dim3(N), dim3(2 * Sh::kLanes), 0, st, sc, bwd, post,
                                       T, N, stay, double_below(S, N, false), kSeries);
                    break;
                }
            }
            if constexpr (S == 64 && SPL == 1) {
                if (N <= kEarlyForwardChunks) {
                    queue_kernel((fwd_post_kernel<S, SPL, DEPTH, OFK_SCAN_TWO_TIER, true>), grid, block, 0, st, sc, bwd, post, T, N, stay, double_below(S, N, false), kSeries);
                    break;
                }
            }
            queue_kernel((fwd_post_kernel<S, SPL, DEPTH, OFK_SCAN_TWO_TIER, false>), grid, block, 0, st, sc, bwd, post, T, N, stay, 0u, kSeries);
            break;
        case OFK_SCAN_PRECISE:
            if constexpr (SPL == kPlainSpl<S>)
                queue_kernel((fwd_post_kernel<S, SPL, DEPTH, OFK_SCAN_PRECISE, false>), grid, block, 0, st, sc, bwd, post, T, N, stay, 0u, kSeries);
            else
                return OFK_BAD_ARGS;
            break;
        case OFK_SCAN_FAST:
            if constexpr (SPL == kPlainSpl<S>)
                queue_kernel((fwd_post_kernel<S, SPL, DEPTH, OFK_SCAN_FAST, false>), grid, block, 0, st, sc, bwd, post, T, N, stay, 0u, kSeries);
            else
                return OFK_BAD_ARGS;
            break;
        default: return OFK_BAD_ARGS;
    }
    return (int)hipGetLastError();
}

template <int S, int SPL, int DEPTH>
int launch_fused(int mode, const void *scores, float *bwd, float *post, int T, int N, float stay, Queue st) {
    using Sh = FusedShape<S, SPL>;
    const dim3 grid((N + Sh::kChunks - 1) / Sh::kChunks), block(Sh::kThreads);
    const _Float16 *sc = static_cast<const _Float16 *>(scores);
    switch (mode) {
        case OFK_SCAN_TWO_TIER:
            queue_kernel((scan_post_kernel<S, SPL, DEPTH, OFK_SCAN_TWO_TIER>), grid, block, 0, st, sc, bwd, post, T, N, stay, kSeries);
            break;
        case OFK_SCAN_PRECISE:
            if constexpr (SPL == kPlainSpl<S>)
                queue_kernel((scan_post_kernel<S, SPL, DEPTH, OFK_SCAN_PRECISE>), grid, block, 0, st, sc, bwd, post, T, N, stay, kSeries);
            else
                return OFK_BAD_ARGS;
            break;
        case OFK_SCAN_FAST:
            if constexpr (SPL == kPlainSpl<S>)
                queue_kernel((scan_post_kernel<S, SPL, DEPTH, OFK_SCAN_FAST>), grid, block, 0, st, sc, bwd, post, T, N, stay, kSeries);
            else
                return OFK_BAD_ARGS;
            break;
        default: return OFK_BAD_ARGS;
    }
    return (int)hipGetLastError();
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// States per lane: the largest of {4, 2, 1} (fewest lanes, least LDS traffic per state)
// that still gives every SIMD of the device (256 CUs x 4) a wave; small batches are
// spread thinner.  1024 states stop at 2, except in the backward sweep (bwd_scan below).
// The sweeps of the smaller models measure faster with two waves per SIMD (hac, 512 chunks:
// backward 1.29 ms against 1.33 ms; forward + posterior beside the beam search 1.41 ms against
// 1.61 ms, which is 13 000 chunks/s of a whole decode).
// So does the backward sweep of 1024 states, which has the machine to itself (256 chunks, five columns: 1.91 ms
// with one wave per SIMD, 1.53 with two).
// `forced` = 4, 2 or 1 overrides the choice (0 = choose).
int states_per_lane(int S, int N, bool backward, int forced) {
    const int min_spl = S >= 1024 ? 2 : 1;
    if (forced == 4 || forced == 2 || forced == 1) return forced < min_spl ? min_spl : forced;
    const long wanted = S <= 256 || backward ? 2048 : 1024;
    for (int spl = 4; spl > min_spl; spl >>= 1) {
        const long waves = ((long)N * (S / spl) + 63) / 64;
        if (waves >= wanted) return spl;
    }
    return min_spl;
}

}  // namespace

#ifndef OFK_DEPTH
#define OFK_DEPTH 8
#endif
#ifndef OFK_DEPTH_1024
#define OFK_DEPTH_1024 6
#endif
// The one-kernel scans keep the rows of two sweeps in flight.  Rows of one chunk lie N * C * 2 bytes
// apart; when that is a multiple of 4 MiB (2048 chunks of 256 states, 512 of 1024) all rows in
// flight fall onto the same DRAM banks, and with sixteen of them (eight per sweep) the kernel ran
// at half its rate and below (measured, 256 states, 2048 chunks: 8.97 ms; with four rows per sweep
// 5.69 ms, the rate of smaller batches; at 512 chunks both depths take 1.59 ms).  Hence half the depth
// here.  The separate sweeps, one row stored for every row read, do not show it, with sixteen rows either (backward, one state to a
// lane, T = 300, eight | sixteen rows: 2000 chunks 0.471 | 0.484, 2048 0.468 | 0.487).
#ifndef OFK_DEPTH_FUSED
#define OFK_DEPTH_FUSED 4
#endif
#ifndef OFK_DEPTH_FUSED_1024
#define OFK_DEPTH_FUSED_1024 3
#endif
// four states to a lane (2048 and more chunks of 256 states): a row more would not fit the 128 registers
#ifndef OFK_DEPTH_FUSED_WIDE
#define OFK_DEPTH_FUSED_WIDE 2
#endif
#define OFK_DISPATCH(BACKWARD, LAUNCH, ...)                                                    \
    switch (state_len * 8 + states_per_lane(1 << (2 * state_len), N, BACKWARD, lanes_asked(mode, spl))) { \
        case 3 * 8 + 4: return LAUNCH<64, 4, OFK_DEPTH>(__VA_ARGS__);                          \
        case 3 * 8 + 2: return LAUNCH<64, 2, OFK_DEPTH>(__VA_ARGS__);                          \
        case 3 * 8 + 1: return LAUNCH<64, 1, OFK_DEPTH>(__VA_ARGS__);                          \
        case 4 * 8 + 4: return LAUNCH<256, 4, OFK_DEPTH>(__VA_ARGS__);                         \
        case 4 * 8 + 2: return LAUNCH<256, 2, OFK_DEPTH>(__VA_ARGS__);                         \
        case 4 * 8 + 1: return LAUNCH<256, 1, OFK_DEPTH>(__VA_ARGS__);                         \
        case 5 * 8 + 4: return LAUNCH<1024, 4, OFK_DEPTH_1024>(__VA_ARGS__);                        \
        case 5 * 8 + 2: return LAUNCH<1024, 2, OFK_DEPTH_1024>(__VA_ARGS__);                        \
        default: return OFK_BAD_ARGS;                                                  \
    }

// States per lane of the two-directional kernel: one direction of a chunk owns whole waves, so
// 64 states need one state per lane; as many lanes as it takes to put four waves on every SIMD,
// within the 1024 threads of a workgroup.
static int fused_states_per_lane(int S, int N, int forced) {
    const int min_spl = S >= 1024 ? 2 : 1, max_spl = S >= 256 ? 4 : 1;
    if (forced == 4 || forced == 2 || forced == 1) return forced < min_spl ? min_spl : (forced > max_spl ? max_spl : forced);
    for (int spl = max_spl; spl > min_spl; spl >>= 1) {
        const long waves = (long)N * 2 * (S / spl) / 64;
        if (waves >= 4096) return spl;
    }
    return min_spl;
}

// states per lane to force: the caller's wish (0 = none) with the default arithmetic, the fewest otherwise
static int lanes_asked(int mode, int spl) { return mode == OFK_SCAN_TWO_TIER ? spl : 1; }

static int scan_posterior(const void *scores, float *bwd, float *post, int T, int N, int state_len, float stay,
                          int mode, int spl, void *stream, void *done) {
    if (!scores || !bwd || !post || T < 1 || N < 1 || !aligned16(scores) || !aligned16(bwd) || !aligned16(post))
        return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
    const int S = 1 << (2 * state_len);
    switch (state_len * 8 + (state_len >= 3 && state_len <= 5 ? fused_states_per_lane(S, N, lanes_asked(mode, spl)) : 0)) {
        case 3 * 8 + 1:  // 64 states: latency-bound, the deeper prefetch pays until the rows are 4 MiB apart
            if ((size_t)N * kCols * S * 2 < ((size_t)4 << 20))
                return launch_fused<64, 1, OFK_DEPTH>(mode, scores, bwd, post, T, N, stay, st);
            return launch_fused<64, 1, OFK_DEPTH_FUSED>(mode, scores, bwd, post, T, N, stay, st);
        case 4 * 8 + 4: return launch_fused<256, 4, OFK_DEPTH_FUSED_WIDE>(mode, scores, bwd, post, T, N, stay, st);
        case 4 * 8 + 2: return launch_fused<256, 2, OFK_DEPTH_FUSED>(mode, scores, bwd, post, T, N, stay, st);
        case 4 * 8 + 1: return launch_fused<256, 1, OFK_DEPTH_FUSED>(mode, scores, bwd, post, T, N, stay, st);
        case 5 * 8 + 4: return launch_fused<1024, 4, OFK_DEPTH_FUSED_1024>(mode, scores, bwd, post, T, N, stay, st);
        case 5 * 8 + 2: return launch_fused<1024, 2, OFK_DEPTH_FUSED_1024>(mode, scores, bwd, post, T, N, stay, st);
        default: return OFK_BAD_ARGS;
    }
}

static int bwd_scan(const void *scores, float *bwd, int T, int N, int state_len, float stay, int mode, int spl,
                    void *stream, void *done) {
    if (!scores || !bwd || T < 1 || N < 1 || !aligned16(scores) || !aligned16(bwd)) return OFK_BAD_ARGS;
    if (state_len < 3 || state_len > 5) return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
    // Up to a chunk for every compute unit, 1024 states take one state to a lane, sixteen waves: four waves on a SIMD fill each
    // other's waits, and a wave with half as many updates has the second tier's single trip more often (ms, two states to a
    // lane | one: 37 chunks, T = 833 0.76 | 0.67; 256, T = 1666 1.45 | 1.32; 9, T = 64 0.091 | 0.078).  Two such workgroups do
    // not fit a unit (257 chunks, T = 400 0.55 | 0.71; 512 0.68 | 0.75; 1024, T = 300 1.05 | 1.15).
    if (state_len == 5 && mode == OFK_SCAN_TWO_TIER && spl == 0 && N <= 256)
        return launch_bwd<1024, 1, OFK_DEPTH_1024>(mode, scores, bwd, T, N, stay, st);
    OFK_DISPATCH(true, launch_bwd, mode, scores, bwd, T, N, stay, st)
}

static int fwd_post_scan(const void *scores, const float *bwd, float *post, int T, int N, int state_len,
                         float stay, int mode, int spl, void *stream, void *done) {
    if (!scores || !bwd || !post || T < 1 || N < 1 || !aligned16(scores) || !aligned16(bwd) || !aligned16(post))
        return OFK_BAD_ARGS;
    if (state_len < 3 || state_len > 5) return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
    OFK_DISPATCH(false, launch_fwd, mode, scores, bwd, post, T, N, stay, st)
}

static int fwd_scan(const void *scores, float *fwd, int T, int N, int state_len, float stay, void *stream, void *done) {
    if (!scores || !fwd || T < 1 || N < 1 || state_len != 5 || !aligned16(scores) || !aligned16(fwd)) return OFK_BAD_ARGS;
    queue_kernel((fwd_scan_kernel<1024, OFK_DEPTH_1024>), dim3(N), dim3(1024), 0, Queue{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)},
                       static_cast<const _Float16 *>(scores), fwd, T, N, stay, double_below(1024, N, false), kSeries);
    return (int)hipGetLastError();
}

// The build compiles this file twice: with four columns, which also holds the entry points, and
// with five, whose kernels the entry points reach through the three functions named *_five.
#if OFK_COLS == 5
extern "C" int ofk_scan_posterior_five(const void *scores, float *bwd, float *post, int T, int N, int state_len,
                                       float stay, int mode, int spl, void *stream, void *done) {
    return scan_posterior(scores, bwd, post, T, N, state_len, stay, mode, spl, stream, done);
}
extern "C" int ofk_bwd_scan_five(const void *scores, float *bwd, int T, int N, int state_len, float stay, int mode,
                                 int spl, void *stream, void *done) {
    return bwd_scan(scores, bwd, T, N, state_len, stay, mode, spl, stream, done);
}
extern "C" int ofk_fwd_post_scan_five(const void *scores, const float *bwd, float *post, int T, int N,
                                      int state_len, float stay, int mode, int spl, void *stream, void *done) {
    return fwd_post_scan(scores, bwd, post, T, N, state_len, stay, mode, spl, stream, done);
}
extern "C" int ofk_fwd_scan_five(const void *scores, float *fwd, int T, int N, int state_len, float stay, void *stream, void *done) {
    return fwd_scan(scores, fwd, T, N, state_len, stay, stream, done);
}
#else
extern "C" int ofk_scan_posterior_five(const void *, float *, float *, int, int, int, float, int, int, void *, void *);
extern "C" int ofk_bwd_scan_five(const void *, float *, int, int, int, float, int, int, void *, void *);
extern "C" int ofk_fwd_post_scan_five(const void *, const float *, float *, int, int, int, float, int, int, void *, void *);
extern "C" int ofk_fwd_scan_five(const void *, float *, int, int, int, float, void *, void *);

extern "C" int ofk_scan_posterior(const void *scores, float *bwd, float *post, int T, int N, int state_len,
                                  int columns, float stay, int mode, int spl, void *stream, void *done) {
    if (columns == 5) return ofk_scan_posterior_five(scores, bwd, post, T, N, state_len, stay, mode, spl, stream, done);
    if (columns != 4) return OFK_BAD_ARGS;
    return scan_posterior(scores, bwd, post, T, N, state_len, stay, mode, spl, stream, done);
}

extern "C" int ofk_bwd_scan(const void *scores, float *bwd, int T, int N, int state_len, int columns, float stay,
                            int mode, int spl, void *stream, void *done) {
    if (columns == 5) return ofk_bwd_scan_five(scores, bwd, T, N, state_len, stay, mode, spl, stream, done);
    if (columns != 4) return OFK_BAD_ARGS;
    return bwd_scan(scores, bwd, T, N, state_len, stay, mode, spl, stream, done);
}

extern "C" int ofk_fwd_post_scan(const void *scores, const float *bwd, float *post, int T, int N, int state_len,
                                 int columns, float stay, int mode, int spl, void *stream, void *done) {
    if (columns == 5) return ofk_fwd_post_scan_five(scores, bwd, post, T, N, state_len, stay, mode, spl, stream, done);
    if (columns != 4) return OFK_BAD_ARGS;
    return fwd_post_scan(scores, bwd, post, T, N, state_len, stay, mode, spl, stream, done);
}

extern "C" int ofk_fwd_scan(const void *scores, float *fwd, int T, int N, int state_len, int columns, float stay, void *stream, void *done) {
    if (columns == 5) return ofk_fwd_scan_five(scores, fwd, T, N, state_len, stay, stream, done);
    if (columns != 4) return OFK_BAD_ARGS;
    return fwd_scan(scores, fwd, T, N, state_len, stay, stream, done);
}

extern "C" int ofk_posterior_rows(const float *bwd, float *post, int T, int N, int state_len, void *stream, void *done) {
    if (!bwd || !post || T < 1 || N < 1 || state_len != 5 || !aligned16(bwd) || !aligned16(post)) return OFK_BAD_ARGS;
    // Four rows to a workgroup, and few workgroups: the search beside this is longer, and more rows in flight only slow it down
    // (128 | 256 | 1024 workgroups, whole call, ms: 37 chunks, T = 833 1.27 | 1.27 | 1.29; 80, T = 1666 2.43 | 2.47 | 2.56).
    int parts = 128 / N;
    parts = parts < 1 ? 1 : parts;
    parts = parts < (T + 4) / 4 ? parts : (T + 4) / 4;
    queue_kernel((posterior_rows_kernel<1024>), dim3(N * parts), dim3(256), 0, Queue{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)}, bwd, post, T, parts);
    return (int)hipGetLastError();
}
#endif
