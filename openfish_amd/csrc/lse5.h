// The log-space update max + log(sum of five exponentials) of the scans, in its three arithmetics, with the
// wave reductions and the fp16 addition that go with it; for the kernels that run a recursion over the
// CRF states (scan.hip says what the arithmetics are).
#pragma once
#include <hip/hip_runtime.h>

#include "dmath.h"
#include "kernels.h"

namespace {


constexpr float kLog2e = 1.44269504088896340736f;
constexpr float kLn2 = 0.69314718055994530942f;

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}

// reductions over the lanes of one chunk inside a wave: LANES is 16 (one DPP row),
// 32 or 64 (whole wave).  Every lane of the group ends with the same bits.
template <int LANES>
__device__ __forceinline__ float group_sum(float x) {
    x += dpp<0x128>(x);  // row_ror:8
    x += dpp<0x124>(x);  // row_ror:4
    x += dpp<0x122>(x);  // row_ror:2
    x += dpp<0x121>(x);  // row_ror:1
    if constexpr (LANES >= 64) {
        // row sums travel across the rows: lane 15 of a row into the next row (rows 1 and 3), then
        // lane 31 into rows 2 and 3; lane 63 holds the total
        x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x142 /* row_bcast:15 */, 0xA, 0xF, false));
        x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x143 /* row_bcast:31 */, 0xC, 0xF, false));
        x = lane_value(x, 63);
    } else if constexpr (LANES == 32) {
        const float lo = lane_value(x, 0) + lane_value(x, 16), hi = lane_value(x, 32) + lane_value(x, 48);
        x = (threadIdx.x & 32) ? hi : lo;
    }
    return x;
}
template <int LANES>
__device__ __forceinline__ float group_max(float x) {
    x = fmaxf(x, dpp<0x128>(x));
    x = fmaxf(x, dpp<0x124>(x));
    x = fmaxf(x, dpp<0x122>(x));
    x = fmaxf(x, dpp<0x121>(x));
    if constexpr (LANES >= 64) {
        x = fmaxf(fmaxf(lane_value(x, 0), lane_value(x, 16)), fmaxf(lane_value(x, 32), lane_value(x, 48)));
    } else if constexpr (LANES == 32) {
        const float lo = fmaxf(lane_value(x, 0), lane_value(x, 16)), hi = fmaxf(lane_value(x, 32), lane_value(x, 48));
        x = (threadIdx.x & 32) ? hi : lo;
    }
    return x;
}

// What the CPU-faithful arithmetic reads: the logarithm's tables in LDS and the coefficients.  The
// coefficients travel as a kernel argument, which puts them into scalar registers for the whole
// kernel (as literals the compiler copies them into vector registers at every use).
struct LogSeries {
    double c[6];
    double e[OFA_EXP_COEF_COUNT];  // exponential: polynomial, rounding shift, log2(e), -ln 2
};
// Unsettled updates are looked at eight lanes each (settle_one, settle_eight): lanes 0 .. 4 evaluate the update's five
// exponentials, lanes 5 and 6 those of the rounding boundaries, drawn in.
__device__ __forceinline__ double certificate_unit() {
    const int k = threadIdx.x & 7;
    return k == 5 ? ofa::kProofLowerUnit : k == 6 ? ofa::kProofUpperUnit : 1.0;
}
struct LogArgs {
    const ofa::LogCell *cells;    // 32 cells, for the always-double arithmetic; null in a kernel that never takes it
    const ofa::LogCell *centred;  // ofa::kLogCentredCells cells, for the two-tier updates
    const double *series;
    const double *expc;
    float *lanes;  // 64 floats of LDS owned by the calling wave (two-tier updates only)
    int hurry = 3;  // the wave's priority during a trip through the second tier
    int rest = 0;   // and outside
    double unit = certificate_unit();
};

// Two-tier update, second tier: the updates whose estimate is unsettled.
//
// Unsettled estimates are right all but one or two times in a hundred (counted over the sweeps of 64, 256 and 1024
// states): the bound has to allow for roundings of the two running sums that never conspire.  So the second tier does not
// work the result out again but proves the estimate (dmath.h, lse5_bounds): seven exponentials side by side in seven lanes,
// five of the update and two of the boundaries, the running sum, one comparison; no logarithm, and
// nothing is handed back to the update's lane.  Where a proof fails, which it always does for |r| up to 32 or above 2^19, the
// update takes the logarithm of the running sum that the proof has formed.
//
// An instruction costs a wave that is alone on its SIMD about four cycles whatever it does (fp64 and
// dependent ones included), so a trip through this tier costs what it issues plus its LDS round trips.
// Three ways, by how many of the wave's updates are unsettled:
//   one (two waves in three that have any, with one state per lane): its seven arguments are read into scalar
//     registers and dealt to seven lanes, no LDS;
//   several: handed through LDS to groups of eight lanes, eight updates at a time;
//   many (only the first hundred time steps have them: values are small there and an ulp is tiny): no proof, every lane takes its
//     update's five exponentials, running sum and logarithm in double.
// Cycles of a lone wave for an update of 64 states with 0 | 1 | 2 to 8 | more of them unsettled: 250 | 620 | 780 | 890; when
// the second tier worked the results out (and took the logarithm in every trip) 245 | 740 | 975 | 985.  Together with the order
// of a step (see lse5_all) the backward sweep at T = 1666 went from 0.44 to 0.39 ms (1 chunk of 64 states), 0.68 to 0.58 (1 of
// 256), 0.85 to 0.74 (512 of 256), 1.54 to 1.43 (256 of 1024), the merged kernel of 1024 chunks of 256 states from 2.60 to 2.42.
// The tables that a kernel of THREADS threads reads, one cell a thread.
template <int MODE, int THREADS, bool WITH_PRECISE = false>
__device__ __forceinline__ void fill_log_tables(ofa::LogCell *cells, ofa::LogCell *centred) {
    constexpr bool kCells = MODE == OFK_SCAN_PRECISE || WITH_PRECISE, kCentred = MODE == OFK_SCAN_TWO_TIER;
    static_assert(THREADS >= (kCentred ? ofa::kLogCentredCells : 0) && (!kCells || THREADS >= 160), "a thread for every cell");
    const int tid = threadIdx.x;
    if (kCells && tid >= 128 && tid < 160) cells[tid - 128] = ofa::log_cell(tid - 128);
    if (kCentred && tid < ofa::kLogCentredCells) centred[tid] = ofa::log_centred_cell(tid);
}

// lane k of the result: x_k of lane `lane`, for k = 0 .. 6 (x_0 in the other lanes).  v_readlane may read a
// vector register one instruction after its write (hence the s_nop: the writes are not in sight), and a scalar
// register that a vector instruction has written may be read by one two instructions later (the order sees to that).
__device__ __forceinline__ float seven_to_lanes(float x0, float x1, float x2, float x3, float x4, float x5, float x6, int lane) {
    float x;
    uint32_t s0, s1, s2, s3, s4, s5, s6;
    asm("s_nop 0\n\t"
        "v_readlane_b32 %[s0], %[x0], %[lane]\n\t"
        "v_readlane_b32 %[s1], %[x1], %[lane]\n\t"
        "v_readlane_b32 %[s2], %[x2], %[lane]\n\t"
        "v_readlane_b32 %[s3], %[x3], %[lane]\n\t"
        "v_readlane_b32 %[s4], %[x4], %[lane]\n\t"
        "v_readlane_b32 %[s5], %[x5], %[lane]\n\t"
        "v_readlane_b32 %[s6], %[x6], %[lane]\n\t"
        "v_mov_b32 %[x], %[s0]\n\t"
        "v_writelane_b32 %[x], %[s1], 1\n\t"
        "v_writelane_b32 %[x], %[s2], 2\n\t"
        "v_writelane_b32 %[x], %[s3], 3\n\t"
        "v_writelane_b32 %[x], %[s4], 4\n\t"
        "v_writelane_b32 %[x], %[s5], 5\n\t"
        "v_writelane_b32 %[x], %[s6], 6"
        : [x] "=&v"(x), [s0] "=&s"(s0), [s1] "=&s"(s1), [s2] "=&s"(s2), [s3] "=&s"(s3), [s4] "=&s"(s4), [s5] "=&s"(s5), [s6] "=&s"(s6)
        : [x0] "v"(x0), [x1] "v"(x1), [x2] "v"(x2), [x3] "v"(x3), [x4] "v"(x4), [x5] "v"(x5), [x6] "v"(x6), [lane] "s"(lane));
    return x;
}

// fp32 running sum of lanes 0 .. 4 of e of the lane's row of 16, rounded after every term, to every lane of
// the row, as a double.  row_newbcast is the one DPP control that 64-bit operations have (their bank mask was seen to be
// ignored).  e has just been written: two wait states before a DPP operand may read it.
__device__ __forceinline__ double running_sum_of_five(double e) {
    double t;
    float s;
    const double one = 1.0;
#define OFK_TERM(K)                                                                           \
    "v_fmac_f64_dpp %[t], %[e], %[one] row_newbcast:" #K " row_mask:0xf bank_mask:0xf\n\t"    \
    "v_cvt_f32_f64 %[s], %[t]\n\t"                                                            \
    "v_cvt_f64_f32 %[t], %[s]\n\t"
    asm("s_nop 1\n\t"
        "v_mov_b64_dpp %[t], %[e] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f32_f64 %[s], %[t]\n\t"
        "v_cvt_f64_f32 %[t], %[s]\n\t"
        OFK_TERM(1) OFK_TERM(2) OFK_TERM(3) OFK_TERM(4)
        : [t] "=&v"(t), [s] "=&v"(s)
        : [e] "v"(e), [one] "v"(one));
#undef OFK_TERM
    return t;
}

// The same for groups of eight lanes, to the upper four lanes of the group: the sum so far comes from the lane below.
__device__ __forceinline__ float running_sum_along_eight(double e) {
    float s = (float)e;
#pragma unroll
    for (int k = 0; k < 4; ++k) s = (float)((double)dpp<0x111>(s) + e);  // row_shr:1
    return dpp<0x00>(s);                                                 // quad_perm:[0,0,0,0]
}

// the argument is a constant wherever this is inlined
__device__ __forceinline__ void set_priority(int level) {
    if (level == 0) __builtin_amdgcn_s_setprio(0);
    else if (level == 1) __builtin_amdgcn_s_setprio(1);
    else if (level == 2) __builtin_amdgcn_s_setprio(2);
    else __builtin_amdgcn_s_setprio(3);
}

// a value that is the same in every lane, kept in a scalar register so that what is decided by it is decided there
__device__ __forceinline__ int scalar(int x) {
    asm("" : "+s"(x));
    return x;
}

// m + ln s as the CPU path rounds it, s being its running sum: what is left to do where a proof fails
__device__ __forceinline__ float from_sum(float m, float s, const LogArgs &logtab) {
    return (float)((double)m + ofa::log_centred(s, logtab.centred[ofa::log_centred_index(s)], logtab.series));
}

// the one unsettled update, of lane `at`; whether its value may have changed
__device__ __forceinline__ bool settle_one(float &value, const float (&v)[5], float m, float lower, float upper, int at, const LogArgs &logtab) {
    const float x = seven_to_lanes(v[0] - m, v[1] - m, v[2] - m, v[3] - m, v[4] - m, lower, upper, at);
    const double e = ofa::exp_ldexp((double)x, logtab.expc, logtab.unit);
    const double s = running_sum_of_five(e);
    const uint32_t above = (uint32_t)__builtin_amdgcn_ballot_w64(s > e);  // in the first row of lanes
    if (__builtin_expect(scalar((int)((above & 0x60u) ^ 0x20u)) == 0, 1)) return false;
    const float r = from_sum(m, lane_value((float)s, 0), logtab);
    value = (int)(threadIdx.x & 63) == at ? r : value;
    return true;
}

// the same, of whichever state I .. SPL - 1 it is
template <int SPL, int I = 0>
__device__ __forceinline__ bool settle_single(float (&value)[SPL], const uint64_t (&mask)[SPL], const float (&v)[SPL][5], const float (&m)[SPL],
                                              const float (&lower)[SPL], const float (&upper)[SPL], const LogArgs &logtab) {
    if constexpr (I + 1 < SPL) {
        if (scalar(__builtin_popcountll(mask[I])) == 0) return settle_single<SPL, I + 1>(value, mask, v, m, lower, upper, logtab);
    }
    return settle_one(value[I], v[I], m[I], lower[I], upper[I], __builtin_ctzll(mask[I]), logtab);
}

// several unsettled updates, ranks first .. first + 7 of them (rank: per state and lane, of the unsettled ones)
template <int SPL>
__device__ __forceinline__ bool settle_eight(float (&value)[SPL], const uint64_t (&mask)[SPL], const int (&rank)[SPL], int first, int total,
                                             const float (&v)[SPL][5], const float (&m)[SPL], const float (&lower)[SPL],
                                             const float (&upper)[SPL], const LogArgs &logtab) {
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        if (__builtin_amdgcn_inverse_ballot_w64(mask[i]) && (SPL == 1 || (unsigned)(rank[i] - first) < 8u)) {
            float *slot = logtab.lanes + 8 * (rank[i] - first);
            *reinterpret_cast<float4 *>(slot) = make_float4(v[i][0] - m[i], v[i][1] - m[i], v[i][2] - m[i], v[i][3] - m[i]);
            *reinterpret_cast<float3 *>(slot + 4) = make_float3(v[i][4] - m[i], lower[i], upper[i]);
        }
    }
    // LDS operations of one wave complete in order
    const double e = ofa::exp_ldexp((double)logtab.lanes[threadIdx.x & 63], logtab.expc, logtab.unit);
    const float s = running_sum_along_eight(e);
    const uint64_t above = __builtin_amdgcn_ballot_w64((double)s > e);
    const int spare = 8 - (total - first);  // groups that hold nothing
    const uint64_t used = ~0ull >> (spare > 0 ? 8 * spare : 0);
    const uint64_t open = ((above & 0x6060606060606060ull) ^ 0x2020202020202020ull) & used;
    if (__builtin_expect(scalar((int)open | (int)(open >> 32)) == 0, 1)) return false;
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        const bool in = __builtin_amdgcn_inverse_ballot_w64(mask[i]) && (SPL == 1 || (unsigned)(rank[i] - first) < 8u);
        const float mine = __int_as_float(__builtin_amdgcn_ds_bpermute((8 * (rank[i] - first) + 4) << 2, __float_as_int(s)));
        const float r = from_sum(m[i], mine, logtab);
        value[i] = in ? r : value[i];
    }
    return true;
}

// mask[i]: the lanes whose update of state i is unsettled; at least one bit is set.  Whether a value may have changed.
// COMPACT: for steps that have no registers left for the double arithmetic written out.
template <int SPL, bool COMPACT>
__device__ __forceinline__ bool resolve_unsettled(float (&value)[SPL], const float (&sum)[SPL], const float (&half)[SPL],
                                                  const uint64_t (&mask)[SPL], const float (&v)[SPL][5], const float (&m)[SPL],
                                                  const LogArgs &logtab) {
    int total = 0;
#pragma unroll
    for (int i = 0; i < SPL; ++i) total += scalar(__builtin_popcountll(mask[i]));
    float lower[SPL], upper[SPL];
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        const ofa::Lse5Bounds b = ofa::lse5_bounds(value[i], half[i], m[i]);
        lower[i] = b.lower;
        upper[i] = b.upper;
    }
    if (__builtin_expect(total == 1, 1)) {
        return settle_single<SPL>(value, mask, v, m, lower, upper, logtab);
    }
    if (total <= 8 * SPL) {
        int rank[SPL], below = 0;
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            rank[i] = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask[i], (uint32_t)below));
            below += scalar(__builtin_popcountll(mask[i]));
        }
        if constexpr (SPL == 1) return settle_eight<SPL>(value, mask, rank, 0, total, v, m, lower, upper, logtab);
        bool changed = false;
        for (int first = 0; first < total; first += 8) changed |= settle_eight<SPL>(value, mask, rank, first, total, v, m, lower, upper, logtab);
        return changed;
    }
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        float s, r;
        if constexpr (COMPACT) {
            // a loop that passes the differences down its registers: an exponential at a time
            float d0 = v[i][0] - m[i], d1 = v[i][1] - m[i], d2 = v[i][2] - m[i], d3 = v[i][3] - m[i], d4 = v[i][4] - m[i];
            s = 0.f;
#pragma unroll 1
            for (int k = 0; k < 5; ++k) {
                s = (float)((double)s + ofa::exp_nonpos_ldexp(d0, logtab.expc));
                d0 = d1;
                d1 = d2;
                d2 = d3;
                d3 = d4;
            }
            r = from_sum(m[i], s, logtab);
        } else {
            const ofa::LogCell cell = logtab.centred[ofa::log_centred_index(sum[i])];  // arrives while the exponentials are evaluated
            s = (float)ofa::exp_nonpos_ldexp(v[i][0] - m[i], logtab.expc);
#pragma unroll
            for (int k = 1; k < 5; ++k) s = (float)((double)s + ofa::exp_nonpos_ldexp(v[i][k] - m[i], logtab.expc));
            r = (float)((double)m[i] + ofa::log_centred(s, cell, logtab.series));
        }
        value[i] = __builtin_amdgcn_inverse_ballot_w64(mask[i]) ? r : value[i];
    }
    return true;
}

// maximum of five in two instructions (the operands are never NaN here; fmaxf would first quiet
// each operand that comes out of inline assembly with an extra instruction)
__device__ __forceinline__ float max5(float a, float b, float c, float d, float e) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3\n\t"
        "v_max3_f32 %0, %0, %4, %5"
        : "=&v"(r) : "v"(a), "v"(b), "v"(c), "v"(d), "v"(e));
    return r;
}

// max + log(sum_i exp(v_i - max)) of the SPL states of a lane, sums taken in the order v[.][0] .. v[.][4].
// `publish` hands the values in `out` to the other lanes (writes to LDS that those do not read yet).  With two tiers
// that is done with the estimates, before the verdict on them is known, and again in the rare case that a value changes: the
// verdict's instructions then run while the writes are under way.  `beside` (argument: whether it is the first call) has what
// else the step has to issue, which goes where the comparison's mask is on its way to the scalar unit, and stores `out`; it
// follows publish each time.
// With two tiers the states share one test and one branch: reading a comparison's mask and branching on
// it costs a lone wave about as much as eight other instructions.
template <int SPL, int MODE, bool COMPACT = false, typename Publish, typename Beside>
__device__ __forceinline__ void lse5_all(float (&out)[SPL], const float (&v)[SPL][5], const LogArgs &logtab, Publish &&publish, Beside &&beside) {
    float m[SPL];
#pragma unroll
    for (int i = 0; i < SPL; ++i) m[i] = max5(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4]);
    if constexpr (MODE == OFK_SCAN_PRECISE) {
#pragma unroll
        for (int i = 0; i < SPL; ++i)
            out[i] = ofa::lse5_cpu_rounding_tab(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4], m[i], logtab.cells, logtab.series, logtab.expc);
        publish();
        beside(true);
    } else if constexpr (MODE == OFK_SCAN_TWO_TIER) {
        float sum[SPL], half[SPL], l2[SPL];
        uint64_t mask[SPL], any = 0;
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            const ofa::Lse5Value e = ofa::lse5_value(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4], m[i]);
            out[i] = e.value;
            sum[i] = e.sum;
            l2[i] = e.l2;
        }
        publish();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            const ofa::Lse5Estimate e = ofa::lse5_verdict(ofa::Lse5Value{out[i], sum[i], l2[i]}, m[i]);
            half[i] = e.half;
            mask[i] = __builtin_amdgcn_ballot_w64(!e.settled);
            asm volatile("" : "+s"(mask[i]));  // compared here, looked at further down
        }
        __builtin_amdgcn_sched_barrier(0);
        beside(true);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < SPL; ++i) any |= mask[i];
        if (any != 0) {
            // the chunk's other waves wait at the barrier for this one
            if (logtab.hurry != logtab.rest) set_priority(logtab.hurry);
            if (resolve_unsettled<SPL, COMPACT>(out, sum, half, mask, v, m, logtab)) {
                publish();
                beside(false);
            }
            if (logtab.hurry != logtab.rest) set_priority(logtab.rest);
        }
    } else {
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            float s = __builtin_amdgcn_exp2f((v[i][0] - m[i]) * kLog2e);
#pragma unroll
            for (int b = 1; b < 5; ++b) s += __builtin_amdgcn_exp2f((v[i][b] - m[i]) * kLog2e);
            out[i] = __builtin_fmaf(__builtin_amdgcn_logf(s), kLn2, m[i]);
        }
        publish();
        beside(true);
    }
}

// The same with the double arithmetic for every lane and no estimate before it: where most updates would turn out unsettled.
template <int SPL, typename Publish, typename Beside>
__device__ __forceinline__ void lse5_all_double(float (&out)[SPL], const float (&v)[SPL][5], const LogArgs &logtab, Publish &&publish, Beside &&beside) {
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        const float m = max5(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4]);
        float s = (float)ofa::exp_nonpos_ldexp(v[i][0] - m, logtab.expc);
#pragma unroll
        for (int k = 1; k < 5; ++k) {
            __builtin_amdgcn_sched_barrier(0);  // an exponential at a time: side by side they take 60 registers more, and no less time
            s = (float)((double)s + ofa::exp_nonpos_ldexp(v[i][k] - m, logtab.expc));
        }
        out[i] = from_sum(m, s, logtab);
    }
    publish();
    beside(true);
}

// whether a wave's values are still below `bits` (of a float) in magnitude: those of a step lie close together, lane 0 speaks for all
__device__ __forceinline__ bool values_below(float value, uint32_t bits) {
    return ((uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(value)) & 0x7fffffffu) < bits;
}

// x + (float)h for the fp16 value h in the low (HI = 0) or high half of a 32-bit register, in one
// instruction: v_fma_mix_f32 converts the half operand on the fly, the product with 1.0 is
// exact, so the result is the correctly rounded fp32 sum, bit for bit what v_cvt_f32_f16
// followed by v_add_f32 gives (checked for every fp16 bit pattern, subnormals included).
template <int HI>
__device__ __forceinline__ float add_half(uint32_t word, float x) {
    float r;
    if constexpr (HI)
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(word), "v"(x));
    else
        asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(word), "v"(x));
    return r;
}

}  // namespace
