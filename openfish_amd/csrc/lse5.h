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

// What the CPU-faithful logarithm reads: its table in LDS and its series coefficients.  The
// coefficients travel as a kernel argument, which puts them into scalar registers for the whole
// kernel (as literals the compiler copies them into vector registers at every use).
struct LogSeries {
    double c[6];
    double e[OFA_EXP_COEF_COUNT];  // exponential: polynomial, rounding shift, log2(e), -ln 2
};
struct LogArgs {
    const ofa::LogCell *cells;    // 32 cells, for the double arithmetic of all lanes
    const ofa::LogCell *centred;  // ofa::kLogCentredCells cells, for the second tier
    const double *series;
    const double *expc;
    float *lanes;  // 64 floats of LDS owned by the calling wave (two-tier updates only)
    int hurry = 3;  // the wave's priority during a trip through the second tier
};

// Two-tier update, second tier: the CPU path's own roundings for the updates whose estimate is unsettled.
//
// An instruction costs a wave that is alone on its SIMD about four cycles whatever it does (fp64 and
// dependent ones included), so a trip through this tier costs what it issues plus its LDS round trips.
// Three ways, by how many of the wave's updates are unsettled:
//   one (two waves in three that have any, with one state per lane): served by the whole wave without
//     LDS.  Its five differences are read into scalar registers and dealt to five lanes, which evaluate
//     the double exponentials side by side; every lane then forms the fp32 running sum through DPP
//     broadcasts and takes the logarithm;
//   several: handed through LDS to rows of 16 lanes, four updates at a time, or with several states per
//     lane to groups of eight lanes, eight at a time;
//   many (only the first few hundred time steps have them: values are small there and an ulp is tiny): the
//     double arithmetic for all lanes at once, which costs about as much as two trips per state of a lane.
// Backward sweep, T = 1666, together with the loads that are no longer all waited for every eight steps:
// 1 chunk of 64 states 0.56 -> 0.44 ms, 1 chunk of 256 states 0.78 -> 0.67, 512 chunks of 256 states 0.98 -> 0.86.
template <int MODE>
__device__ __forceinline__ void fill_log_tables(ofa::LogCell *cells, ofa::LogCell *centred) {
    const int tid = threadIdx.x;
    if (MODE != OFK_SCAN_FAST && tid >= 128 && tid < 160) cells[tid - 128] = ofa::log_cell(tid - 128);
    if (MODE == OFK_SCAN_TWO_TIER && tid < ofa::kLogCentredCells) centred[tid] = ofa::log_centred_cell(tid);
}

// lane k of the result: d_k of lane `lane`, for k = 0 .. 4 (d_0 in the other lanes).  v_readlane may read a
// vector register one instruction after its write (hence the s_nop: the writes are not in sight), and a scalar
// register that a vector instruction has written may be read by one two instructions later (the order sees to that).
__device__ __forceinline__ float five_to_lanes(float d0, float d1, float d2, float d3, float d4, int lane) {
    float x;
    uint32_t s0, s1, s2, s3, s4;
    asm("s_nop 0\n\t"
        "v_readlane_b32 %[s0], %[d0], %[lane]\n\t"
        "v_readlane_b32 %[s1], %[d1], %[lane]\n\t"
        "v_readlane_b32 %[s2], %[d2], %[lane]\n\t"
        "v_readlane_b32 %[s3], %[d3], %[lane]\n\t"
        "v_readlane_b32 %[s4], %[d4], %[lane]\n\t"
        "v_mov_b32 %[x], %[s0]\n\t"
        "v_writelane_b32 %[x], %[s1], 1\n\t"
        "v_writelane_b32 %[x], %[s2], 2\n\t"
        "v_writelane_b32 %[x], %[s3], 3\n\t"
        "v_writelane_b32 %[x], %[s4], 4"
        : [x] "=&v"(x), [s0] "=&s"(s0), [s1] "=&s"(s1), [s2] "=&s"(s2), [s3] "=&s"(s3), [s4] "=&s"(s4)
        : [d0] "v"(d0), [d1] "v"(d1), [d2] "v"(d2), [d3] "v"(d3), [d4] "v"(d4), [lane] "s"(lane));
    return x;
}

// fp32 running sum of lanes 0 .. 4 of e of the lane's row of 16, rounded after every term, to every lane of
// the row.  row_newbcast is the one DPP control that 64-bit operations have (their bank mask was seen to be
// ignored).  e has just been written: two wait states before a DPP operand may read it.
__device__ __forceinline__ float running_sum_of_five(double e) {
    double t;
    float s;
    const double one = 1.0;
#define OFK_TERM(K)                                                                           \
    "v_cvt_f64_f32 %[t], %[s]\n\t"                                                            \
    "v_fmac_f64_dpp %[t], %[e], %[one] row_newbcast:" #K " row_mask:0xf bank_mask:0xf\n\t"    \
    "v_cvt_f32_f64 %[s], %[t]\n\t"
    asm("s_nop 1\n\t"
        "v_mov_b64_dpp %[t], %[e] row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_cvt_f32_f64 %[s], %[t]\n\t"
        OFK_TERM(1) OFK_TERM(2) OFK_TERM(3) OFK_TERM(4)
        : [t] "=&v"(t), [s] "=&v"(s)
        : [e] "v"(e), [one] "v"(one));
#undef OFK_TERM
    return s;
}

// The same for groups of eight lanes, to lane 4 of the group only: the sum so far comes from the lane below.
__device__ __forceinline__ float running_sum_along_eight(double e) {
    float s = (float)e;
#pragma unroll
    for (int k = 0; k < 4; ++k) s = (float)((double)dpp<0x111>(s) + e);  // row_shr:1
    return s;
}

// mask[i]: the lanes whose update of state i is unsettled; at least one bit is set
template <int SPL>
__device__ __forceinline__ void resolve_unsettled(float (&value)[SPL], const float (&sum)[SPL], const uint64_t (&mask)[SPL],
                                                  const float (&v)[SPL][5], const float (&m)[SPL], const LogArgs &logtab) {
    const int lane = threadIdx.x & 63;
    if (SPL == 1 && (mask[0] & (mask[0] - 1)) == 0) {
        const int at = __builtin_ctzll(mask[0]);
        const float near = lane_value(sum[0], at);
        const ofa::LogCell cell = logtab.centred[ofa::log_centred_index(near)];  // arrives while the exponentials are evaluated
        const float mm = lane_value(m[0], at);
        const float x = five_to_lanes(v[0][0] - m[0], v[0][1] - m[0], v[0][2] - m[0], v[0][3] - m[0], v[0][4] - m[0], at);
        const float s = running_sum_of_five(ofa::exp_ldexp((double)x, logtab.expc));  // in the first row of lanes
        const float r = lane_value((float)((double)mm + ofa::log_centred(s, cell, logtab.series)), 0);
        value[0] = lane == at ? r : value[0];
        return;
    }
    int total = 0, rank[SPL];
#pragma unroll
    for (int i = 0; i < SPL; ++i) {
        rank[i] = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask[i] >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask[i], (uint32_t)total));
        total += __builtin_amdgcn_readfirstlane(__builtin_popcountll(mask[i]));
    }
    constexpr int kSlots = SPL == 1 ? 4 : 8, kStride = 64 / kSlots;  // updates per trip, lanes per update
    if (total <= 2 * kSlots * SPL - (SPL == 1 ? kSlots : 0)) {
        for (int first = 0; first < total; first += kSlots) {
            bool in[SPL];
#pragma unroll
            for (int i = 0; i < SPL; ++i) {
                in[i] = ((mask[i] >> lane) & 1) && (unsigned)(rank[i] - first) < (unsigned)kSlots;
                if (in[i]) {
                    float *slot = logtab.lanes + kStride * (rank[i] - first);
                    *reinterpret_cast<float4 *>(slot) = make_float4(v[i][0] - m[i], v[i][1] - m[i], v[i][2] - m[i], v[i][3] - m[i]);
                    *reinterpret_cast<float4 *>(slot + 4) = make_float4(v[i][4] - m[i], 0.f, m[i], sum[i]);
                }
            }
            // LDS operations of one wave complete in order
            const float2 ms = *reinterpret_cast<const float2 *>(logtab.lanes + (lane & -kStride) + 6);
            const float x = logtab.lanes[lane];
            const ofa::LogCell cell = logtab.centred[ofa::log_centred_index(ms.y)];  // arrives while the exponentials are evaluated
            const double e = ofa::exp_ldexp((double)x, logtab.expc);
            const float s = SPL == 1 ? running_sum_of_five(e) : running_sum_along_eight(e);
            const float r = (float)((double)ms.x + ofa::log_centred(s, cell, logtab.series));
#pragma unroll
            for (int i = 0; i < SPL; ++i) {
                const float mine = __int_as_float(__builtin_amdgcn_ds_bpermute((kStride * (rank[i] - first) + 4) << 2, __float_as_int(r)));
                value[i] = in[i] ? mine : value[i];
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            const float r = ofa::lse5_cpu_rounding_tab(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4], m[i], logtab.cells, logtab.series, logtab.expc);
            value[i] = (mask[i] >> lane) & 1 ? r : value[i];
        }
    }
}

// maximum of three in one instruction (the operands are never NaN here; fmaxf would first quiet
// each operand that comes out of inline assembly with an extra instruction)
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// max + log(sum_i exp(v_i - max)) of the SPL states of a lane, sums taken in the order v[.][0] .. v[.][4].
// With two tiers the states share one test and one branch: reading a comparison's mask and branching on
// it costs a lone wave about as much as eight other instructions.
template <int SPL, int MODE>
__device__ __forceinline__ void lse5_all(float (&out)[SPL], const float (&v)[SPL][5], const LogArgs &logtab) {
    float m[SPL];
#pragma unroll
    for (int i = 0; i < SPL; ++i) m[i] = max3(max3(v[i][0], v[i][1], v[i][2]), v[i][3], v[i][4]);
    if constexpr (MODE == OFK_SCAN_PRECISE) {
#pragma unroll
        for (int i = 0; i < SPL; ++i)
            out[i] = ofa::lse5_cpu_rounding_tab(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4], m[i], logtab.cells, logtab.series, logtab.expc);
    } else if constexpr (MODE == OFK_SCAN_TWO_TIER) {
        float sum[SPL];
        uint64_t mask[SPL], any = 0;
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            const ofa::Lse5Estimate e = ofa::lse5_estimate(v[i][0], v[i][1], v[i][2], v[i][3], v[i][4], m[i]);
            out[i] = e.value;
            sum[i] = e.sum;
            mask[i] = __builtin_amdgcn_ballot_w64(!e.settled);
            any |= mask[i];
        }
        if (any != 0) {
            // the chunk's other waves wait at the barrier for this one
            if (logtab.hurry == 3) __builtin_amdgcn_s_setprio(3);
            else if (logtab.hurry == 1) __builtin_amdgcn_s_setprio(1);
            resolve_unsettled<SPL>(out, sum, mask, v, m, logtab);
            __builtin_amdgcn_s_setprio(0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < SPL; ++i) {
            float s = __builtin_amdgcn_exp2f((v[i][0] - m[i]) * kLog2e);
#pragma unroll
            for (int b = 1; b < 5; ++b) s += __builtin_amdgcn_exp2f((v[i][b] - m[i]) * kLog2e);
            out[i] = __builtin_fmaf(__builtin_amdgcn_logf(s), kLn2, m[i]);
        }
    }
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
