// Beam search over CRF scores, gfx950.
//
// Every chunk is served by two wavefronts of a workgroup (with the forward sweep in it, beam_kernel
// with FWD > 0, by several more).  The loader wave streams the
// rows the search needs (scores[t] as fp16 and bwd[t+1] as fp32) from HBM into an LDS
// ring, several rows ahead; the search wave runs the search with the 32-wide beam
// resident in registers/LDS.  The two communicate through two LDS counters (rows ready /
// rows consumed), so the search never waits on a dependent HBM gather.  A workgroup holds
// two or four chunks, so that its waves spread over the four SIMDs of a compute unit.
//
// Search wave lane layout: lanes 2i and 2i+1 both hold beam element i; lane 2i+h holds
// its step candidates with new base 2h and 2h+1, the even lane also its stay candidate,
// so that lane order is the CPU path's candidate order (steps 4i+b, then stays) and
// ranks are masked bit counts.
// The search reproduces the CPU path (reference src/beam_search.c:117-439) to the
// bit: same fp32 operation order, double-precision log-sum-exp for merges, the
// same cut-off bisection, first-come compaction and final best-to-slot-0 swap.
// Instead of sorting, the cut-off uses wave ballots and population counts, and
// survivors are ranked with ballot prefix counts.
//
// Stay/step merging: a stay of element i merges with the step (j, b_i) whose hash
// crc(hash_j, b_i) equals hash_i.  The 2-bit CRC update is a bijection of the
// 32-bit state, so this is the same as hash_j == crc^-1(hash_i, b_i) =: want_i, the hash
// of the element's sequence without its last base.  Every beam element carries both
// words (a candidate's `want` is its parent's hash, or its parent's `want` for a stay), and
// the element j is found through a hash index in LDS: every live element files
// one word (the hash, with generation and slot in place of the bits that choose the bucket) under
// those bits of its hash, reads its own entry back, and looks up the entry filed under the same bits of `want`.  If every element finds its own
// entry intact, all hashes are pairwise distinct and every existing partner is found by
// exactly one probe (the full 32 bits are compared); otherwise (two elements in one
// bucket, one step in ten, twenty or forty by the size of the index; equal hashes, only after a CRC collision) the step
// falls back to comparing `want` with all 32 hashes.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <mutex>
#include <type_traits>

#include "kernels.h"
#include "queue.h"
#include "lse5.h"

namespace {

constexpr int kW = OFK_BEAM_WIDTH;
constexpr int kTraceRows = 128;  // rows that the traceback takes at a time
constexpr uint32_t kPoly = 0x82f63b78u;
constexpr uint32_t kSeed = 0x12345678u;

constexpr uint32_t crc_bits(uint32_t crc, uint32_t bits, int n) {
    for (int i = 0; i < n; ++i) {
        const uint32_t feed = (bits ^ crc) & 1u;
        crc >>= 1;
        if (feed) crc ^= kPoly;
        bits >>= 1;
    }
    return crc;
}
// CRC-32C is linear over GF(2): two update steps are (crc >> 2) xor a table entry chosen
// by the two low bits of crc ^ bits, and the entry for 3 is the xor of those for 1 and 2.
constexpr uint32_t kTab1 = crc_bits(1u, 0u, 2);
constexpr uint32_t kTab2 = crc_bits(2u, 0u, 2);
static_assert(crc_bits(3u, 0u, 2) == (kTab1 ^ kTab2), "crc linearity");
static_assert((kTab1 >> 30) == 1u && (kTab2 >> 30) == 2u, "top bits identify the table entry");

__device__ __forceinline__ uint32_t crc_tab(uint32_t x) {
    return ((0u - (x & 1u)) & kTab1) ^ ((0u - ((x >> 1) & 1u)) & kTab2);
}
__device__ __forceinline__ uint32_t crc2(uint32_t crc, uint32_t base) {
    return (crc >> 2) ^ crc_tab((crc ^ base) & 3u);
}
// (a & b) ^ c in one instruction (in the order that the compiler finds by itself the inverse below takes two more)
__device__ __forceinline__ uint32_t and_xor(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_bitop3_b32(a, b, c, 0x6a); }
// the hash h with crc2(h, base & 3) == crc: ((crc ^ entry k) << 2) | (k ^ base), k the two top bits.  With the entries' top bits
// left out those of crc stay, and come round to the bottom.
__device__ __forceinline__ uint32_t crc2_inverse(uint32_t crc, uint32_t base) {
    const uint32_t bit0 = (uint32_t)((int32_t)(crc << 1) >> 31), bit1 = (uint32_t)((int32_t)crc >> 31);
    uint32_t x = and_xor(bit0, kTab1 & 0x3fffffffu, crc);
    x = and_xor(bit1, kTab2 & 0x3fffffffu, x);
    return and_xor(base, 3u, __builtin_amdgcn_alignbit(x, x, 30));
}
__device__ __forceinline__ uint32_t crc32_word(uint32_t crc, uint32_t word) {
    for (int i = 0; i < 16; ++i) {
        crc = crc2(crc, word & 3u);
        word >>= 2;
    }
    return crc;
}

__device__ __forceinline__ float lane_f(float x, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane));
}
__device__ __forceinline__ uint32_t lane_u(uint32_t x, int lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)x, lane);
}
// Maximum over the wave, every lane active.  The rotate-and-max steps are single DPP
// instructions written out by hand (the compiler's lowering of fmaxf after a DPP move
// adds a move and a canonicalisation per step); each needs two idle cycles after the
// instruction that wrote its source.  The last two steps carry the row maxima across
// rows, so lane 63 ends up with the result.  The inputs are never NaN.
__device__ __forceinline__ float wave_max(float x) {
    asm volatile(
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(x));
    return lane_f(x, 63);
}
// What a lane will store for its three candidates once their ranks are known, worked out in the
// wait states of the wave maximum: a wave that is alone on its SIMD pays a full issue slot for every
// s_nop, so the two idle cycles each rotate-and-max step needs after its source was written are filled
// with instructions that had to be issued anyway.
//   h0 = crc2(hash, b0), h1 = crc2(hash, b0 + 1) = h0 ^ kTab1   (b0 is even)
//   info0 = (st4 & state_mask) | b0 | from, info1 = info0 | 1, infos = state | from | stay bit
//   cs = the stay's score after the merges, rests = cs minus its guide term (the steps' scores are still on their way from LDS)
// The lane maximum of x0, x1 and the stay's (one v_max3) opens the block; the read of lane 63, where the six steps leave the
// wave's maximum, wants one instruction between itself and the last of them, and the vector unit two before it uses what was read.
// The first two cuts come out of it as well, lo = best - log_cut (-FLT_MAX at least), cut = (lo + best) / 2 with the halves of both bounds: behind
// inline assembly whose results it reads at once the compiler idles an instruction.
struct NextRecords {
    uint32_t h0, h1, info0, info1, infos;
    float rest0, rest1, rests;
};
struct Cuts {
    float lo, half_lo, half_hi, cut;
};
__device__ __forceinline__ Cuts wave_max_beside_records(float x0, float x1, float stay_or_fold, NextRecords &n, float &cs, uint32_t hash,
                                                        uint32_t b0, uint32_t state, uint32_t from_stay, uint32_t st4,
                                                        uint32_t state_mask, uint32_t from, uint64_t step_wins, float lowest, float gs, float log_cut) {
    uint32_t t0, t1, best;
    float x;
    Cuts c;
    asm volatile(
        "v_max3_f32 %[x], %[x0], %[x1], %[x2]\n\t"
        "v_xor_b32 %[t0], %[hash], %[b0]\n\t"
        "v_and_or_b32 %[i0], %[st4], %[mask], %[b0]\n\t"
        "v_max_f32_dpp %[x], %[x], %[x] row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_bfe_i32 %[t1], %[t0], 1, 1\n\t"
        "v_bfe_i32 %[t0], %[t0], 0, 1\n\t"
        "v_max_f32_dpp %[x], %[x], %[x] row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_and_b32 %[t1], %[tab2], %[t1]\n\t"
        "v_and_b32 %[t0], %[tab1], %[t0]\n\t"
        "v_max_f32_dpp %[x], %[x], %[x] row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_xor_b32 %[t0], %[t0], %[t1]\n\t"
        "v_lshrrev_b32 %[t1], 2, %[hash]\n\t"
        "v_max_f32_dpp %[x], %[x], %[x] row_ror:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_xor_b32 %[h0], %[t0], %[t1]\n\t"
        "v_or_b32 %[i0], %[i0], %[from]\n\t"
        "v_max_f32_dpp %[x], %[x], %[x] row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"
        "v_xor_b32 %[h1], %[tab1], %[h0]\n\t"
        "v_or_b32 %[i1], 1, %[i0]\n\t"
        "v_max_f32_dpp %[x], %[x], %[x] row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"
        "v_cndmask_b32 %[cs], %[x2], %[lowest], %[wins]\n\t"
        "v_readlane_b32 %[best], %[x], 63\n\t"
        "v_or_b32 %[is], %[state], %[fromstay]\n\t"
        "v_sub_f32 %[rs], %[cs], %[gs]\n\t"
        "v_sub_f32 %[lo], %[best], %[logcut]\n\t"
        "v_mul_f32 %[hh], %[best], 0.5\n\t"
        "v_max_f32 %[lo], %[lowest], %[lo]\n\t"
        "v_mul_f32 %[hl], 0.5, %[lo]\n\t"
        "v_add_f32 %[cut], %[hl], %[hh]"
        : [lo] "=&v"(c.lo), [hl] "=&v"(c.half_lo), [hh] "=&v"(c.half_hi), [cut] "=&v"(c.cut), [x] "=&v"(x), [best] "=&s"(best), [t0] "=&v"(t0), [t1] "=&v"(t1), [h0] "=&v"(n.h0), [h1] "=&v"(n.h1),
          [i0] "=&v"(n.info0), [i1] "=&v"(n.info1), [is] "=&v"(n.infos), [rs] "=&v"(n.rests), [cs] "=&v"(cs)
        : [hash] "v"(hash), [b0] "v"(b0), [tab1] "s"(kTab1), [tab2] "s"(kTab2), [st4] "v"(st4), [mask] "s"(state_mask),
          [from] "v"(from), [state] "v"(state), [fromstay] "v"(from_stay), [x0] "v"(x0), [x1] "v"(x1), [x2] "v"(stay_or_fold),
          [wins] "s"(step_wins), [lowest] "v"(lowest), [gs] "v"(gs), [logcut] "v"(log_cut));
    return c;
}
__device__ __forceinline__ int wave_sum_i(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x124, 0xF, 0xF, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x122, 0xF, 0xF, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x121, 0xF, 0xF, true);
    return __builtin_amdgcn_readlane(x, 0) + __builtin_amdgcn_readlane(x, 16) +
           __builtin_amdgcn_readlane(x, 32) + __builtin_amdgcn_readlane(x, 48);
}
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// per lane: yes where the lane's bit of a wave-wide mask is set, no elsewhere; the mask goes into
// the select as it is (a comparison result the wave already holds in scalar registers)
__device__ __forceinline__ int pick_by_bit(uint64_t mask, int yes, int no) {
    return __builtin_amdgcn_inverse_ballot_w64(mask) ? yes : no;
}
__device__ __forceinline__ float pick_by_bit(uint64_t mask, float yes, float no) {
    return __builtin_amdgcn_inverse_ballot_w64(mask) ? yes : no;
}
// x + (the lane's bit of mask), one add-with-carry
__device__ __forceinline__ int add_bit_of(int x, uint64_t mask) {
    int r;
    uint64_t carry;
    asm("v_addc_co_u32_e64 %0, %1, %2, 0, %3" : "=v"(r), "=&s"(carry) : "v"(x), "s"(mask));
    return r;
}
__device__ __forceinline__ int popc64(uint64_t x) { return __builtin_popcountll(x); }
// LDS accesses through a 32-bit LDS address
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#define LDS_AS __attribute__((address_space(3)))
__device__ __forceinline__ f32x2 lds_load_f2(uint32_t at) { return *(const LDS_AS f32x2 *)(uintptr_t)at; }

__device__ __forceinline__ float lds_load_f(uint32_t at) { return *(const LDS_AS float *)(uintptr_t)at; }
__device__ __forceinline__ void lds_store_f2(uint32_t at, float a, float b) {
    f32x2 v;
    v.x = a;
    v.y = b;
    *(LDS_AS f32x2 *)(uintptr_t)at = v;
}
__device__ __forceinline__ void lds_store_f(uint32_t at, float a) { *(LDS_AS float *)(uintptr_t)at = a; }
// (x & bits) | base in one instruction
__device__ __forceinline__ uint32_t and_or(uint32_t x, uint32_t bits, uint32_t base) { return (x & bits) | base; }
// The LDS address of an object as a plain number that the compiler keeps in a register: where it can see the constant, it works
// the address out again at every use and tests it for the null of a flat pointer.
__device__ __forceinline__ uint32_t lds_address(const void *p) {
    uint32_t at = (uint32_t)(uintptr_t)(const LDS_AS uint32_t *)p;
    asm volatile("" : "+v"(at));
    return at;
}

// The lane, worked out where it is wanted: for places off the search's way, so that no register holds it through the search (the
// merged kernel of large batches has 96).
__device__ __forceinline__ int lane_now() {
    uint32_t none = 0;
    asm volatile("" : "+v"(none));  // or the compiler takes it from elsewhere after all
    return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, none));
}

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Hand-over of LDS rows between the waves of a workgroup.  The fences name the
// local address space only: they wait for outstanding LDS operations, not for the
// global loads and stores each wave keeps in flight.
__device__ __forceinline__ void publish(int *flag, int value) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __hip_atomic_store(flag, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ int observe(int *flag) {
    const int v = __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    return v;
}

// log(e^x + e^y) with the correction evaluated in double and dropped for gaps >= 17
// (reference src/beam_search.c:43-47).  The correction log(1 + e^-gap) comes from a
// piecewise polynomial kept in LDS: a handful of dependent FMAs instead of an exp
// followed by a log, which matters because every merge sits on the search's serial path.
__device__ __forceinline__ float log_sum_exp(float x, float y, const double *table) {
    const float gap = fabsf(x - y);
    const float top = x > y ? x : y;
    int cell = (int)(gap * 4.0f);
    cell = cell < OFK_LSE_CELLS - 1 ? cell : OFK_LSE_CELLS - 1;
    const double *c = table + cell * OFK_LSE_COEFS;
    const double s = __builtin_fma((double)gap, 8.0, -(double)(2 * cell + 1));  // (gap - centre of the cell) * 8, exactly
    double p = c[8];
#pragma unroll
    for (int k = 7; k >= 0; --k) p = __builtin_fma(p, s, c[k]);
    const double corr = gap < 17.0f ? p : 0.0;
    return (float)((double)top + corr);
}

// The same fold from the hardware's fp32 exp2/log2, with the verdict whether its rounded result is
// certain to be the one above.  top + l2 * ln2f (one fused multiply-add, l2 = log2(1 + exp2(-gap c)))
// differs from top + log(1 + e^-gap) by at most, in units of 2^-24:
//   0.72  v_exp_f32 (largest relative error over every input in [-160, 0]: 1.423), times e/(1+e) <= 1/2
//   0.45  the argument of exp2: gap c rounded to fp32 with c = fl(log2 e): 7.3e-8 gap e^-gap <= 2.7e-8
//   1.00  1 + e rounded to fp32
//   1.39  v_log_f32 on [1, 2] (largest absolute error over every input: 1.0 below 2, 2.0 at 2), times ln 2
//   0.08  ln2f against ln 2, the rounding of the residual
// together 3.64; the bound used is 4.0.  (The two hardware figures are measured on the device at
// hand, over every fp32 input of their ranges, by tests/test_gpu_hw_math.py.)  The result is settled when the distance from the
// unrounded sum to the nearer rounding boundary of the result exceeds that bound (the residual of
// the fused multiply-add, taken exactly with a second one).  Half an ulp is 2^-24 of the binade of the
// float below r in magnitude (r (1 - 2^-24), rounded: for a power of two it lies in the binade below, where its nearer
// boundary is; every other float stays in its own); results below 2^-102 in magnitude never count as settled.
struct FoldValue {
    float value, top, l2;
};
__device__ __forceinline__ FoldValue log_sum_exp_value(float x, float y) {
    const float gap = fabsf(x - y);
    FoldValue f;
    f.top = x > y ? x : y;
    const float e = __builtin_amdgcn_exp2f(gap * -1.44269504088896340736f);
    f.l2 = __builtin_amdgcn_logf(1.0f + e);
    f.value = __builtin_fmaf(f.l2, 0.69314718055994530942f, f.top);
    return f;
}
__device__ __forceinline__ bool log_sum_exp_settled(FoldValue f) {
    const float rho = __builtin_fmaf(f.l2, 0.69314718055994530942f, -(f.value - f.top));
    const float binade = __uint_as_float(__float_as_uint(f.value * 0x1.fffffep-1f) & 0x7f800000u);
    return __builtin_fmaf(binade, 0x1p-24f, -fabsf(rho)) > 4.0f * 0x1p-24f;
}

__device__ __forceinline__ uint32_t float_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return u ^ ((u >> 31) ? 0xFFFFFFFFu : 0x80000000u);
}
__device__ __forceinline__ float key_float(uint32_t k) {
    return __uint_as_float(k ^ ((k >> 31) ? 0x80000000u : 0xFFFFFFFFu));
}

template <int N, int FIRST = 0, typename F>
__device__ __forceinline__ void static_for_upwards(F &&f) {
    if constexpr (FIRST < N) {
        f(std::integral_constant<int, FIRST>{});
        static_for_upwards<N, FIRST + 1>(f);
    }
}

template <int BYTES>
struct Vec;
template <>
struct Vec<4> { typedef uint32_t type; };
template <>
struct Vec<16> { typedef uint32_t type __attribute__((ext_vector_type(4))); };

// one wave's share of a row of ROW_BYTES bytes: lane l owns vectors (i*64 + l).  Rows of 256
// bytes are split into 4-byte vectors, one per lane; all others into 16-byte
// vectors, of which the last round may cover only the lower lanes (rows of five-column scores
// are 2560 or 10240 bytes).
template <int ROW_BYTES>
struct RowRegs {
    static constexpr int kVec = ROW_BYTES == 256 ? 4 : 16;
    static constexpr int kVecs = ROW_BYTES / kVec;
    static constexpr int kCnt = (kVecs + 63) / 64;
    static_assert(ROW_BYTES % kVec == 0, "rows are whole vectors");
    typedef typename Vec<kVec>::type V;
    V v[kCnt];
    static __device__ __forceinline__ bool mine(int i, int lane) { return (i + 1) * 64 <= kVecs || i * 64 + lane < kVecs; }
    __device__ __forceinline__ void load(const char *row, int lane) {
#pragma unroll
        for (int i = 0; i < kCnt; ++i)
            if (mine(i, lane)) v[i] = *reinterpret_cast<const V *>(row + (size_t)(i * 64 + lane) * kVec);
    }
    __device__ __forceinline__ void store(char *row, int lane) const {
#pragma unroll
        for (int i = 0; i < kCnt; ++i)
            if (mine(i, lane)) *reinterpret_cast<V *>(row + (size_t)(i * 64 + lane) * kVec) = v[i];
    }
};

// A row of scores on its way to a ring slot that only the search reads: four planes of S values, one for every dropped base, a blank
// column left out.  An element's four steps then lie side by side at 8 * state, whatever the layout of the caller's scores: one address
// instruction and one LDS read instead of four and two.  A lane owns pairs of neighbouring states, COLS words each.
template <int S, int COLS>
struct PlaneRow {
    static constexpr int kPairs = S / 2, kCnt = (kPairs + 63) / 64;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));
    u32x4 w[kCnt];
    uint32_t w4[COLS == 5 ? kCnt : 1];  // the fifth word
    static __device__ __forceinline__ bool mine(int i, int lane) { return (i + 1) * 64 <= kPairs || i * 64 + lane < kPairs; }
    __device__ __forceinline__ void load(const char *row, int lane) {
#pragma unroll
        for (int i = 0; i < kCnt; ++i)
            if (mine(i, lane)) {
                const uint32_t *p = reinterpret_cast<const uint32_t *>(row) + COLS * (i * 64 + lane);
                w[i] = *reinterpret_cast<const u32x4 *>(p);
                if constexpr (COLS == 5) w4[i] = p[4];
            }
    }
    static __device__ __forceinline__ uint32_t low_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
    static __device__ __forceinline__ uint32_t high_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
    static __device__ __forceinline__ uint32_t high_low(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040302u); }
    static __device__ __forceinline__ uint32_t low_high(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060100u); }
    __device__ __forceinline__ void store(char *row, int lane) const {
#pragma unroll
        for (int i = 0; i < kCnt; ++i)
            if (mine(i, lane)) {
                uint32_t *p = reinterpret_cast<uint32_t *>(row) + i * 64 + lane;
                if constexpr (COLS == 4) {  // t0 t1 | t2 t3 of one state, then of the next
                    p[0 * kPairs] = low_halves(w[i].x, w[i].z);
                    p[1 * kPairs] = high_halves(w[i].x, w[i].z);
                    p[2 * kPairs] = low_halves(w[i].y, w[i].w);
                    p[3 * kPairs] = high_halves(w[i].y, w[i].w);
                } else {  // blank t0 | t1 t2 | t3 blank | t0 t1 | t2 t3
                    p[0 * kPairs] = high_low(w[i].x, w[i].w);
                    p[1 * kPairs] = low_high(w[i].y, w[i].w);
                    p[2 * kPairs] = high_low(w[i].y, w4[i]);
                    p[3 * kPairs] = low_high(w[i].z, w4[i]);
                }
            }
    }
};

// FWD is the number of waves per chunk that run the forward recursion beside the search (0: the search alone).
template <int S, int CPG, int FWD>
struct BeamCfg {
    static constexpr int kBits = S == 64 ? 6 : S == 256 ? 8 : 10;
    // two waves of recursion at 256 states: the LDS (75 and 78 KB) and the registers of two workgroups fit a compute unit (see beam_kernel for
    // what comes of it)
    static constexpr bool kDense = FWD == 2;
    // LDS ring depth, which is also how many time steps of the search are written out one after another.  Four, but for two chunks of
    // 1024 states to a unit that they share with the forward sweep, and where two workgroups are to fit one.
    static constexpr int kLdsRows = kDense || (S >= 1024 && CPG > 1) ? 3 : 4;
    static constexpr int kHandBack = FWD == 0 && kLdsRows == 4 ? 2 : 1;  // rows the search asks for and gives back at a time
    static constexpr int kRegRows = S >= 1024 ? (FWD == 0 ? 3 : 2) : (kDense ? 3 : 6);  // rows in flight in registers (2, 3 or 6)
};

// one beam element as handed from one time step to the next: three words of a 16-byte slot, written
// by one 96-bit store (an LDS store costs by its width, whatever the number of enabled lanes)
struct __attribute__((aligned(16))) Elem {
    uint32_t hash;
    float rest;     // candidate score minus the guide term of its state: what the next time step starts from
                    // (at the last time step: the candidate score itself, which picks the best survivor)
    uint32_t info;  // state | prev << 10 | stay << 15: the 16-bit slot the traceback reads
    uint32_t pad;
};

struct BeamShared {
    Elem elem[kW + 64];           // slots 0 .. kW-1; entry kW + lane is lane's dump slot for candidates that are not kept
    float stay_score[kW];         // only used by the serial replay of merges
    uint32_t claim[4 * kW + 64];  // only used when the hash index was not conclusive: who claimed step candidate 4j+b
    int ready, consumed;          // rows stored by the loader wave, rows the search wave is done with (with FWD > 0 in FwdLds)
    int searched, mapped;         // the search has ended; waves of the traceback that have their blocks' maps in LDS
};

// LDS of one chunk.  Score rows are kept in planes for the search alone; where the recursion reads them too, as the caller lays them
// out: COLS = 4 transitions per state, or 5 with an unused blank first.  So are rows of 1024 states, 32 stores of a word for the loader
// in planes: 37 chunks, T = 833 0.500 ms, as they are 0.477.
template <int S, int COLS, int FWD>
struct ScoreRow {
    static constexpr bool kPlanes = FWD == 0 && S < 1024;
    static constexpr int kHalves = (kPlanes ? 4 : COLS) * S;
    typedef typename std::conditional<kPlanes, PlaneRow<S, COLS>, RowRegs<2 * COLS * S>>::type Regs;
};
template <int S, int CPG, int COLS, int FWD>
struct __attribute__((aligned(16))) BeamRing {
    _Float16 row_s[BeamCfg<S, CPG, FWD>::kLdsRows][ScoreRow<S, COLS, FWD>::kHalves];
    float row_b[BeamCfg<S, CPG, FWD>::kLdsRows][S];
};
// Hash index of one chunk: 2^kBits buckets of one word.  Hash bits 2 .. kBits + 1 are the bucket's byte address; in the entry
// their place is free for the element's slot (bits 4 .. 8) and the generation (bits 2, 3 and 9 .. kBits + 1), so that one word
// holds all that a look-up has to compare, and what is left of the comparison with the entry looked for is the partner's slot.
// (Two words an entry, hash and generation << 5 | slot, took half the buckets, two more comparisons and 12 more LDS cycles a step.)
// Low two bits of the generation: the ring slot of the time step; the rest counts ring rounds from 1, and when it is
// used up the search's wave clears the table (about 6 cycles a step).  With w live elements two of them share a bucket in about
// w^2 / (2 * buckets) of the time steps: with 25 to 32 of them one step in 8 to 13 of 4096 buckets, in 16 to 26 of 8192, in 32 to 52 of 16384.
template <int S, int CPG, int FWD>
struct BeamIdx {
    static constexpr bool kLone = CPG == 1 && FWD == 0;  // a compute unit's LDS for one chunk
    static constexpr int kBits = kLone ? 14 : (BeamCfg<S, CPG, FWD>::kDense || CPG > 2 || (S >= 1024 && FWD == 0)) ? 12 : 13;
    static constexpr int kBuckets = 1 << kBits;
    static constexpr uint32_t kAddress = (uint32_t)(kBuckets - 1) << 2;  // hash bits that address a bucket
    static constexpr uint32_t kSlot = 31u << 4;
    static constexpr uint32_t kRound = 1u << 9, kRoundEnd = 1u << (kBits + 2);
    // Waves that trace a chunk's path back, each with a buffer of 8 KB in the index: the search's, the loader's and, of a lone chunk, the
    // two that were there for the set-up, or two of the recursion's.  The maps they exchange, 16 KB, lie behind the buffers where there is
    // room, and apart in the merged kernels of four and eight waves: 148 KB of LDS a workgroup of 256 states (five columns 152; 115 and 119
    // without them), 127 (136) of 1024 states.  The 12 to 33 KB that are left of a unit take a workgroup of another decode's backward sweep,
    // 6 or 15 KB, but of its sequence stage, 13 bytes a step, only with shorter chunks.  An index of 16 KB has two buffers and no maps: one wave.
    static constexpr int kTeam = kLone || FWD >= 4 ? 4 : kBits == 13 ? 2 : 1;
    static constexpr bool kMapsApart = FWD >= 4;
};
// What the forward recursion and the posterior of a chunk share.
constexpr int kVecRows = 4;  // two would do (see beam_kernel); four let the posterior lag (1024 chunks of 256 states: 2.66 ms against 2.78)
template <int S, int FWD>
struct __attribute__((aligned(16))) FwdLds {
    // Progress of the chunk's waves, side by side so that one LDS read of a wave, a lane to a counter, sees all of it: rows of the state
    // vector that each wave of the recursion has written, rows that the posterior's wave has read, ring rows ready and consumed.
    static constexpr int kTaken = FWD, kReady = FWD + 1, kConsumed = FWD + 2;
    static constexpr int kCounters = FWD + 3 <= 8 ? 8 : 16;
    int progress[kCounters];
    __attribute__((aligned(16))) float vec[kVecRows][S];  // row t in vec[t % kVecRows]
    float tier_lanes[64 * FWD];
};
template <int S>
struct FwdLds<S, 0> {};
struct FwdTables {
    ofa::LogCell centred[ofa::kLogCentredCells];
};
struct NoTables {};
struct TraceMaps {
    uint32_t map[(OFK_MAX_T + kTraceRows - 1) / kTraceRows][64];
};
template <int S, int CPG, int COLS, int FWD>
struct __attribute__((aligned(16))) BeamLds {
    BeamRing<S, CPG, COLS, FWD> ring;
    BeamShared sh;
    uint32_t idx_dump[64];  // where a dead lane files its leftovers instead of a bucket of the index
    FwdLds<S, FWD> fwd;
    typename std::conditional<BeamIdx<S, CPG, FWD>::kMapsApart, TraceMaps, NoTables>::type trace;
};
// scores of the step candidates 4i+b while stays merge into them, aligned so that a candidate's address is put together by `or`;
// then a slot for every lane whose stay has no partner to write to
struct __attribute__((aligned(512))) BeamCand {
    float step[4 * kW];
    float dump[64];
};
// All LDS of a workgroup, one object: the index tables come first and each is aligned to its
// size, so that a bucket's address is (hash & bits) | table, one instruction.
template <int S, int CPG, int COLS, int FWD>
struct __attribute__((aligned(16))) BeamGroupLds {
    uint32_t idx[CPG][BeamIdx<S, CPG, FWD>::kBuckets];
    BeamCand cand[CPG];
    BeamLds<S, CPG, COLS, FWD> chunk[CPG];
    double lse[OFK_LSE_DOUBLES];  // coefficient table of the folds, one copy per workgroup
    typename std::conditional<FWD == 0, NoTables, FwdTables>::type logs;
};

// The scores of one lane's states for one step of the recursion, read from a row in LDS: fp16 pairs in
// 32-bit words.  Five-column rows are read in aligned words (a state's transitions start at a word or in the
// middle of one, by its parity) and shifted into place.  Addresses are plain numbers: where the compiler sees the object behind them
// it puts the distance from LDS address 0 into every one anew, past what an instruction's offset holds.
template <int SPL, int COLS>
struct LdsRow {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    uint32_t w[2 * SPL];
    static __device__ __forceinline__ uint32_t word(uint32_t at) { return *(const LDS_AS uint32_t *)(uintptr_t)at; }
    static __device__ __forceinline__ uint32_t first(int s0) {  // bytes from the row's start; s0 is even where a lane has two states or more
        return COLS == 4 ? 8u * (uint32_t)s0 : SPL == 1 ? ((5u * (uint32_t)s0 + 1u) >> 1) << 2 : 10u * (uint32_t)s0;
    }
    __device__ __forceinline__ void load(uint32_t at, int s0) {
        if constexpr (COLS == 4) {
            if constexpr (SPL == 1) {
                const u32x2 x = *(const LDS_AS u32x2 *)(uintptr_t)at;
                w[0] = x.x; w[1] = x.y;
            } else {
#pragma unroll
                for (int i = 0; i < SPL / 2; ++i) {
                    const u32x4 x = *(const LDS_AS u32x4 *)(uintptr_t)(at + 16u * (uint32_t)i);
                    w[4 * i] = x.x; w[4 * i + 1] = x.y; w[4 * i + 2] = x.z; w[4 * i + 3] = x.w;
                }
            }
        } else if constexpr (SPL == 1) {
            const uint32_t a = word(at), b = word(at + 4), c = word(at + (s0 & 1 ? 4u : 8u)), by = s0 & 1 ? 0u : 16u;
            w[0] = __builtin_amdgcn_alignbit(b, a, by);
            w[1] = __builtin_amdgcn_alignbit(c, b, by);
        } else {
#pragma unroll
            for (int i = 0; i < SPL / 2; ++i) {
                const uint32_t p = at + 20u * (uint32_t)i, a = word(p), b = word(p + 4), c = word(p + 8);
                w[4 * i] = __builtin_amdgcn_alignbit(b, a, 16);
                w[4 * i + 1] = __builtin_amdgcn_alignbit(c, b, 16);
                w[4 * i + 2] = word(p + 12);
                w[4 * i + 3] = word(p + 16);
            }
        }
    }
};


// CPG chunks per workgroup.  The waves of a group are dealt round over the four SIMDs of
// its compute unit (wave k and wave k + 4 share one), while two-wave groups were measured
// to pile onto two SIMDs.  With two chunks a group is four waves, two of them searching;
// with four chunks it is eight waves and every SIMD holds exactly one search wave and one
// loader, which is what a batch of more than two chunks per compute unit needs.
//
// FWD > 0: the forward recursion and the posterior of the same chunks run in the same workgroup and read the
// rows the loader has put into LDS, so that scores and bwd cross HBM once for both.  As two kernels side by
// side they were bound by that traffic at large batches (1024 chunks of 256 states with five columns: 13.9 GB
// in 2.98 ms, what a copy reaches; 256 of 1024 states the same in 2.84); here 7.9 GB take 2.54 and 1.74 ms,
// bound by the chain of a step and by its instructions.
//   search | posterior | FWD waves of recursion | loader
// There is no barrier after the set-up: the waves of a chunk hand rows over through counters in LDS.  A wave of
// the recursion writes its part of row t + 1 of the state vector and then its counter (a wave's LDS operations
// are carried out in order), and starts on a row once all counters of its chunk have reached it.  Row t + 1
// takes the place of row t + 1 - kVecRows, which the other waves of the recursion have read if they have
// published row t (kVecRows >= 2), and the posterior's wave if it says so.  The loader refills a ring slot when
// search, recursion and posterior are all past it.  A wave only waits for rows that the others can produce
// without it: loader row t for consumers past row t - LR, recursion step t for row t of the ring and of the vector
// and the posterior past row t + 1 - kVecRows, the posterior's row t for row t of the vector.  So all waits end.
// Priorities: search 3, recursion 2 (3 in the second tier), posterior 1; with the recursion at 0 it takes 3 to 5 %
// more at large batches, with the search below the recursion 256 states lose 0.2 ms at 512 chunks.
//
// FWD: one state per lane (4 waves) with one workgroup of two chunks on a compute unit.  Above 512 chunks of 256
// states two workgroups were to share a unit (78 KB of LDS, 96 registers per lane): two states per lane and smaller
// rings.  They do not: by the counters 2.2 of the 5 waves launched for a SIMD are resident, which is one workgroup a unit at a time, and the vector
// ALUs are busy 0.61 of 2.14 ms (1024 chunks).  A workgroup's ten waves lie 3 + 3 + 2 + 2 on SIMDs that hold five each, so a second one
// fits only with its larger shares on the other two.  1024 states: two per lane, one chunk per workgroup (four per lane: 2.15 ms against 1.74 at 256 chunks).
template <int S, int CPG, int COLS, int FWD>
constexpr int kBeamThreads = BeamIdx<S, CPG, FWD>::kLone ? 256 : 64 * CPG * (FWD == 0 ? 2 : FWD + 3);  // a lone chunk: two waves more for the set-up
template <int S, int CPG, int COLS, int FWD>
__global__ __launch_bounds__((kBeamThreads<S, CPG, COLS, FWD>), (BeamCfg<S, CPG, FWD>::kDense ? 5 : 1)) void beam_kernel(const _Float16 *__restrict__ scores,
                                                   const float *__restrict__ bwd, float *__restrict__ post,
                                                   ofk_beam_slot_t *__restrict__ beam,
                                                   int32_t *__restrict__ states, uint8_t *__restrict__ moves,
                                                   int T, int N, float log_cut, float stay, int flags,
                                                   const double *__restrict__ lse_table, LogSeries series) {
    using Cfg = BeamCfg<S, CPG, FWD>;
    using Idx = BeamIdx<S, CPG, FWD>;
    constexpr int BITS = Cfg::kBits;
    constexpr int LR = Cfg::kLdsRows;
    constexpr int RR = Cfg::kRegRows;

    constexpr int kGroupChunks = CPG;
    // bytes, so that the size is not rounded up to the alignment the index tables want
    __shared__ __attribute__((aligned(Idx::kBuckets * 4))) unsigned char
        lds_bytes[sizeof(BeamGroupLds<S, CPG, COLS, FWD>)];
    auto &all = *reinterpret_cast<BeamGroupLds<S, CPG, COLS, FWD> *>(lds_bytes);
    auto &lds = all.chunk;
    auto &lse = all.lse;

    // waves 0 .. kGroupChunks-1 search, the last kGroupChunks load; between them those of the forward sweep
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    constexpr int kFirstFwd = 2 * kGroupChunks, kFirstLoader = kGroupChunks * (FWD == 0 ? 1 : FWD + 2);
    const bool recursion = FWD > 0 && wave >= kFirstFwd && wave < kFirstLoader;
    const int member = recursion ? (wave - kFirstFwd) / (FWD > 0 ? FWD : 1) : wave % kGroupChunks;
    const int n = blockIdx.x * kGroupChunks + member;
    const int lane = lane_now();
    auto &row_s = lds[member].ring.row_s;
    auto &row_b = lds[member].ring.row_b;
    BeamShared &sh = lds[member].sh;
    const size_t row_stride = (size_t)N * COLS * S;
    const _Float16 *sc_n = scores + (size_t)n * COLS * S;
    const float *bw_n = bwd + (size_t)n * (size_t)(T + 1) * S;

    int *ready, *consumed;  // rows stored by the loader wave, rows the search wave is done with
    if constexpr (FWD == 0) {
        ready = &sh.ready;
        consumed = &sh.consumed;
    } else {
        ready = &lds[member].fwd.progress[FwdLds<S, FWD>::kReady];
        consumed = &lds[member].fwd.progress[FwdLds<S, FWD>::kConsumed];
    }
    if (wave < kGroupChunks && lane == 0) {
        *ready = 0;
        *consumed = 0;
        sh.searched = 0;
        sh.mapped = 0;
        if constexpr (FWD > 0)
            for (int x = 0; x < FwdLds<S, FWD>::kCounters; ++x) lds[member].fwd.progress[x] = 0;
    }
    if constexpr (FWD > 0) fill_log_tables<OFK_SCAN_TWO_TIER, kBeamThreads<S, CPG, COLS, FWD>>(nullptr, all.logs.centred);
    for (int x = (int)threadIdx.x; x < OFK_LSE_DOUBLES; x += kBeamThreads<S, CPG, COLS, FWD>) lse[x] = lse_table[x];
    // the hash index starts empty: no entry may look like one of a real generation (their rounds start at 1)
    for (int x = (int)threadIdx.x; x < kGroupChunks * Idx::kBuckets / 4; x += kBeamThreads<S, CPG, COLS, FWD>)
        reinterpret_cast<uint4 *>(&all.idx[0][0])[x] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    if (n >= N) return;  // odd batch: the last group has one chunk
    ofk_beam_slot_t *const bv = beam + (size_t)n * (size_t)(T + 1) * kW;

    static_assert((FWD & (FWD - 1)) == 0 && FWD <= 8, "a lane reads one counter");
    constexpr int kTeam = Idx::kTeam;
    int mate = 0;  // of those that trace this chunk's path back: the search's wave is the first
    if constexpr (FWD > 0) {
        typedef FwdLds<S, FWD> Fwd;
        Fwd &fw = lds[member].fwd;
        // The counter of the lane, no wait included: what is read after it, in the order of the program, is from after it, because a
        // wave's LDS operations are carried out in order (as are those of the wave that wrote rows first and its counter then).
        auto progress = [&](int counter) {
            const int rows = __hip_atomic_load(&fw.progress[counter], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            wave_fence();
            return rows;
        };
        if (recursion) {
            // ---- one wave of the forward recursion (same arithmetic as fwd_post_roles_kernel) ----
            const int lane = lane_now();
            constexpr int SPL = S / (64 * FWD), Q = S / 4;
            const int w = (wave - kFirstFwd) % FWD;
            const int s0 = SPL * (64 * w + lane), q = s0 >> 2;
            const LogArgs logtab{nullptr, all.logs.centred, series.c, series.e, fw.tier_lanes + 64 * w, 3, 2};
            __builtin_amdgcn_s_setprio(2);
            float f[SPL];
#pragma unroll
            for (int k = 0; k < SPL; ++k) f[k] = 0.f;
            // what the lane reads and writes of a row: its scores in the ring, its predecessors and its own places in the vector
            const uint32_t vec_at = lds_address(&fw.vec[0][q]), own_at = lds_address(&fw.vec[0][s0]);
            uint32_t row_at = lds_address(&row_s[0][0]) + LdsRow<SPL, COLS>::first(s0);
            asm volatile("" : "+v"(row_at));
            uint32_t slot = 0;  // bytes
            const uint32_t mark_at = lds_address(&fw.progress[w]);
            auto vec_row = [](int t) { return (uint32_t)(t % kVecRows) * (uint32_t)(4 * S); };
            auto write_row = [&](int t) {
                const uint32_t at = own_at + vec_row(t);
                if constexpr (SPL == 1) {
                    lds_store_f(at, f[0]);
                } else {
#pragma unroll
                    for (int k = 0; k < SPL; k += 2) lds_store_f2(at + 4u * (uint32_t)k, f[k], f[k + 1]);
                }
            };
            auto publish_row = [&](int t) {
                wave_fence();
                __hip_atomic_store((LDS_AS int *)(uintptr_t)mark_at, t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            };
            write_row(0);
            publish_row(0);
            // Step t needs row t of the vector from every wave, row t of the ring, and rows 0 .. t + 1 - kVecRows read by the posterior:
            // row t + 1 goes where row t + 1 - kVecRows was.
            const int counter = lane & (Fwd::kCounters - 1);
            const int wanted = counter < FWD || counter == Fwd::kReady ? 1 : counter == Fwd::kTaken ? 2 - kVecRows : -(1 << 30);
            for (int t = 0; t < T; ++t) {
                // One look at all of that.  (The ring's counter, the posterior's and the other waves' polled one after another: 512 chunks
                // of 256 states 1.041 | 1.008 ms, with five columns 1.060 | 1.036, 1024 of them 2.36 | 2.31.  The rows read together
                // with the counters, again if it was too early: 1.037, 1.077, 2.28; 256 of 1024 states 1.76 instead of 1.68, and the
                // clock lower for all that follows.)
                while (ballot(progress(counter) < t + wanted) != 0) {}
                LdsRow<SPL, COLS> row;
                row.load(row_at + slot, s0);
                const uint32_t vec = vec_at + vec_row(t);
                const float p0 = lds_load_f(vec), p1 = lds_load_f(vec + 4 * Q), p2 = lds_load_f(vec + 8 * Q), p3 = lds_load_f(vec + 12 * Q);
                float v[SPL][5];
#pragma unroll
                for (int k = 0; k < SPL; ++k) {
                    v[k][0] = f[k] + stay;
                    v[k][1] = ::add_half<0>(row.w[2 * k], p0);
                    v[k][2] = ::add_half<1>(row.w[2 * k], p1);
                    v[k][3] = ::add_half<0>(row.w[2 * k + 1], p2);
                    v[k][4] = ::add_half<1>(row.w[2 * k + 1], p3);
                }
                slot = slot == (uint32_t)((LR - 1) * sizeof(row_s[0])) ? 0u : slot + (uint32_t)sizeof(row_s[0]);
                lse5_all<SPL, OFK_SCAN_TWO_TIER>(f, v, logtab, [&] { write_row(t + 1); }, [](bool) {});
                publish_row(t + 1);
            }
            if (kTeam <= 2 || w + 2 >= kTeam) return;
            mate = w + 2;
            __builtin_amdgcn_s_setprio(0);
        }
        if (wave >= kGroupChunks && wave < kFirstFwd) {
            // ---- posterior: softmax over the states of fwd[t] + bwd[t], t = 0 .. T ----
            const int lane = lane_now();
            __builtin_amdgcn_s_setprio(1);
            constexpr int G = S / 256;  // pieces of four states per lane
            static_assert(G >= 1, "a lane holds at least four states");
            float4 b[G];
            float top = -FLT_MAX;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                b[g] = *reinterpret_cast<const float4 *>(bw_n + 256 * g + 4 * lane);
                top = fmaxf(top, fmaxf(fmaxf(b[g].x, b[g].y), fmaxf(b[g].z, b[g].w)));
            }
            const float shift = group_max<64>(top) - 10.0f;  // as in fwd_post_kernel
            float *prow = post + (size_t)n * (size_t)(T + 1) * S + 4 * lane;
            int slot = 0;
            const int counter = lane & (Fwd::kCounters - 1);
            const int wanted = counter < FWD ? 1 : -(1 << 30);
            for (int t = 0; t <= T; ++t) {
                while (ballot(progress(counter) < t + wanted) != 0) __builtin_amdgcn_s_sleep(2);
                float4 e[G];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    e[g] = *reinterpret_cast<const float4 *>(&fw.vec[t % kVecRows][256 * g + 4 * lane]);
                    if (t > 0) b[g] = *reinterpret_cast<const float4 *>(&row_b[slot][256 * g + 4 * lane]);
                }
                if (t > 0) slot = slot + 1 == LR ? 0 : slot + 1;
                publish(&fw.progress[Fwd::kTaken], t + 1);
                float total = 0.f;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    e[g].x = __builtin_amdgcn_exp2f(((e[g].x + b[g].x) - shift) * kLog2e);
                    e[g].y = __builtin_amdgcn_exp2f(((e[g].y + b[g].y) - shift) * kLog2e);
                    e[g].z = __builtin_amdgcn_exp2f(((e[g].z + b[g].z) - shift) * kLog2e);
                    e[g].w = __builtin_amdgcn_exp2f(((e[g].w + b[g].w) - shift) * kLog2e);
                    total += (e[g].x + e[g].y) + (e[g].z + e[g].w);
                }
                const float inv = __builtin_amdgcn_rcpf(group_sum<64>(total));
#pragma unroll
                for (int g = 0; g < G; ++g)
                    *reinterpret_cast<float4 *>(prow + 256 * g) = make_float4(e[g].x * inv, e[g].y * inv, e[g].z * inv, e[g].w * inv);
                prow += S;
            }
            return;
        }
    }
    auto load_rows = [&]() __attribute__((always_inline)) {
        // ---- loader wave: row t = (scores[t], bwd[t+1]) into ring slot t % LR ----
        const int lane = lane_now();
        // The ring is spelled out as named registers (not an array indexed by a loop that
        // also contains the spin wait) so that every row stays in VGPRs.
        typedef typename ScoreRow<S, COLS, FWD>::Regs Scores;
        Scores s0, s1, s2, s3, s4, s5;
        RowRegs<4 * S> g0, g1, g2, g3, g4, g5;
        auto fetch = [&](Scores &rs, RowRegs<4 * S> &rb, int t) {
            if (t < T) {
                rs.load(reinterpret_cast<const char *>(sc_n + (size_t)t * row_stride), lane);
                rb.load(reinterpret_cast<const char *>(bw_n + (size_t)(t + 1) * S), lane);
            }
        };
        auto hand_over = [&](Scores &rs, RowRegs<4 * S> &rb, int t) {
            if (t < T) {
                // the ring is full most of the time (a search step takes about 1200 cycles): poll
                // seldom, the rows in registers and in the ring leave ample slack for waking up late
                if constexpr (FWD == 0) {
                    while (t - observe(consumed) >= LR) __builtin_amdgcn_s_sleep(8);
                } else {
                    // the recursion is done with row p of scores once it has published row p + 1 of its vector,
                    // the posterior with row p of bwd (bwd[p + 1]) once it has taken row p + 1
                    typedef FwdLds<S, FWD> Fwd;
                    const int counter = lane & (Fwd::kCounters - 1);
                    const int wanted = counter <= Fwd::kTaken ? 2 - LR : counter == Fwd::kConsumed ? 1 - LR : -(1 << 30);
                    while (t >= LR && ballot(observe(&lds[member].fwd.progress[counter]) < t + wanted) != 0) __builtin_amdgcn_s_sleep(2);
                }
                const int slot = t % LR;
                rs.store(reinterpret_cast<char *>(row_s[slot]), lane);
                rb.store(reinterpret_cast<char *>(row_b[slot]), lane);
                fetch(rs, rb, t + RR);
                publish(ready, t + 1);
            }
        };
        fetch(s0, g0, 0);
        fetch(s1, g1, 1);
        if constexpr (RR >= 3) fetch(s2, g2, 2);
        if constexpr (RR == 6) {
            fetch(s3, g3, 3);
            fetch(s4, g4, 4);
            fetch(s5, g5, 5);
        }
        for (int t0 = 0; t0 < T; t0 += RR) {
            hand_over(s0, g0, t0);
            hand_over(s1, g1, t0 + 1);
            if constexpr (RR >= 3) hand_over(s2, g2, t0 + 2);
            if constexpr (RR == 6) {
                hand_over(s3, g3, t0 + 3);
                hand_over(s4, g4, t0 + 4);
                hand_over(s5, g5, t0 + 5);
            }
        }
    };

    auto search = [&]() __attribute__((always_inline)) {
    // ---- search wave ----
    const int i = lane >> 1;  // lanes 2i and 2i+1 hold element i; candidate order is lane order
    const int h = lane & 1;
    typedef __attribute__((address_space(3))) uint32_t lds_u32;
    // LDS addresses of this chunk's index table (a multiple of its size) and of this lane's spare entry
    const uint32_t idx_base = lds_address(&all.idx[member][0]);
    const uint32_t idx_dump = lds_address(&lds[member].idx_dump[lane]);

    // seeding: the 32 best states of bwd[0] in ascending state order (src/beam_search.c:151-175)
    {
        constexpr int PER = S / 64;
        float v[PER];
        uint32_t key[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            v[j] = bw_n[j * 64 + lane];
            key[j] = float_key(v[j]);
        }
        uint32_t prefix = 0;  // largest K with #{key >= K} >= 32, i.e. the 32nd largest value
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t trial = prefix | (1u << bit);
            int c = 0;
#pragma unroll
            for (int j = 0; j < PER; ++j) c += key[j] >= trial ? 1 : 0;
            if (wave_sum_i(c) >= kW) prefix = trial;
        }
        const float thr = key_float(prefix);
        if (lane < kW) sh.elem[lane] = Elem{0u, 0.f, 0u, 0u};
        wave_fence();
        int taken = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const bool ok = v[j] >= thr;
            const uint64_t m = ballot(ok);
            const int rank = taken + popc64(m & (((uint64_t)1 << lane) - 1));
            if (ok && rank < kW) {
                const uint32_t s = (uint32_t)(j * 64 + lane);
                // flags bit 1 (tests): seeds that agree in their low four state bits share a hash
                const uint32_t hs = crc32_word(kSeed, (flags & 2) ? (s & 15u) : s);
                sh.elem[rank] = Elem{hs, 0.f, s, 0u};
            }
            taken += popc64(m);
        }
        wave_fence();
    }
    uint32_t hash, want, info;  // want: the hash of the sequence without its last base, what a partner's hash has to equal
    float score;
    {
        const Elem e = sh.elem[i];
        hash = e.hash;
        info = e.info;
        score = e.rest;
    }
    int state = (int)(info & 1023u);
    int w = kW;

    // The search is a chain of dependent short instructions; when it shares a SIMD with
    // throughput-bound waves (the forward scan runs at the same time) it should win the
    // issue arbitration.
    __builtin_amdgcn_s_setprio(3);
    // Only the even lane of a pair carries the element's stay.  The odd lane adds -inf instead of the stay score, so that its stay
    // candidate, like all candidates of a dead element, whose score is -inf, never passes a cut and never wins a maximum, without a mask.
    const float stay_h = h == 0 ? stay : -INFINITY;
    const uint32_t from = (uint32_t)i << 10, from_stay = from | (1u << 15);  // the element's index as "prev" of its candidates
    int rows_ready = 0;  // last value seen of the loader's counter; it is usually several rows ahead
    const int b0 = 2 * h;
    const uint32_t cand_base = lds_address(&all.cand[member].step[0]);
    const uint32_t elem_base = lds_address(&sh.elem[0]);
    const uint32_t cand_mine = cand_base + 8u * (uint32_t)lane;           // candidates 4i+b0, 4i+b0+1
    const uint32_t cand_dump = cand_base + 4u * (uint32_t)(4 * kW + lane);  // where a stay without a partner writes
    // What a time step reads from LDS depends only on the beam it starts from, so it is
    // fetched as soon as that beam is known (at the end of the previous step): the row
    // entries of the lane's candidates, and the hash index: the element's own entry goes in, is
    // read back, and the entry filed under `want` is read.
    // fp16 scores of the lane's two step candidates: both in one word (planes), or each in the low half of a word
    constexpr bool kPlanes = ScoreRow<S, COLS, FWD>::kPlanes;
    uint32_t r0h, r1h;
    f32x2 g01;
    float gst;
    uint32_t probe;      // index entry found under `want`
    uint32_t expected;   // what it is if a partner is there, but for the partner's slot
    uint32_t entry, mine_back;  // the element's own entry, as written and as found again
    uint32_t step_at;           // a partner is step candidate 4j + last base of this element
    uint64_t vm = ~0ull, vs = 0x5555555555555555ull;  // lanes of live elements; of their stay candidates, which sit on the even lanes
    const int i_stay = h == 0 ? i : kW;  // of an odd lane never below the beam's width
    uint32_t hash_keep = ~Idx::kAddress, slot_bits = Idx::kSlot;
    asm volatile("" : "+v"(hash_keep), "+v"(slot_bits));  // a vector instruction takes one scalar operand
    const uint32_t slot_tag = (uint32_t)i << 4;
    uint32_t round = 0;  // generation of the present ring round
    // ring addresses: the same in every lane, kept in scalar registers
    const uint32_t ring_s = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(lds_u32 *)&row_s[0][0]);
    const uint32_t ring_b = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uintptr_t)(lds_u32 *)&row_b[0][0]);
    uint32_t step_row = ring_s + 4u * (uint32_t)h;  // the lane's two of an element's four steps, less 8 * state
    asm volatile("" : "+v"(step_row));
    // The ring slot of a time step's row is known where steps are written out (K), elsewhere (K < 0) it is worked out.
    auto ring_slot = [&](int tt, auto k_tag) {
        constexpr int K = decltype(k_tag)::value;
        return K >= 0 ? (uint32_t)K : (uint32_t)tt % (uint32_t)LR;
    };
    auto wait_row = [&](int tt, auto k_tag) {
        constexpr int K = decltype(k_tag)::value;
        if constexpr (K >= 0 && K % Cfg::kHandBack != 0) return;
        int rows = tt + (K >= 0 ? Cfg::kHandBack : 1);
        rows = rows < T ? rows : T;
        while (__builtin_expect(rows_ready < rows, 0)) {  // the counter is one LDS word: the same value in every lane
            rows_ready = __builtin_amdgcn_readfirstlane(observe(ready));
            if (rows_ready < rows) __builtin_amdgcn_s_sleep(1);
        }
    };
    auto next_round = [&](uint32_t slot) {
        if (slot != 0) return;
        round += Idx::kRound;
        if (__builtin_expect(round == Idx::kRoundEnd, 0)) {
            round = Idx::kRound;
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            uint32_t zero;
            asm volatile("v_mov_b32 %0, 0" : "=v"(zero));  // here, not in registers through the search
            u32x4 none;
            none.x = none.y = none.z = none.w = zero;
#pragma unroll 1
            for (uint32_t at = 0; at < 4u * Idx::kBuckets; at += 1024u) *(LDS_AS u32x4 *)(uintptr_t)(idx_base + at + 16u * (uint32_t)lane_now()) = none;
            wave_fence();
        }
    };
    auto fetch_row = [&](int tt, auto k_tag) {
        const uint32_t slot = ring_slot(tt, k_tag);
        const uint32_t gen = round | (slot << 2);
        // hash index of the beam this step starts from; dead lanes file their leftovers apart
        const uint32_t own = (uint32_t)pick_by_bit(vm, (int)and_or(hash, Idx::kAddress, idx_base), (int)idx_dump);
        entry = and_or(hash, hash_keep, slot_tag | gen);
        lds_u32 *own_p = (lds_u32 *)(uintptr_t)own;
        own_p[0] = entry;
        __builtin_amdgcn_sched_barrier(0);  // the entries go out first, the row is asked for next: `want` takes a while
        wave_fence();  // one wave's LDS operations are carried out in order: the reads below see every lane's entry
        // scores of the candidates with bases b0, b0 + 1, which lie in the column of the dropped base; guide terms rb[lo4 + b0 + {0,1}]
        // and rb[state]
        const uint32_t st4 = (uint32_t)state << 2;
        const uint32_t cand = and_or(st4, (uint32_t)(S - 1), (uint32_t)b0);  // lo4 + b0
        const uint32_t rs = ring_s + slot * (uint32_t)sizeof(row_s[0]), rb = ring_b + slot * (uint32_t)sizeof(row_b[0]);
        if constexpr (kPlanes) {
            r0h = *(const lds_u32 *)(uintptr_t)(((uint32_t)state << 3) + step_row + slot * (uint32_t)sizeof(row_s[0]));
        } else {
            const uint32_t top = (uint32_t)state >> (BITS - 2);  // the dropped base
            uint32_t at_s;  // rs[COLS * (lo4 + b0 + {0,1}) + (COLS - 4) + top]
            if constexpr (COLS == 4) at_s = (((cand << 2) | top) << 1) + rs;
            else at_s = cand * 10u + (top << 1) + rs;
            typedef __attribute__((address_space(3))) uint16_t lds_u16;
            r0h = *(const lds_u16 *)(uintptr_t)(at_s + 2u * (COLS - 4));
            r1h = *(const lds_u16 *)(uintptr_t)(at_s + 2u * (COLS - 4) + 2u * COLS);
        }
        g01 = lds_load_f2((cand << 2) + rb);
        gst = lds_load_f(st4 + rb);
        __builtin_amdgcn_sched_barrier(0);
        want = crc2_inverse(hash, info);  // the last base: the two lowest bits
        probe = *(const lds_u32 *)(uintptr_t)and_or(want, Idx::kAddress, idx_base);
        mine_back = own_p[0];
        step_at = and_or(st4, 12u, cand_base);
        asm volatile("" : "+v"(step_at));
        __builtin_amdgcn_sched_barrier(0);  // nothing that waits for the row goes before the look-up
        expected = and_or(want, hash_keep, gen);
    };
    typedef std::integral_constant<int, -1> AnySlot;
    wait_row(0, std::integral_constant<int, 0>{});  // as many rows as the steps written out expect to find, not row 0 alone
    next_round(0);
    fetch_row(0, AnySlot{});
    const uint64_t replay_all = (flags & 1) ? ~0ull : 0ull;
    ofk_beam_slot_t *bv_row = bv;  // row t of the persisted slots
    // One time step.  The last one (LAST) differs in what it hands on (nothing is fetched for a next
    // step, the best survivor goes to slot 0) and is compiled apart, so that the others carry no
    // test for it.
    //
    // The wave is alone on its SIMD: a step costs its instructions, about four cycles each, plus the
    // LDS round trips and the reads of comparison masks by the scalar unit (about twenty cycles) that
    // nothing is placed into (about 1110 cycles for 1 chunk of 64 or 256 states: 0.80 ms at T = 1666; before steps were written out and
    // rows kept in planes 0.93; in the order of the text, with every wait where its value is first needed, 1.02).  Hence the order
    // below: what does not depend on a round trip is issued while it is under way, comparisons are issued in groups whose masks are
    // read afterwards.  That order is fenced where the compiler would count a mask as soon as it is compared: the counts of the cut-off behind all
    // six comparisons, the fold's verdict behind the logarithm, the proof's behind the comparisons of the next masks (0.847 | 0.800 ms
    // together; 512 chunks of 64 states 0.957 | 0.915).
    auto step = [&](const int next_t, auto k_tag, auto last_tag) {  // next_t - 1 is the time step, K the ring slot of row next_t
        constexpr int K = decltype(k_tag)::value;
        constexpr bool LAST = decltype(last_tag)::value;
        // (score + transition) + guide, the CPU path's order of additions; the fp16 transition is
        // converted inside the first addition
        float c0 = ::add_half<0>(r0h, score) + g01.x;
        float c1 = ::add_half<kPlanes ? 1 : 0>(kPlanes ? r0h : r1h, score) + g01.y;
        float cs0 = (score + stay_h) + gst;
        lds_store_f2(cand_mine, c0, c1);  // for the merges below

        // which previous element j has hash_j == want_i: off the index if every live element found its
        // own entry intact, else by comparing with every hash
        uint32_t at = and_or(probe, slot_bits, step_at);
        uint64_t moved = ballot(mine_back != entry);
        if constexpr (K < 0) moved |= replay_all;
        // (probe ^ expected) & ~kSlot, which is nothing if there is a partner: live even lanes whose stay has one
        uint64_t mine_mask = ballot(__builtin_amdgcn_bitop3_b32(probe, Idx::kSlot, expected, 0x12) == 0u) & vs;
        if (__builtin_expect(moved != 0, 0)) {
            // Two live elements in one bucket (or with one hash).  Bit k of m says whether hash k of this
            // half of the beam equals `want`: each comparison is shifted into an accumulator with an
            // add-with-carry (a = 2a + equal), two accumulators so that no instruction waits for the one
            // before it.
            uint32_t hq[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) hq[k] = sh.elem[16 * h + k].hash;
            uint32_t lo8, hi8;
            {
                uint64_t e0, e1, e2, e3, f0, f1, f2, f3, carry;
                asm("v_cmp_eq_u32_e64 %[e3], %[w], %[x3]\n\t"
                    "v_cmp_eq_u32_e64 %[f3], %[w], %[y3]\n\t"
                    "v_cmp_eq_u32_e64 %[e2], %[w], %[x2]\n\t"
                    "v_cmp_eq_u32_e64 %[f2], %[w], %[y2]\n\t"
                    "v_cmp_eq_u32_e64 %[e1], %[w], %[x1]\n\t"
                    "v_cmp_eq_u32_e64 %[f1], %[w], %[y1]\n\t"
                    "v_cmp_eq_u32_e64 %[e0], %[w], %[x0]\n\t"
                    "v_cmp_eq_u32_e64 %[f0], %[w], %[y0]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], 0, 0, %[e3]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], 0, 0, %[f3]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e2]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f2]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e1]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f1]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e0]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f0]"
                    : [ax] "=&v"(lo8), [ay] "=&v"(hi8), [e0] "=&s"(e0), [e1] "=&s"(e1), [e2] "=&s"(e2),
                      [e3] "=&s"(e3), [f0] "=&s"(f0), [f1] "=&s"(f1), [f2] "=&s"(f2), [f3] "=&s"(f3),
                      [c] "=&s"(carry)
                    : [w] "v"(want), [x0] "v"(hq[4]), [x1] "v"(hq[5]), [x2] "v"(hq[6]), [x3] "v"(hq[7]),
                      [y0] "v"(hq[12]), [y1] "v"(hq[13]), [y2] "v"(hq[14]), [y3] "v"(hq[15]));
                asm("v_cmp_eq_u32_e64 %[e3], %[w], %[x3]\n\t"
                    "v_cmp_eq_u32_e64 %[f3], %[w], %[y3]\n\t"
                    "v_cmp_eq_u32_e64 %[e2], %[w], %[x2]\n\t"
                    "v_cmp_eq_u32_e64 %[f2], %[w], %[y2]\n\t"
                    "v_cmp_eq_u32_e64 %[e1], %[w], %[x1]\n\t"
                    "v_cmp_eq_u32_e64 %[f1], %[w], %[y1]\n\t"
                    "v_cmp_eq_u32_e64 %[e0], %[w], %[x0]\n\t"
                    "v_cmp_eq_u32_e64 %[f0], %[w], %[y0]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e3]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f3]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e2]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f2]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e1]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f1]\n\t"
                    "v_addc_co_u32_e64 %[ax], %[c], %[ax], %[ax], %[e0]\n\t"
                    "v_addc_co_u32_e64 %[ay], %[c], %[ay], %[ay], %[f0]"
                    : [ax] "+v"(lo8), [ay] "+v"(hi8), [e0] "=&s"(e0), [e1] "=&s"(e1), [e2] "=&s"(e2),
                      [e3] "=&s"(e3), [f0] "=&s"(f0), [f1] "=&s"(f1), [f2] "=&s"(f2), [f3] "=&s"(f3),
                      [c] "=&s"(carry)
                    : [w] "v"(want), [x0] "v"(hq[0]), [x1] "v"(hq[1]), [x2] "v"(hq[2]), [x3] "v"(hq[3]),
                      [y0] "v"(hq[8]), [y1] "v"(hq[9]), [y2] "v"(hq[10]), [y3] "v"(hq[11]));
            }
            uint32_t m = lo8 | (hi8 << 8);
            m <<= 16 * h;
            // the two lanes of an element looked at 16 hashes each and join their masks
            m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1 /* quad_perm:[1,0,3,2] */, 0xF, 0xF, true);
            const uint32_t live = w >= 32 ? 0xFFFFFFFFu : ((1u << w) - 1u);
            const uint32_t match = m & live;
            mine_mask = ballot(match != 0u) & vs;
            const uint32_t j = (uint32_t)__builtin_ctz(match | 0x80000000u) & 31u;
            at = step_at + 16u * j;
            // Merges in parallel need every stay to have one partner and every step candidate one claimant.
            // Otherwise (only possible after a CRC collision; flags bit 0 forces it) the merges are
            // replayed one by one in the CPU path's order, from the scores as they were before any merge.
            const uint32_t claim_at = (uint32_t)pick_by_bit(mine_mask, (int)(4u * j + ((uint32_t)state & 3u)), 4 * kW + lane_now());
            sh.claim[claim_at] = (uint32_t)i;
            wave_fence();
            const uint32_t claimed = sh.claim[claim_at];
            const uint32_t odd = (match & (match - 1u)) | (claimed ^ (uint32_t)i);
            if ((ballot(odd != 0u) & mine_mask) != 0 || (flags & 1)) {
                if (h == 0) sh.stay_score[i] = cs0;
                wave_fence();
                if (lane_now() == 0) {
                    for (int a = 0; a < w; ++a) {
                        const uint32_t ha = sh.elem[a].hash;
                        const uint32_t base = sh.elem[a].info & 3u;
                        for (int b = 0; b < w; ++b) {
                            if (crc2(sh.elem[b].hash, base) != ha) continue;
                            float *st = &all.cand[member].step[4 * b + (int)base];
                            const float both = log_sum_exp(sh.stay_score[a], *st, lse);
                            if (sh.stay_score[a] > *st) {
                                sh.stay_score[a] = both;
                                *st = -FLT_MAX;
                            } else {
                                *st = both;
                                sh.stay_score[a] = -FLT_MAX;
                            }
                        }
                    }
                }
                wave_fence();
                const f32x2 c01 = lds_load_f2(cand_mine);
                c0 = c01.x;
                c1 = c01.y;
                if (h == 0) cs0 = sh.stay_score[i];
                mine_mask = 0;
            }
        }

        // merge stays with the step spelling the same sequence (src/beam_search.c:281-316).  Every lane
        // has filed its two step candidates; a stay with a partner reads the partner's score, folds the
        // two, keeps its half of the outcome and overwrites the partner with the other half; every
        // lane reads its step candidates back.  Lanes without a merge go through the same
        // instructions with whatever their registers hold and a dump slot as target: no exec
        // masking on the way.  Conditions are kept as wave-wide masks in scalar registers and combined
        // there; a select takes its mask as it is.
        wave_fence();
        const float other = lds_load_f(at);
        // meanwhile: everything this step needs of row t is in registers; and the slot the traceback
        // reads is persisted (src/beam_search.c:417-427).  Both halves hold the same element and store the
        // same slot; slots past the width are never followed by the traceback.
        if constexpr (K < 0) {
            bv_row[i] = (ofk_beam_slot_t)info;
            bv_row += kW;
        } else {
            bv_row[(K + LR - 1) % LR * kW + i] = (ofk_beam_slot_t)info;
            if constexpr (K == 0) bv_row += LR * kW;
        }
        // no wait before this store: the wave's reads of row t are ahead of it in the LDS queue
        if constexpr (K < 0 || K % Cfg::kHandBack == 0)
            __hip_atomic_store(consumed, next_t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint32_t hash_again = hash;  // for the stay's record, in registers side by side with the rest of it
        asm volatile("" : "+v"(hash_again));
        const uint64_t stay_above = ballot(cs0 > other);  // its mask is not asked for before the fold is on its way
        const uint32_t target = (uint32_t)pick_by_bit(mine_mask, (int)at, (int)cand_dump);
        // The fold from hardware exp/log, which the step goes on with.  Whether it rounds like the CPU path's double
        // arithmetic (all but a few merges in a thousand at usual score magnitudes) is looked at while the new beam is on its
        // way; if not, the step is done again from here with the double fold.
        const FoldValue estimate = log_sum_exp_value(cs0, other);
        __builtin_amdgcn_sched_barrier(0);
        const uint64_t step_wins = mine_mask & ~stay_above;
        typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
        u32x3 e;
        auto finish = [&](const float folded) {
        lds_store_f(target, pick_by_bit(step_wins, folded, -FLT_MAX));
        wave_fence();
        const f32x2 c01 = lds_load_f2(cand_mine);

        // cut-off (src/beam_search.c:320-381)
        // Dead lanes carry -inf as their score, and so do their candidates (and the stays of odd lanes, see stay_h): they pass no cut, while the
        // losers of merges, -FLT_MAX, pass the one that keeps everything.
        // The best score does not wait for the step candidates to come back: a fold is not below either of
        // the two scores it joins, so the maximum of the scores before the merges and of the folds is that after them.
        const float stay_or_fold = pick_by_bit(mine_mask, folded, cs0);
        NextRecords next;
        float cs;
        const Cuts first = wave_max_beside_records(c0, c1, stay_or_fold, next, cs, hash, (uint32_t)b0, (uint32_t)state, from_stay,
                                                   (uint32_t)state << 2, (uint32_t)(S - 1), from, step_wins, -FLT_MAX, gst, log_cut);
        const float s0 = c01.x, s1 = c01.y;  // the steps' scores after the merges
        next.rest0 = s0 - g01.x;
        next.rest1 = s1 - g01.y;

        // Nearly every step has more candidates above the first cut than the width, and goes on to the cut
        // halfway to the best score: both are counted at once.
        // Of the bounds of the bisection their halves are kept, which makes the cut between them, (lo + hi) / 2 on the CPU path, one
        // addition and the two that can come next a fused multiply-add each: halving is exact (down to 2^-125) and changes no rounding.
        const float lo = first.lo;  // -FLT_MAX: no cut at all, or nobody alive
        float half_lo = first.half_lo, half_hi = first.half_hi, cut = first.cut;
        const uint64_t a0 = ballot(s0 >= lo), a1 = ballot(s1 >= lo), as = ballot(cs >= lo);
        uint64_t k0 = ballot(s0 >= cut), k1 = ballot(s1 >= cut), ks = ballot(cs >= cut);
        __builtin_amdgcn_sched_barrier(0);  // all comparisons, then the first count: a mask takes its time to the scalar unit
        int kept = popc64(a0) + popc64(a1) + popc64(as);
        // kept candidates on lower lanes: masked bit counts
        auto lower = [&](uint64_t mask, int start) {
            return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)mask, (uint32_t)start));
        };
        int steps_kept = popc64(k0) + popc64(k1);  // of `kept` those that are steps
        if (__builtin_expect(kept <= kW, 0)) {
            k0 = a0;
            k1 = a1;
            ks = as;
            steps_kept = popc64(k0) + popc64(k1);
        } else {
            // Bisection between the cut and the best score.  Every cut tried in here lies above
            // (-FLT_MAX + best) / 2, so the losers of merges never pass.  The cut between the bounds is the CPU path's (cut + hi) / 2 or
            // (cut + lo) / 2: one of the two bounds is the cut just tried.  Two guesses in a row settle most steps; they
            // are nested and not left by jumps, for which the compiler builds a ladder of blocks that costs as much as a guess.
            float next_up, next_down;  // both cuts that can come next, worked out while the masks travel to the scalar unit
            auto look_ahead = [&] {
                next_up = __builtin_fmaf(cut, 0.5f, half_hi);
                next_down = __builtin_fmaf(cut, 0.5f, half_lo);
                asm volatile("" : "+v"(next_up), "+v"(next_down));
            };
            auto next_guess = [&] {
                const bool up = kept > kW;
                const float half = 0.5f * cut;
                half_lo = up ? half : half_lo;
                half_hi = up ? half_hi : half;
                cut = up ? next_up : next_down;
            };
            auto count = [&] {
                k0 = ballot(s0 >= cut);
                k1 = ballot(s1 >= cut);
                ks = ballot(cs >= cut);
                look_ahead();
                __builtin_amdgcn_sched_barrier(0);
                steps_kept = popc64(k0) + popc64(k1);
                kept = steps_kept + popc64(ks);
            };
            auto too_many_or_few = [&] { return (unsigned)(kept - (kW * 8) / 10) > (unsigned)(kW - (kW * 8) / 10); };  // not 25..32
            look_ahead();
            kept = steps_kept + popc64(ks);
            if (too_many_or_few()) {
                next_guess();
                count();
                if (too_many_or_few()) {
                    next_guess();
                    count();
                    if (too_many_or_few()) {
                        // The tenth guess: the CPU path moves its bounds once more, tries a cut whose count it
                        // never looks at, and settles for the upper bound, whatever that keeps: of more candidates
                        // than the width the first ones, in candidate order, stay.
#pragma unroll 1
                        for (int guess = 5;; ++guess) {
                            next_guess();
                            if (guess == 10) cut = 2.0f * half_hi;
                            count();
                            if (!too_many_or_few() || guess == 10) break;
                        }
                        if (kept > kW) {
                            const int rank0 = lower(k1, lower(k0, 0));
                            const int rank1 = add_bit_of(rank0, k0);
                            const int ranks = lower(ks, steps_kept);
                            k0 &= ballot(rank0 < kW);
                            k1 &= ballot(rank1 < kW);
                            ks &= ballot(ranks < kW);
                            kept = kW;
                            steps_kept = popc64(k0) + popc64(k1);
                        }
                    }
                }
            }
        }

        // survivors in candidate order: steps (i, b) by i then b, then stays by i
        {
            // k0, k1 and ks hold this lane's own verdicts at its bit (dead lanes and the stays of the odd
            // lanes never pass): the masks select directly, nothing is compared again
            const int rank0 = lower(k1, lower(k0, 0));
            const int rank1 = add_bit_of(rank0, k0);
            const int ranks = lower(ks, steps_kept);
            // every lane stores all three of its candidates, the ones that are dropped into its own dump
            // slot: no exec masking on the path from the cut-off to the next beam
            const int dump = kW + lane;
            const int slot0 = pick_by_bit(k0, rank0, dump);
            const int slot1 = pick_by_bit(k1, rank1, dump);
            const int slots = pick_by_bit(ks, ranks, dump);
            if constexpr (LAST) {
                // the last beam is ranked by its candidate scores (src/beam_search.c:398-414)
                next.rest0 = s0;
                next.rest1 = s1;
                next.rests = cs;
            }
            auto put = [&](int slot, uint32_t hsh, uint32_t inf, float rst) {
                uint32_t at_elem;
                asm("v_lshl_add_u32 %0, %1, 4, %2" : "=v"(at_elem) : "v"(slot), "v"(elem_base));
                u32x3 rec;
                rec.x = hsh;
                rec.y = __float_as_uint(rst);
                rec.z = inf;
                *(LDS_AS u32x3 *)(uintptr_t)at_elem = rec;
            };
            put(slot0, next.h0, next.info0, next.rest0);
            put(slot1, next.h1, next.info1, next.rest1);
            put(slots, hash_again, next.infos, next.rests);
            wave_fence();
            // every lane reads its slot; slots past the new width hold leftovers: they count as dead through
            // their score and persist as zero, which is what the CPU path's untouched slots hold (a beam
            // cut below 1 empties the beam, and the traceback then walks such slots)
            e = *(const LDS_AS u32x3 *)(uintptr_t)(elem_base + 16u * (uint32_t)i);
        }
        w = kept;
        };
        finish(estimate.value);
        // while the beam is on its way: are the folds proven, and who is alive (the best candidate is always kept: w is zero only
        // after NaN scores)
        __builtin_amdgcn_sched_barrier(0);
        uint64_t open = ballot(!log_sum_exp_settled(estimate));
        asm volatile("" : "+s"(open));  // compared here, looked at further down
        uint64_t vm_next = ballot(i < w), vs_next = ballot(i_stay < w);
        asm volatile("" : "+s"(vm_next), "+s"(vs_next));
        __builtin_amdgcn_sched_barrier(0);
        if (__builtin_expect((open & mine_mask) != 0, 0)) {
            finish(log_sum_exp(cs0, other, lse));  // of the same beam: vm and vs are still its masks
            vm_next = ballot(i < w);
            vs_next = ballot(i_stay < w);
        }
        vm = vm_next;
        vs = vs_next;
        if constexpr (!LAST) {
            next_round(ring_slot(next_t, k_tag));
            wait_row(next_t, k_tag);
            __builtin_amdgcn_sched_barrier(0);
        }
        hash = e.x;
        info = (uint32_t)pick_by_bit(vm, (int)e.z, 0);
        score = pick_by_bit(vm, __uint_as_float(e.y), -INFINITY);
        state = (int)(info & 1023u);
        if constexpr (!LAST) fetch_row(next_t, k_tag);

        // last block: the best survivor goes to slot 0 (src/beam_search.c:398-414)
        if constexpr (LAST) {
            const bool in = i < w;
            const float top_score = wave_max(score);
            const uint64_t at_top = ballot(in && h == 0 && score == top_score);
            const int arg_lane = (top_score > -FLT_MAX && at_top != 0) ? __builtin_ctzll(at_top) : 0;  // an even lane
            const int arg = arg_lane >> 1;
            if (arg != 0) {
                const uint32_t in0 = lane_u(info, 0), ina = lane_u(info, arg_lane);
                if (i == 0) info = ina;
                if (i == arg) info = in0;
            }
            bv_row[i] = (ofk_beam_slot_t)info;
        }
    };
    // LR steps at a time: what goes by the ring slot, the parity of hand-overs and the row of persisted slots is then
    // part of the instructions.  (Serial replay of the merges, for tests: one step at a time.)
    int next_t = 1;
    if (replay_all == 0) {
        for (; next_t + LR <= T; next_t += LR)
            static_for_upwards<LR>([&](auto k) {
                constexpr int K = (decltype(k)::value + 1) % LR;
                step(next_t + decltype(k)::value, std::integral_constant<int, K>{}, std::false_type{});
            });
    }
    for (; next_t < T; ++next_t) step(next_t, AnySlot{}, std::false_type{});
    step(T, AnySlot{}, std::true_type{});
    };

    if (wave < kGroupChunks) {
        search();
        // The slots are in memory, and what was done in LDS is done, before the other waves go on.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if constexpr (kTeam > 1) __hip_atomic_store(&sh.searched, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else {
        if (wave >= kFirstLoader) {
            mate = 1 + (wave - kFirstLoader) / kGroupChunks;
            if (mate == 1) load_rows();
        }
        if (kTeam == 1 || mate * kTraceRows >= T) return;  // no block to trace
        while (__hip_atomic_load(&sh.searched, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) __builtin_amdgcn_s_sleep(16);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }

    // ---- traceback from slot 0 of the last block (src/beam_search.c:432-439) ----
    // Followed one row at a time the walk is a chain of T dependent LDS reads.  It is done per block
    // of 128 rows instead, staged in LDS (in the memory of the hash index, which is dead now), in two
    // passes.  Pass 1 walks the block's eight sub-blocks of 16 rows at the same time, each from all
    // 32 slots it could be entered through (lanes 0..31 the four newer sub-blocks, lanes 32..63 the
    // four older ones): where every entry leaves its sub-block.  Eight lane reads then thread the
    // real entry through the block.  Pass 2 walks the eight sub-blocks again, each from its real
    // entry (eight lanes per sub-block, lane q keeping rows 2q and 2q+1 of the walk), and the
    // wave stores 128 states and moves side by side.  Rows that a block lacks at its old end are
    // staged as slots that point at themselves.  The next block's slots travel from global memory
    // while a block is walked.
    //
    // Pass 1 needs nothing of another block.  Where the index has room the waves of the chunk deal the blocks round, leave each
    // block's eight maps in LDS, a word a lane, and meet once; every wave then threads the entry through all blocks and walks its own
    // again (kernels, T = 1666, one wave | with the others, us: 1 chunk of 64 states 880 | 862, 512, two waves, 985 | 978; 512 of 256 states
    // merged 1001 | 993, 256 of 1024 1672 | 1666).  They wait for the search alone, and the search's wave for their maps only here, so all
    // waits end.  The kernel's waves share a compute unit, whose first-level cache writes through: their fences need not write the second
    // level back (which took 10 us of the merged kernel of 512 chunks of 256 states, 17 of 256 of 1024).
    {
        constexpr int RB = kTraceRows;  // rows per block
        const int lane = lane_now();
        constexpr int kStage = RB * kW * (int)sizeof(ofk_beam_slot_t);  // bytes of a staged block
        static_assert((kTeam > 1 ? kTeam * kStage + (Idx::kMapsApart ? 0 : (int)sizeof(TraceMaps)) : 2 * kStage) <= Idx::kBuckets * 4, "the index has room");
        int32_t *st_out = states + (size_t)n * T;
        uint8_t *mv_out = moves + (size_t)n * T;
        const uint32_t idx_base = lds_address(&all.idx[member][0]);
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        u32x4 pre[8];  // a block on its way from global memory: 16-byte piece 64 k + lane in pre[k]
        // block b covers rows hi - rows + 1 .. hi with hi = T - RB b; piece x of the buffer holds
        // row x / 4 - (RB - rows) of those, or slots pointing at themselves before that
        auto load_block = [&](int hi) {
            const int rows = hi < RB ? hi : RB;
            const u32x4 *src = reinterpret_cast<const u32x4 *>(bv + (size_t)(hi - rows + 1) * kW);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int x = 64 * k + lane - 4 * (RB - rows);
                pre[k] = src[x > 0 ? x : 0];  // every lane loads (pieces before the block's first are not used)
            }
        };
        auto store_block = [&](int hi, uint32_t buf) {
            const int rows = hi < RB ? hi : RB;
            const uint32_t c8 = (uint32_t)(lane & 3) * 8u;  // first of the eight slots of an identity piece
            u32x4 self;
            self.x = ((c8 + 0u) << 10) | ((c8 + 1u) << 26);
            self.y = ((c8 + 2u) << 10) | ((c8 + 3u) << 26);
            self.z = ((c8 + 4u) << 10) | ((c8 + 5u) << 26);
            self.w = ((c8 + 6u) << 10) | ((c8 + 7u) << 26);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int x = 64 * k + lane - 4 * (RB - rows);
                *(LDS_AS u32x4 *)(uintptr_t)(buf + 16u * (uint32_t)(64 * k + lane)) = x >= 0 ? pre[k] : self;
            }
        };
        auto slot_at = [&](uint32_t row_base, uint32_t cur, int row) {  // slot `cur` of row `row` above row_base
            uint32_t at;
            asm("v_lshl_add_u32 %0, %1, 1, %2" : "=v"(at) : "v"(cur), "v"(row_base));
            return (uint32_t) * (const LDS_AS uint16_t *)(uintptr_t)(at + 64u * (uint32_t)row);
        };
        // pass 1: sub-block s = 4 (lane / 32) + k covers buffer rows 127 - 16 s down to 112 - 16 s; where entry lane % 32 leaves it is byte
        // k of the lane's word
        auto map_block = [&](uint32_t buf) {
            uint32_t cur[4];
            const uint32_t low1 = buf + 64u * (uint32_t)(112 - 64 * (lane >> 5));  // oldest row of this lane's sub-block k = 0
#pragma unroll
            for (int k = 0; k < 4; ++k) cur[k] = (uint32_t)lane & 31u;
#pragma unroll
            for (int r = 15; r >= 0; --r) {
                uint32_t e[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) e[k] = slot_at(low1 - (uint32_t)(16 * 64 * k), cur[k], r);
#pragma unroll
                for (int k = 0; k < 4; ++k) cur[k] = (e[k] >> 10) & 31u;
            }
            return cur[0] | cur[1] << 8 | cur[2] << 16 | cur[3] << 24;
        };
        // lanes 8 s .. 8 s + 7 walk sub-block s in pass 2; lane q of them keeps rows 2q, 2q+1 of the walk
        const int sb2 = lane >> 3, q = lane & 7;
        uint32_t cursor = 0;  // slot through which the walk enters the block: the same in every lane
        auto thread_block = [&](uint32_t map) {  // and the slot through which it enters the lane's sub-block
            uint32_t enter = 0;
#pragma unroll
            for (int sb = 0; sb < 8; ++sb) {
                enter = sb2 == sb ? cursor : enter;
                cursor = ((uint32_t)__builtin_amdgcn_readlane((int)map, (int)(cursor + 32u * (uint32_t)(sb >> 2))) >> (8 * (sb & 3))) & 31u;
            }
            return enter;
        };
        uint32_t newer = 0, older = 0;
        auto walk_block = [&](uint32_t buf, uint32_t walk) {
            const uint32_t low2 = buf + 64u * (uint32_t)(112 - 16 * sb2);
#pragma unroll
            for (int r = 15; r >= 0; --r) {
                const uint32_t e = slot_at(low2, walk, r);
                if (r & 1) newer = q == (15 - r) / 2 ? e : newer;
                else older = q == (15 - r) / 2 ? e : older;
                walk = (e >> 10) & 31u;
            }
        };
        // buffer row of `newer`: 127 - 16 sb2 - 2 q; the block's rows start at buffer row RB - rows,
        // which is row hi - rows + 1 of the chunk, i.e. time step hi - rows
        auto store_path = [&](int hi) {
            const int rows = hi < RB ? hi : RB;
            const int p_new = 127 - 16 * sb2 - 2 * q;
            const int t_new = hi - rows + (p_new - (RB - rows));
            if (p_new >= RB - rows) {
                st_out[t_new] = (int32_t)(newer & 1023u);
                mv_out[t_new] = (t_new == 0 || !(newer >> 15)) ? (uint8_t)1 : (uint8_t)0;
            }
            if (p_new - 1 >= RB - rows) {
                st_out[t_new - 1] = (int32_t)(older & 1023u);
                mv_out[t_new - 1] = (t_new - 1 == 0 || !(older >> 15)) ? (uint8_t)1 : (uint8_t)0;
            }
        };
        if constexpr (kTeam == 1) {
            load_block(T);
            store_block(T, idx_base);
            int blk = 0;
            for (int hi = T; hi > 0; hi -= RB, ++blk) {  // two buffers in turn
                const uint32_t buf = idx_base + (uint32_t)(blk & 1) * (uint32_t)kStage;
                if (hi > RB) load_block(hi - RB);
                wave_fence();
                walk_block(buf, thread_block(map_block(buf)));
                // the next block goes into the other buffer before this block's results are stored: the wait
                // for its loads then does not wait for those stores as well
                if (hi > RB) store_block(hi - RB, idx_base + (uint32_t)((blk + 1) & 1) * (uint32_t)kStage);
                store_path(hi);
            }
        } else {
            // block b is wave b % kTeam's.  The newest of a wave's blocks comes last in pass 1, so that it is staged where pass 2 begins.
            const int blocks = (T + RB - 1) / RB, waves = blocks < kTeam ? blocks : kTeam;
            const uint32_t buf = idx_base + (uint32_t)(mate * kStage);
            uint32_t maps = idx_base + (uint32_t)(kTeam * kStage);
            if constexpr (Idx::kMapsApart) maps = lds_address(&lds[member].trace);
            maps += 4u * (uint32_t)lane;
            int b = blocks - 1 - (blocks - 1 - mate) % kTeam;  // the oldest of the wave's
            load_block(T - RB * b);
            for (; b >= 0; b -= kTeam) {
                wave_fence();
                store_block(T - RB * b, buf);
                if (b >= kTeam) load_block(T - RB * (b - kTeam));
                wave_fence();
                *(LDS_AS uint32_t *)(uintptr_t)(maps + 256u * (uint32_t)b) = map_block(buf);
            }
            if (mate + kTeam < blocks) load_block(T - RB * (mate + kTeam));
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            if (lane == 0) __hip_atomic_fetch_add(&sh.mapped, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            while (observe(&sh.mapped) < waves) {}
            uint32_t map = *(const LDS_AS uint32_t *)(uintptr_t)maps;
            for (b = 0; b < blocks; ++b) {
                const uint32_t here = map;
                if (b + 1 < blocks) map = *(const LDS_AS uint32_t *)(uintptr_t)(maps + 256u * (uint32_t)(b + 1));
                const uint32_t enter = thread_block(here);
                if (b % kTeam != mate) continue;
                const int hi = T - RB * b;
                wave_fence();
                walk_block(buf, enter);
                wave_fence();
                if (b + kTeam < blocks) {
                    store_block(hi - RB * kTeam, buf);
                    if (b + 2 * kTeam < blocks) load_block(hi - 2 * RB * kTeam);
                }
                store_path(hi);
            }
        }
    }
}

// Chunks of a search that share a workgroup, and so a compute unit's LDS.  256 units: up to 512 chunks fit two to a unit; larger
// batches go four to a group where the LDS of four chunks fits (64 and 256 states).  Few chunks have a unit each: two searches on one wait for
// each other's LDS operations, and with the LDS to itself a chunk has an index so large that one step in forty instead of one in
// twenty (1024 states: in ten) meets two elements in a bucket.  Search, two to a unit | one,
// T = 1666 (1024 states 833), ms: 64 states, 1 chunk 0.943 | 0.929, 16 1.033 | 0.936, 160 1.05 | 0.96; 256 states, 16
// 1.024 | 0.941, 160 1.04 | 0.99; 1024 states, 37 0.565 | 0.490, 100 0.577 | 0.504, 160 (split: units are short) 0.74 | 1.0.
//
// Such a group leaves no room for a second on its unit.  So a search that is alone on the device takes units as long as those
// it leaves hold a second decode of the same size that begins while it runs, two chunks (1024 states: one) to a unit: workgroups are dealt
// round eight XCDs of 32 units, 20 and 10 of them with 160 chunks, 22 and 11 with 170.  Two callers whose calls begin at
// random, a call's mean | 90th percentile, ms, two to a unit | one: 256 states, 160 chunks 1.98 2.19 | 2.02 2.30, 170 2.01 2.25 |
// 2.12 2.50, 200 2.03 2.28 | 2.23 2.78; 64 states, 160 1.71 1.96 | 1.68 1.92, 170 1.72 1.96 | 1.74 2.16 (one caller: 256 states, 160
// chunks 1.785 | 1.73, 200 1.80 | 1.755).  Where other decodes may be under way, three of them, a lane each, find units for all their chunks.
int search_group(int S, int N, int flags) {
    const bool alone = (flags & OFK_SEARCH_ALONE) != 0;
    if (N <= (S >= 1024 ? (alone ? 128 : 32) : (alone ? 160 : 64))) return 1;
    return S <= 256 && N > OFK_SPARSE_SEARCH_MAX_CHUNKS ? 4 : 2;
}

template <int S, int COLS>
int launch_beam(const void *scores, const float *bwd, ofk_beam_slot_t *beam, int32_t *states,
                uint8_t *moves, int T, int N, float log_cut, float stay, int flags, const double *lse_table,
                Queue st) {
    const int group = search_group(S, N, flags);
    if (group == 1) {
        queue_kernel((beam_kernel<S, 1, COLS, 0>), dim3(N), dim3(kBeamThreads<S, 1, COLS, 0>), 0, st, static_cast<const _Float16 *>(scores), bwd,
                           nullptr, beam, states, moves, T, N, log_cut, stay, flags, lse_table, LogSeries{});
        return (int)hipGetLastError();
    }
    if constexpr (S <= 256) {
        if (group == 4) {
            queue_kernel((beam_kernel<S, 4, COLS, 0>), dim3((N + 3) / 4), dim3(512), 0, st,
                               static_cast<const _Float16 *>(scores), bwd, nullptr, beam, states, moves, T, N, log_cut,
                               stay, flags, lse_table, LogSeries{});
            return (int)hipGetLastError();
        }
    }
    queue_kernel((beam_kernel<S, 2, COLS, 0>), dim3((N + 1) / 2), dim3(256), 0, st,
                       static_cast<const _Float16 *>(scores), bwd, nullptr, beam, states, moves, T, N, log_cut, stay,
                       flags, lse_table, LogSeries{});
    return (int)hipGetLastError();
}

const LogSeries kSeries = {OFA_LOG_SERIES, OFA_EXP_COEFS};

// search, forward recursion and posterior in one workgroup: CPG chunks of it, FWD waves of recursion each
template <int S, int CPG, int COLS, int FWD>
int launch_beam_forward(const void *scores, const float *bwd, float *post, ofk_beam_slot_t *beam, int32_t *states,
                        uint8_t *moves, int T, int N, float log_cut, float stay, int flags, const double *lse_table,
                        Queue st) {
    queue_kernel((beam_kernel<S, CPG, COLS, FWD>), dim3((N + CPG - 1) / CPG), dim3(kBeamThreads<S, CPG, COLS, FWD>), 0, st,
                       static_cast<const _Float16 *>(scores), bwd, post, beam, states, moves, T, N, log_cut, stay, flags,
                       lse_table, kSeries);
    return (int)hipGetLastError();
}

int dispatch_beam(const void *scores, const float *bwd, ofk_beam_slot_t *beam, int32_t *states, uint8_t *moves,
                  int T, int N, int state_len, int columns, float log_cut, float stay, int flags,
                  const double *lse_table, Queue st) {
    switch (state_len * 8 + columns) {
        case 3 * 8 + 4: return launch_beam<64, 4>(scores, bwd, beam, states, moves, T, N, log_cut, stay, flags, lse_table, st);
        case 4 * 8 + 4: return launch_beam<256, 4>(scores, bwd, beam, states, moves, T, N, log_cut, stay, flags, lse_table, st);
        case 5 * 8 + 4: return launch_beam<1024, 4>(scores, bwd, beam, states, moves, T, N, log_cut, stay, flags, lse_table, st);
        case 3 * 8 + 5: return launch_beam<64, 5>(scores, bwd, beam, states, moves, T, N, log_cut, stay, flags, lse_table, st);
        case 4 * 8 + 5: return launch_beam<256, 5>(scores, bwd, beam, states, moves, T, N, log_cut, stay, flags, lse_table, st);
        case 5 * 8 + 5: return launch_beam<1024, 5>(scores, bwd, beam, states, moves, T, N, log_cut, stay, flags, lse_table, st);
        default: return OFK_BAD_ARGS;
    }
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// The same search with its scratch memory (the persisted beam slots the traceback walks, and the
// log-sum-exp table) in a static device array instead of buffers of a gpubuf: for callers that
// must not allocate.  Every GPU the library runs on holds its own copy of the array until the
// process ends; `scratch` below is only the host-side handle of it, the device address comes
// from hipGetSymbolAddress, once per device.
// ---------------------------------------------------------------------------------------------
namespace {

constexpr size_t kStaticTableBytes = 8192;  // 612 doubles, rounded up
static __device__ __align__(256) unsigned char scratch[kStaticTableBytes + OFK_STATIC_SLOT_BYTES];

constexpr int kMaxDevices = 64;
unsigned char *g_scratch_of[kMaxDevices];  // device address of `scratch` per device, once looked up
std::mutex g_scratch_mutex;

}  // namespace

// Set-up of the static scratch array on the current device: looks up the array's device address and
// copies the log-sum-exp table behind it (a blocking copy).  Once per device; later calls return at once.
extern "C" int ofk_beam_search_static_prepare(const double *lse_table_host) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return OFK_BAD_ARGS;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_of[dev]) return 0;
    if (!lse_table_host) return OFK_BAD_ARGS;
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    e = hipMemcpy(p, lse_table_host, sizeof(double) * OFK_LSE_DOUBLES, hipMemcpyHostToDevice);
    if (e != hipSuccess) return (int)e;
    g_scratch_of[dev] = static_cast<unsigned char *>(p);
    return 0;
}

// 1 if the current device's array has been set up, 0 if not (or if the device cannot be told)
extern "C" int ofk_beam_search_static_ready(void) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    return g_scratch_of[dev] ? 1 : 0;
}

extern "C" int ofk_beam_search_static(const void *scores, const float *bwd, int32_t *states, uint8_t *moves, int T,
                                      int N, int state_len, int columns, float log_beam_cut, float stay, int flags,
                                      void *stream) {
    if (!scores || !bwd || !states || !moves || T < 1 || T > OFK_MAX_T || N < 1) return OFK_BAD_ARGS;
    if ((reinterpret_cast<uintptr_t>(scores) | reinterpret_cast<uintptr_t>(bwd)) & 15u) return OFK_BAD_ARGS;
    if ((size_t)N * (size_t)(T + 1) * kW * sizeof(ofk_beam_slot_t) > (size_t)OFK_STATIC_SLOT_BYTES) return OFK_TOO_LARGE;
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= kMaxDevices) return OFK_BAD_ARGS;
    unsigned char *base;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        base = g_scratch_of[dev];
    }
    if (!base) return OFK_NOT_PREPARED;
    // nothing in the array has to start at zero: the search writes every slot the traceback reads
    ofk_beam_slot_t *beam = reinterpret_cast<ofk_beam_slot_t *>(base + kStaticTableBytes);
    const double *lse_table = reinterpret_cast<const double *>(base);
    const Queue st{static_cast<hipStream_t>(stream), nullptr};
    return dispatch_beam(scores, bwd, beam, states, moves, T, N, state_len, columns, log_beam_cut, stay, flags,
                         lse_table, st);
}

extern "C" int ofk_search_chunks_per_group(int N, int state_len, int flags) { return search_group(1 << (2 * state_len), N, flags); }

extern "C" int ofk_beam_search(const void *scores, const float *bwd, ofk_beam_slot_t *beam, int32_t *states,
                               uint8_t *moves, int T, int N, int state_len, int columns, float log_beam_cut,
                               float stay, const double *lse_table, int flags, void *stream, void *done) {
    if (!scores || !bwd || !beam || !states || !moves || !lse_table || T < 1 || T > OFK_MAX_T || N < 1) return OFK_BAD_ARGS;
    if ((reinterpret_cast<uintptr_t>(scores) | reinterpret_cast<uintptr_t>(bwd) | reinterpret_cast<uintptr_t>(beam)) & 15u)
        return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
    return dispatch_beam(scores, bwd, beam, states, moves, T, N, state_len, columns, log_beam_cut, stay, flags,
                         lse_table, st);
}

extern "C" int ofk_beam_search_forward(const void *scores, const float *bwd, float *post, ofk_beam_slot_t *beam,
                                       int32_t *states, uint8_t *moves, int T, int N, int state_len, int columns,
                                       float log_beam_cut, float stay, const double *lse_table, int flags, void *stream, void *done) {
    if (!scores || !bwd || !post || !beam || !states || !moves || !lse_table || T < 1 || T > OFK_MAX_T || N < 1) return OFK_BAD_ARGS;
    if ((reinterpret_cast<uintptr_t>(scores) | reinterpret_cast<uintptr_t>(bwd) | reinterpret_cast<uintptr_t>(post) |
         reinterpret_cast<uintptr_t>(beam)) & 15u)
        return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
#define OFK_FORWARD(S, CPG, COLS, FWD) \
    return launch_beam_forward<S, CPG, COLS, FWD>(scores, bwd, post, beam, states, moves, T, N, log_beam_cut, stay, flags, lse_table, st)
    const bool dense = N > OFK_SPARSE_SEARCH_MAX_CHUNKS;
    switch (state_len * 8 + columns) {
        case 4 * 8 + 4: if (dense) OFK_FORWARD(256, 2, 4, 2); OFK_FORWARD(256, 2, 4, 4);
        case 4 * 8 + 5: if (dense) OFK_FORWARD(256, 2, 5, 2); OFK_FORWARD(256, 2, 5, 4);
        case 5 * 8 + 4: OFK_FORWARD(1024, 1, 4, 8);
        case 5 * 8 + 5: OFK_FORWARD(1024, 1, 5, 8);
        default: return OFK_BAD_ARGS;
    }
#undef OFK_FORWARD
}
