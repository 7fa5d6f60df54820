// Per-block quality, base calls and phred characters of one chunk per workgroup, gfx950.
//
// Follows the CPU path (reference src/beam_search.c:441-496 for the quality of a
// block, src/beam_search.c:49-99 and src/decode_cpu.c:218-225 for the sequence):
//   1. and 2. a running sum of the moves gives every time step its base position, and the
//      bases of the sequence;
//   3. every time step in parallel: posterior of the path k-mer plus its distinct
//      one-base shifts (fp32 sums in the CPU path's order), clamped, to the power 0.4;
//   4. every base in parallel: the fp32 sums over its dwell are taken in time order,
//      exactly as the serial loop takes them, then the phred character follows.
// pow is evaluated in double and rounded once to fp32.  The phred character is a
// step function of the miss probability 1 - base/total; its 49 thresholds are
// found on the host with the host's own log10f and handed in, so the character
// does not depend on a device log10.
#include <hip/hip_runtime.h>

#include "kernels.h"
#include "queue.h"

namespace {

// The characters of a chunk lie at any address; their copy in LDS lies at the same distance from a multiple of 16, so that whole
// 16-byte pieces move by one store a lane.  Bytes [lo, hi) of the chunk, by the lanes of `lanes` (lane 0 .. lanes - 1).
__device__ __forceinline__ void copy_out(unsigned char *dst, const unsigned char *lds, int lo, int hi, int lane, int lanes) {
    const int skew = (int)(reinterpret_cast<uintptr_t>(dst) & 15u);
    const int first = (lo + skew + 15) & ~15, last = (hi + skew) & ~15;  // whole pieces, counted from dst - skew
    unsigned char *d = dst - skew;
    const unsigned char *l = lds - skew;
    for (int i = first + 16 * lane; i < last; i += 16 * lanes)
        *reinterpret_cast<uint4 *>(d + i) = *reinterpret_cast<const uint4 *>(l + i);
    const int head_end = first < hi + skew ? first : hi + skew;
    const int tail = last > head_end ? last : head_end;
    for (int i = lo + skew + lane; i < head_end; i += lanes) d[i] = l[i];
    for (int i = tail + lane; i < hi + skew; i += lanes) d[i] = l[i];
}

// A posterior that is gathered.  Rows of 256 and 1024 states give a line or two for several values each and none of them again: they
// pass by the caches.  Rows of 64 states are two lines, which nine values share.  Stage inside decodes, us, kept | passed by: 256 chunks
// of 1024 states 84 | 70, 512 of 256 states 131 | 130, 403 of them (T = 1201) 81 | 79, 1024 of 64 states 125 | 182.
template <int S>
__device__ __forceinline__ float gathered(const float *p) {
    if constexpr (S >= 256) return __builtin_nontemporal_load(p);
    else return *p;
}

// LDS of a chunk: two 4-byte tables, a 2-byte one and three of bytes with room for their skews.
constexpr size_t sequence_lds(int T) {
    const size_t t16 = ((size_t)T + 15) & ~(size_t)15;
    return 4 * t16 + 4 * (t16 + 16) + 2 * t16 + 3 * (t16 + 16);
}

// What bounds it: up to a chunk per compute unit the waits of its few dependent rounds of memory accesses, above that the sectors
// that the posteriors are gathered from (0.59 GB with 512 chunks of 256 states, 0.13 ms at 4.5 TB/s).  All that does not need
// the posteriors comes first: base positions, the characters of the sequence and the zeros behind both strings, which one wave
// then writes to their place (host memory, in a decode) while the others gather.  What is left after the gathers is a base's
// character.  Inside decodes, ms, against gathers first, bytes last and one at a time, 256 lanes: 1 chunk of 64 states 0.021 ->
// 0.014; 512 of 256 states 0.167 -> 0.130, 1024 of them 0.328 -> 0.263; 256 of 1024 0.103 -> 0.084 (0.070 past the caches).
template <int S, int kThreads>
__global__ __launch_bounds__(kThreads) void sequence_kernel(
    const float *__restrict__ post, int32_t *__restrict__ states, const uint8_t *__restrict__ moves,
    float *__restrict__ qual_data, float *__restrict__ base_probs, float *__restrict__ total_probs,
    char *__restrict__ sequence, char *__restrict__ qstring, int T, ofk_phred_table_t phred,
    const float *__restrict__ path_sums, uint8_t *__restrict__ moves_out) {
    constexpr int kWaves = kThreads / 64;
    constexpr int kGather = kThreads - 64;  // the last wave writes the finished bytes
    static_assert(OFK_MAX_T <= 128 * 64, "two counts of moves to a lane");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    __shared__ int s_count[128];  // moves of every 64 time steps
    const int t16 = (T + 15) & ~15;
    const int n = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t first = (size_t)n * T;
    unsigned char *out_seq = reinterpret_cast<unsigned char *>(sequence) + first;
    unsigned char *out_qual = reinterpret_cast<unsigned char *>(qstring) + first;
    unsigned char *out_moves = moves_out + first;
    float *s_prob = reinterpret_cast<float *>(lds);                        // [T] called-base probability
    int *s_start = reinterpret_cast<int *>(s_prob + t16);                  // [T+1] first time step of base p
    uint16_t *s_state = reinterpret_cast<uint16_t *>(s_start + t16 + 16);  // [T]
    unsigned char *bytes = reinterpret_cast<unsigned char *>(s_state + t16);
    unsigned char *s_seq = bytes + (reinterpret_cast<uintptr_t>(out_seq) & 15u);                    // [T]
    unsigned char *s_qual = bytes + t16 + 16 + (reinterpret_cast<uintptr_t>(out_qual) & 15u);       // [T]
    unsigned char *s_move = bytes + 2 * (t16 + 16) + (reinterpret_cast<uintptr_t>(out_moves) & 15u);  // [T]

    const float *post_n = post + (size_t)n * (size_t)(T + 1) * S;
    int32_t *st_n = states + first;
    const uint8_t *mv_n = moves + first;

    // 1. moves of every 64 time steps
    const int pieces = (T + 63) / 64;
    for (int e = wave; e < pieces; e += kWaves) {
        const int t = 64 * e + lane;
        uint8_t move = 0;
        if (t < T) {
            const int st = st_n[t];
            move = mv_n[t];
            s_state[t] = (uint16_t)st;
            s_move[t] = move;
            st_n[t] = st & 3;
        }
        const uint64_t mask = __ballot(move != 0);
        if (lane == 0) s_count[e] = __popcll(mask);
    }
    __syncthreads();

    // 2. base position of every time step, and what follows from the path alone.  Every wave takes the running sum of
    // the counts by itself: lane i those of pieces i and 64 + i.
    int low = lane < pieces ? s_count[lane] : 0, high = 64 + lane < pieces ? s_count[64 + lane] : 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int l = __shfl_up(low, d), h = __shfl_up(high, d);
        low += lane >= d ? l : 0;
        high += lane >= d ? h : 0;
    }
    high += __builtin_amdgcn_readlane(low, 63);
    const int seq_len = __builtin_amdgcn_readlane(high, 63);
    for (int e = wave; e < pieces; e += kWaves) {
        const int t = 64 * e + lane;
        const bool begins = t < T && s_move[t] != 0;
        const uint64_t mask = __ballot(begins);
        const int before = e == 0 ? 0 : e <= 64 ? __builtin_amdgcn_readlane(low, e - 1) : __builtin_amdgcn_readlane(high, e - 65);
        if (begins) {
            const int pos = before + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            s_start[pos] = t;
            s_seq[pos] = "ACGT"[s_state[t] & 3];
        }
        if (t < T && t >= seq_len) {
            s_seq[t] = 0;
            s_qual[t] = 0;
        }
    }
    if (tid == 0) s_start[seq_len] = T;
    __syncthreads();

    // 3. one wave writes what is known, the others take the quality of every block
    if (wave == kWaves - 1) {
        copy_out(out_seq, s_seq, 0, T, lane, 64);
        copy_out(out_qual, s_qual, seq_len, T, lane, 64);
        if (moves_out) copy_out(out_moves, s_move, 0, T, lane, 64);
    } else {
        for (int t = tid; t < T; t += kGather) {
            const int st = s_state[t];
            const int base = st & 3;
            float prob;
            if (path_sums) {  // the sum below, taken for every state by path_sums_kernel: one read instead of nine
                prob = path_sums[(first + t) * S + st];
            } else {
                const float *p = post_n + (size_t)(t + 1) * S;
                prob = gathered<S>(p + st);
                int nb[8];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    nb[2 * b] = (st >> 2) + (S / 4) * b;
                    nb[2 * b + 1] = ((st << 2) & (S - 1)) + b;
                }
                float x[8];  // all in flight together
#pragma unroll
                for (int k = 0; k < 8; ++k) x[k] = gathered<S>(p + nb[k]);
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    bool fresh = nb[k] != st;
#pragma unroll
                    for (int m = 0; m < k; ++m) fresh = fresh && nb[m] != nb[k];
                    const float with = prob + x[k];
                    prob = fresh ? with : prob;
                }
            }
            if (prob > 1.0f) prob = 1.0f;
            else if (prob < 0.0f) prob = 0.0f;
            prob = (float)pow((double)prob, (double)0.4f);
            const float wrong = (1.0f - prob) / 3.0f;
            s_prob[t] = prob;
            float4 q;
            q.x = base == 0 ? prob : wrong;
            q.y = base == 1 ? prob : wrong;
            q.z = base == 2 ? prob : wrong;
            q.w = base == 3 ? prob : wrong;
            reinterpret_cast<float4 *>(qual_data)[first + t] = q;
        }
    }
    __syncthreads();

    // 4. one base per thread
    for (int p = tid; p < T; p += kThreads) {
        const size_t o = first + p;
        if (p >= seq_len) {
            base_probs[o] = 0.f;
            total_probs[o] = 0.f;
            continue;
        }
        const int t0 = s_start[p], t1 = s_start[p + 1];
        float bp = 0.f, tp = 0.f;
        for (int t = t0; t < t1; ++t) {
            const float prob = s_prob[t], wrong = (1.0f - prob) / 3.0f;
            const int base = s_state[t] & 3;
            bp += prob;
            tp += base == 0 ? prob : wrong;
            tp += base == 1 ? prob : wrong;
            tp += base == 2 ? prob : wrong;
            tp += base == 3 ? prob : wrong;
        }
        const float miss = 1.0f - (bp / tp);
        int ch = 83;
#pragma unroll
        for (int j = 0; j < OFK_PHRED_STEPS; ++j) ch -= miss >= phred.thr[j] ? 1 : 0;
        if (miss != miss) ch = 0;
        s_qual[p] = (unsigned char)ch;
        base_probs[o] = -10.0f * (float)log10((double)miss);  // diagnostic copy, not used for the character
        total_probs[o] = tp;
    }
    __syncthreads();
    copy_out(out_qual, s_qual, 0, seq_len, tid, kThreads);
}


// ---------------------------------------------------------------------------------------------
// For every chunk, time step and state: the posterior of the k-mer plus that of its distinct
// one-base shifts, summed in the CPU path's order -- what step 3 of sequence_kernel gathers for
// the one state on the path.  Those nine scattered reads per time step fetch about half of the
// posteriors, 64 bytes for every 4 wanted, and made up most of that kernel's time; they come
// after the beam search, which leaves most of the machine idle for a millisecond.  This kernel
// runs beside the search, reads every row once, in order, and the sequence stage then takes one
// value per time step.
//
// A wave owns whole rows (four at a time with 64 states) and keeps the current one in LDS, 256
// floats per 64 lanes; lane j holds states 4j .. 4j+3 of each 256.  Those four share their
// four predecessors (st >> 2) + b * S/4, and the successors 4 * (st mod S/4) + b of a state are
// four neighbours in the row: eight LDS reads per lane cover all 32 values.  Which of a state's
// eight neighbours count (not the state itself, not an earlier neighbour) does not depend on
// the time step and is worked out once per lane.  A wave's LDS operations complete in order, so
// the waves of a group never wait for each other.
// ---------------------------------------------------------------------------------------------
template <int S>
__global__ __launch_bounds__(256) void path_sums_kernel(const float *__restrict__ post, float *__restrict__ sums,
                                                        int T, long rows) {
    constexpr int Q = S / 4;
    constexpr int G = S >= 256 ? S / 256 : 1;       // float4 pieces of a row per lane
    constexpr int kRowsPerTile = S >= 256 ? 1 : 4;  // rows a wave takes at a time
    constexpr int kTile = S >= 256 ? S : 256;       // floats
    __shared__ __attribute__((aligned(16))) float tiles[4][kTile];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float *tile = tiles[wave];
    const int sub = S >= 256 ? 0 : lane >> 4;           // row of the tile this lane works on
    const int j0 = S >= 256 ? lane : lane & 15;         // quad of states within 256 (within the row, with 64 states)
    float *row = tile + (S >= 256 ? 0 : 64 * sub);      // this lane's row in LDS

    // per state: which neighbours are added (bit k: neighbour k, predecessors at even k)
    uint32_t fresh[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int st = 4 * (j0 + 64 * g) + i;
            int nb[8];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                nb[2 * b] = (st >> 2) + Q * b;
                nb[2 * b + 1] = ((st << 2) & (S - 1)) + b;
            }
            uint32_t bits = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                bool f = nb[k] != st;
#pragma unroll
                for (int m = 0; m < k; ++m) f = f && nb[m] != nb[k];
                bits |= f ? 1u << k : 0u;
            }
            fresh[g][i] = bits;
        }
    }

    const long tiles_n = (rows + kRowsPerTile - 1) / kRowsPerTile;
    const long step = (long)gridDim.x * 4;
    long tix = (long)blockIdx.x * 4 + wave;
    // row r of the output is time step r % T of chunk r / T and reads row r % T + 1 of that chunk's posteriors
    auto in_row = [&](long r) { return post + ((size_t)(r / T) * (size_t)(T + 1) + (size_t)(r % T) + 1) * S; };
    float4 cur[G], nxt[G];
    auto fetch = [&](long t_ix, float4 (&v)[G]) {
        const long r = t_ix * kRowsPerTile + sub;
#pragma unroll
        for (int g = 0; g < G; ++g)
            v[g] = (t_ix < tiles_n && r < rows) ? *reinterpret_cast<const float4 *>(in_row(r) + 4 * (j0 + 64 * g))
                                                : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    fetch(tix, cur);
    for (; tix < tiles_n; tix += step) {
        fetch(tix + step, nxt);
#pragma unroll
        for (int g = 0; g < G; ++g) *reinterpret_cast<float4 *>(row + 4 * (j0 + 64 * g)) = cur[g];
        __builtin_amdgcn_wave_barrier();
        const long r = tix * kRowsPerTile + sub;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int j = j0 + 64 * g;  // the lane's states 4j .. 4j+3 share their predecessors j + b * Q
            float prev[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) prev[b] = row[j + Q * b];
            const float own[4] = {cur[g].x, cur[g].y, cur[g].z, cur[g].w};
            float out[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int st = 4 * j + i;
                const float4 nx = *reinterpret_cast<const float4 *>(row + 4 * (st & (Q - 1)));
                const float next[4] = {nx.x, nx.y, nx.z, nx.w};
                float prob = own[i];  // fp32 sums in the CPU path's order
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float with_prev = prob + prev[b];
                    prob = (fresh[g][i] >> (2 * b)) & 1u ? with_prev : prob;
                    const float with_next = prob + next[b];
                    prob = (fresh[g][i] >> (2 * b + 1)) & 1u ? with_next : prob;
                }
                out[i] = prob;
            }
            if (r < rows)
                *reinterpret_cast<float4 *>(sums + (size_t)r * S + 4 * j) = make_float4(out[0], out[1], out[2], out[3]);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int g = 0; g < G; ++g) cur[g] = nxt[g];
    }
}

template <int S>
int launch_path_sums(const float *post, float *sums, int T, int N, Queue st) {
    const long rows = (long)N * T;
    // Half as many workgroups as chunks, up to one per compute unit (one wave per SIMD): with 512
    // chunks of 256 states the kernel then ends well inside the beam search it runs beside and does
    // not slow it (measured: 256 groups 1.185 ms of search against 1.183 alone, 512 groups 1.195,
    // 1024 groups 1.27; 128 groups outlast the search).
    int wgs = N / 2;
    wgs = wgs < 64 ? 64 : (wgs > 256 ? 256 : wgs);
    queue_kernel((path_sums_kernel<S>), dim3(wgs), dim3(256), 0, st, post, sums, T, rows);
    return (int)hipGetLastError();
}

template <int S, int kThreads>
int launch_sequence_with(const float *post, int32_t *states, const uint8_t *moves, float *qual_data,
                         float *base_probs, float *total_probs, char *sequence, char *qstring, int T, int N,
                         const ofk_phred_table_t &phred, const float *path_sums, uint8_t *moves_out, Queue st) {
    const size_t lds = sequence_lds(T);
    if (lds > 64 * 1024 - 1024) {  // beyond the default limit of dynamic LDS; the compute unit has 160 KB
        const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void *>(&sequence_kernel<S, kThreads>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (rc != hipSuccess) return (int)rc;
    }
    queue_kernel((sequence_kernel<S, kThreads>), dim3(N), dim3(kThreads), lds, st, post, states, moves, qual_data,
                       base_probs, total_probs, sequence, qstring, T, phred, path_sums, moves_out);
    return (int)hipGetLastError();
}

template <int S>
int launch_sequence(const float *post, int32_t *states, const uint8_t *moves, float *qual_data,
                    float *base_probs, float *total_probs, char *sequence, char *qstring, int T, int N,
                    const ofk_phred_table_t &phred, const float *path_sums, uint8_t *moves_out, Queue st) {
    // Up to a chunk per compute unit, 960 gathering lanes (two time steps each at T = 1666, nine at 8192): the rounds of memory accesses
    // are what is waited for.  Beyond, two workgroups of half the size fill a unit and one's gathers run beside the other's characters.
    // 1024 | 512 | 256 lanes, us: 16 chunks of 64 states 14 | 17 | 25, 256 of 1024 84 | 86 | 92, 512 of 256 131 | 129 | 145, 1024 of 256
    // 270 | 263 | 283.
    if (N <= 256)
        return launch_sequence_with<S, 1024>(post, states, moves, qual_data, base_probs, total_probs, sequence, qstring, T, N, phred,
                                             path_sums, moves_out, st);
    return launch_sequence_with<S, 512>(post, states, moves, qual_data, base_probs, total_probs, sequence, qstring, T, N, phred,
                                        path_sums, moves_out, st);
}

}  // namespace

extern "C" int ofk_path_sums(const float *post, float *sums, int T, int N, int state_len, void *stream, void *done) {
    if (!post || !sums || T < 1 || N < 1) return OFK_BAD_ARGS;
    if ((reinterpret_cast<uintptr_t>(post) | reinterpret_cast<uintptr_t>(sums)) & 15u) return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
    switch (state_len) {
        case 3: return launch_path_sums<64>(post, sums, T, N, st);
        case 4: return launch_path_sums<256>(post, sums, T, N, st);
        case 5: return launch_path_sums<1024>(post, sums, T, N, st);
        default: return OFK_BAD_ARGS;
    }
}

extern "C" int ofk_sequence(const float *post, int32_t *states, const uint8_t *moves, float *qual_data,
                            float *base_probs, float *total_probs, char *sequence, char *qstring, int T, int N,
                            int state_len, const ofk_phred_table_t *phred, const float *path_sums, uint8_t *moves_out,
                            void *stream, void *done) {
    // the per-chunk tables live in LDS: 13 bytes per time step
    if ((!post && !path_sums) || !states || !moves || !qual_data || !base_probs || !total_probs || !sequence || !qstring ||
        !phred || T < 1 || T > OFK_MAX_T || N < 1)
        return OFK_BAD_ARGS;
    if (reinterpret_cast<uintptr_t>(qual_data) & 15u) return OFK_BAD_ARGS;
    const Queue st{static_cast<hipStream_t>(stream), static_cast<hipEvent_t>(done)};
    switch (state_len) {
        case 3: return launch_sequence<64>(post, states, moves, qual_data, base_probs, total_probs, sequence, qstring, T, N, *phred, path_sums, moves_out, st);
        case 4: return launch_sequence<256>(post, states, moves, qual_data, base_probs, total_probs, sequence, qstring, T, N, *phred, path_sums, moves_out, st);
        case 5: return launch_sequence<1024>(post, states, moves, qual_data, base_probs, total_probs, sequence, qstring, T, N, *phred, path_sums, moves_out, st);
        default: return OFK_BAD_ARGS;
    }
}
