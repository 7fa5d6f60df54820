/*
 * Host side of the MI355X decoder: the public openfish entry points and the
 * stage-level C-ABI, in C, above the kernel launchers of kernels.h.
 *
 * One decode is one of three arrangements of the same stages (the beam search needs only scores and bwd, the
 * posterior only feeds the quality stage, reference src/beam_search.c:193,450):
 *   split    bwd scan -> { beam search || fwd scan + posterior } -> sequence
 *   merged   bwd scan -> beam search with the fwd scan and the posterior in its workgroups -> sequence
 *   one      both scans + posterior in one kernel -> { beam search || per-state sums of posteriors } -> sequence
 * Every call chooses (arrangement_by_default) unless the gpubuf says which.  The sequence stage
 * writes bases and qualities into pinned host memory itself.  Errors follow the reference convention
 * (reference src/hip_utils.h:11-28, src/error.h:44-72): message on stderr, then exit.
 */
#include <errno.h>
#include <float.h>
#include <math.h>
#include <pthread.h>
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#include <openfish/openfish.h>
#include <openfish/openfish_amd.h>
#include <openfish/openfish_error.h>

#include "kernels.h"

/* ---- logging (reference src/error.c:33-41) -------------------------------- */

static enum openfish_log_level_opt g_log_level = OPENFISH_LOG_VERB;

enum openfish_log_level_opt get_openfish_log_level(void) { return g_log_level; }
void set_openfish_log_level(enum openfish_log_level_opt level) { g_log_level = level; }

void openfish_log_emit(enum openfish_log_level_opt need, const char *tag, const char *colour,
                       const char *func, const char *file, int line, int where, const char *fmt, ...) {
    if (g_log_level < need) return;
    va_list ap;
    if (colour) fprintf(stderr, "[%s::%s]%s ", func, tag, colour);
    else fprintf(stderr, "[%s] %s: ", tag, func);
    va_start(ap, fmt);
    vfprintf(stderr, fmt, ap);
    va_end(ap);
    if (colour) fputs("\033[0m", stderr);
    if (where) fprintf(stderr, " At %s:%d", file, line);
    fputc('\n', stderr);
}

/* ---- error convention ------------------------------------------------------ */

#define HIP_OK(call)                                                                              \
    do {                                                                                          \
        hipError_t e_ = (call);                                                                   \
        if (e_ != hipSuccess) {                                                                   \
            fprintf(stderr, "HIP error: %s, in file: %s, line number: %d\n", hipGetErrorString(e_), \
                    __FILE__, __LINE__);                                                          \
            exit(1);                                                                              \
        }                                                                                         \
    } while (0)

static void die(const char *what) {
    OPENFISH_ERROR("%s", what);
    exit(EXIT_FAILURE);
}

static void launch_ok(int rc, const char *kernel) {
    if (rc == 0) return;
    if (rc == OFK_BAD_ARGS) fprintf(stderr, "openfish: %s: arguments do not fit the kernel (shape, alignment or state_len)\n", kernel);
    else fprintf(stderr, "HIP error: %s, launching %s\n", hipGetErrorString((hipError_t)rc), kernel);
    exit(1);
}

static void *host_alloc(size_t bytes) {
    void *p = malloc(bytes ? bytes : 1);
    if (!p) {
        fprintf(stderr, "openfish: out of host memory (%zu bytes)\n", bytes);
        exit(EXIT_FAILURE);
    }
    return p;
}

/* ---- table of log(1 + e^-gap) for the beam search's merges -------------------
 *
 * The CPU path folds two scores with log(1.0 + exp(-gap)) in double (reference
 * src/beam_search.c:43-47).  On the device that value is read off a piecewise
 * polynomial: per cell of width 1/4 the degree-8 interpolant through the Chebyshev
 * nodes, fitted here in long double.  The interpolation error is below 1e-15, far
 * under the 2^-46 at which a folded fp32 score could round differently.
 */

static void build_lse_table(double *tab) {
    const int n = OFK_LSE_COEFS; /* nodes = coefficients */
    const long double pi = 3.14159265358979323846264338327950288L;
    for (int cell = 0; cell < OFK_LSE_CELLS; ++cell) {
        const long double centre = 0.25L * cell + 0.125L;
        long double x[OFK_LSE_COEFS], dd[OFK_LSE_COEFS], mono[OFK_LSE_COEFS], basis[OFK_LSE_COEFS];
        for (int j = 0; j < n; ++j) {
            x[j] = cosl(pi * (2 * j + 1) / (2.0L * n)); /* s in [-1, 1], gap = centre + s / 8 */
            dd[j] = log1pl(expl(-(centre + x[j] / 8.0L)));
        }
        for (int k = 1; k < n; ++k) /* Newton divided differences */
            for (int j = n - 1; j >= k; --j) dd[j] = (dd[j] - dd[j - 1]) / (x[j] - x[j - k]);
        for (int j = 0; j < n; ++j) mono[j] = 0, basis[j] = 0;
        basis[0] = 1; /* basis = prod_{m<k} (s - x[m]) as monomials */
        for (int k = 0; k < n; ++k) {
            for (int j = 0; j < n; ++j) mono[j] += dd[k] * basis[j];
            for (int j = n - 1; j >= 1; --j) basis[j] = basis[j - 1] - x[k] * basis[j];
            basis[0] = -x[k] * basis[0];
        }
        for (int j = 0; j < n; ++j) tab[cell * n + j] = (double)mono[j];
    }
}

void openfish_amd_lse_table(double *out) { build_lse_table(out); }

/* ---- gpubuf ---------------------------------------------------------------- */

/* Bytes of moves from which they travel beside the sequence stage; fewer are not worth three calls and a launch more (whole calls, us, by a
 * copy | by the stage: 5 chunks of 32 steps 80 | 75; 16 of 64 states, T = 1666 1298 | 1287; 64 1315 | 1307; 150 of 256 1602 | 1610). */
#define OFA_COPY_MOVES ((size_t)131072)

#define OFA_MAGIC 0x6f66616d64677075ull /* "ofamdgpu" */

enum { EV_JOIN, EV_START, EV_BWD_END, EV_BEAM_END, EV_FWD_END, EV_FWD_SCAN_END, EV_SEQ_END, EV_SUMS_END, EV_MOVES, EV_TAIL, EV_SIDE_TAIL, EV_COUNT };
/* The events between kernels are carried by the kernels whose end they mark (queue.h); with both sweeps in one kernel EV_BWD_END is its
 * end and EV_FWD_END is not used, EV_FWD_SCAN_END only where the forward sweep runs beside the backward one.  EV_START, EV_MOVES and the
 * two tails are markers. */

/* arrangements of the scans: both sweeps in one kernel; backward sweep, then forward sweep beside the beam search;
 * backward sweep, then forward sweep within the beam search's kernel */
enum { ARR_ONE = 0, ARR_SPLIT = 1, ARR_MERGED = 2 };

typedef struct {
    openfish_gpubuf_t pub; /* first: the pointer handed to callers is this struct */
    unsigned long long magic;
    int T, N, state_len;
    void *slab;            /* one device allocation behind all pub fields */
    float *path_sums;      /* N x T x states: per state, the posteriors a block's quality is made of, summed */
    unsigned char *h_out;  /* pinned host memory for moves | sequence | qstring */
    unsigned char *d_out;  /* the same memory as the device addresses it */
    double *lse_table;     /* device copy of the log(1 + e^-gap) table */
    int device;
    hipStream_t s_main, s_side; /* of the decode under way; shared with other gpubufs of the device, see take_main_lane */
    int main_lane, side_lane; /* side_lane -1: none */
    hipEvent_t ev[EV_COUNT];
    float ms[OPENFISH_AMD_STAGE_COUNT];
    int timed;
    int pending;           /* a decode has been enqueued and not yet waited for */
    int pend_T, pend_N, pend_sums;    /* its shape */
    int pend_copy;         /* its moves travel by a copy on the side lane */
    int pend_split;        /* how its scans were queued (which events were recorded): ARR_* */
    int pend_apart;        /* split, with the forward sweep beside the backward one */
    int scan_mode;         /* OFK_SCAN_*: arithmetic of the scans of this gpubuf's decodes */
    int scan_spl;          /* states per lane of the scans, 0 = chosen from the batch size */
    int debug_flags;       /* bit 0: serial replay of the beam search's merges; bit 1: colliding seed hashes */
    int split_scans;       /* the arrangement asked for: ARR_*, or -1 (default): chosen per call */
    ofk_phred_table_t phred; /* thresholds for (phred_shift, phred_scale) */
    float phred_shift, phred_scale;
    int phred_valid;
} ofa_gpubuf_t;

static size_t round_up(size_t x) { return (x + 255) & ~(size_t)255; }

static int states_of(int state_len) { return 1 << (2 * state_len); }

static void check_state_len(int state_len) {
    if (state_len < 3 || state_len > 5) die("state_len must be 3, 4 or 5 (64, 256 or 1024 states)");
}

/* ---- streams ----------------------------------------------------------------
 *
 * A process has a handful of hardware queues (four unless the environment says otherwise, one of them the null
 * stream's) and the runtime deals its streams round them; kernels of one queue run one after another whatever
 * streams they are on, and what waits for an event holds up all that is behind it in its queue.  With two streams
 * per gpubuf, created without regard to that, one gpubuf in four or so had both in one queue (its split decodes ran
 * the forward sweep after the search: 512 chunks of 256 states 2.55 ms instead of 2.24, 37 of 1024 states with
 * T = 833 2.29 instead of 1.70), and two batches in flight could share one queue (512 chunks each: 4.35 ms for the
 * two instead of 3.67) or one of them the null stream's, which every decode starts with a look at.
 *
 * So the gpubufs of a device share three streams in three queues, none of them the null stream's.  A decode takes the
 * least loaded for its kernels and, for what runs beside them (forward sweep, sums, a copy), the least loaded of the
 * other two.  Nothing in the API tells the queue of a stream, but it stays the same for its life: every
 * new stream is tried against the null stream and those found before it (ofk_meet, 0.03 ms a try), and held if it
 * will not do, so that the next goes elsewhere.  Where three queues are not to be found (fewer allowed, or too busy to
 * start two kernels within the time of a try) the gpubufs make do with what there is; only speed depends on it.
 * The streams are created with a device's first gpubuf and destroyed with its last.  Waits of the host are for events
 * of the decode in question, never for a stream. */
#define OFA_LANES 3
#define OFA_LANE_TRIES 8
#define OFA_MAX_DEVICES 64
typedef struct {
    hipStream_t stream[OFA_LANES];
    int load[OFA_LANES]; /* 2 for every decode whose kernels are there, 1 for every one with something beside them */
    int last;            /* where the last decode's kernels went */
    int gpubufs;         /* that use them */
} ofa_lanes_t;
static ofa_lanes_t g_lanes[OFA_MAX_DEVICES];
static pthread_mutex_t g_lanes_mutex = PTHREAD_MUTEX_INITIALIZER;

static int run_side_by_side(hipStream_t a, hipStream_t b, volatile int *h_mark, int *d_mark) {
    h_mark[0] = h_mark[1] = 0;
    launch_ok(ofk_meet(d_mark, 1, a), "meet");
    launch_ok(ofk_meet(d_mark, 0, b), "meet");
    HIP_OK(hipStreamSynchronize(a));
    HIP_OK(hipStreamSynchronize(b));
    return h_mark[1];
}

/* mark: eight bytes of pinned memory, as host and device address them */
static void find_lanes(ofa_lanes_t *l, volatile int *h_mark, int *d_mark) {
    hipStream_t other[OFA_LANE_TRIES];
    int found = 0, others = 0;
    while (found < OFA_LANES && found + others < OFA_LANE_TRIES) {
        hipStream_t s;
        HIP_OK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        int apart = run_side_by_side(NULL, s, h_mark, d_mark);
        for (int i = 0; apart && i < found; ++i) apart = run_side_by_side(l->stream[i], s, h_mark, d_mark);
        if (apart) l->stream[found++] = s;
        else other[others++] = s;
    }
    while (found < OFA_LANES) l->stream[found++] = other[--others];
    while (others > 0) HIP_OK(hipStreamDestroy(other[--others]));
}

static void open_lanes(ofa_gpubuf_t *g) {
    HIP_OK(hipGetDevice(&g->device));
    if (g->device < 0 || g->device >= OFA_MAX_DEVICES) die("gpubuf: device number out of range");
    ofa_lanes_t *l = &g_lanes[g->device];
    pthread_mutex_lock(&g_lanes_mutex);
    if (l->gpubufs++ == 0) find_lanes(l, (volatile int *)g->h_out, (int *)g->d_out);
    pthread_mutex_unlock(&g_lanes_mutex);
}

static void close_lanes(ofa_gpubuf_t *g) {
    ofa_lanes_t *l = &g_lanes[g->device];
    pthread_mutex_lock(&g_lanes_mutex);
    if (--l->gpubufs == 0)
        for (int i = 0; i < OFA_LANES; ++i) HIP_OK(hipStreamDestroy(l->stream[i]));
    pthread_mutex_unlock(&g_lanes_mutex);
}

/* the least loaded lane other than `taken`, of equals the first after `last` */
static int least_loaded(const ofa_lanes_t *l, int last, int taken) {
    int best = -1;
    for (int k = 1; k <= OFA_LANES; ++k) {
        const int i = (last + k) % OFA_LANES;
        if (i != taken && (best < 0 || l->load[i] < l->load[best])) best = i;
    }
    return best;
}

/* A lane for the kernels of a decode.  Returns whether another decode is under way on the device. */
static int take_main_lane(ofa_gpubuf_t *g) {
    ofa_lanes_t *l = &g_lanes[g->device];
    pthread_mutex_lock(&g_lanes_mutex);
    int others = 0;
    for (int i = 0; i < OFA_LANES; ++i) others |= l->load[i] > 0;
    g->main_lane = l->last = least_loaded(l, l->last, -1);
    g->side_lane = -1;
    l->load[g->main_lane] += 2;
    g->s_main = l->stream[g->main_lane];
    pthread_mutex_unlock(&g_lanes_mutex);
    return others;
}

/* another one for what runs beside them */
static void take_side_lane(ofa_gpubuf_t *g) {
    ofa_lanes_t *l = &g_lanes[g->device];
    pthread_mutex_lock(&g_lanes_mutex);
    g->side_lane = least_loaded(l, g->main_lane, g->main_lane);
    l->load[g->side_lane] += 1;
    g->s_side = l->stream[g->side_lane];
    pthread_mutex_unlock(&g_lanes_mutex);
}

static void leave_lanes(ofa_gpubuf_t *g) {
    ofa_lanes_t *l = &g_lanes[g->device];
    pthread_mutex_lock(&g_lanes_mutex);
    l->load[g->main_lane] -= 2;
    if (g->side_lane >= 0) l->load[g->side_lane] -= 1;
    pthread_mutex_unlock(&g_lanes_mutex);
}

openfish_gpubuf_t *openfish_gpubuf_init(const int T, const int N, const int state_len) {
    check_state_len(state_len);
    if (T < 1 || N < 1) die("gpubuf: T and N must be positive");
    if (T > OFK_MAX_T) die("gpubuf: chunks longer than 8192 time steps are not supported");
    const size_t S = (size_t)states_of(state_len), nt = (size_t)N * (size_t)T;
    const size_t tens = sizeof(float) * (size_t)N * (size_t)(T + 1) * S;
    ofa_gpubuf_t *g = (ofa_gpubuf_t *)host_alloc(sizeof *g);
    memset(g, 0, sizeof *g);
    g->magic = OFA_MAGIC;
    g->T = T;
    g->N = N;
    g->state_len = state_len;
    g->split_scans = -1;

    /* field sizes as in the reference (src/decode_hip.hip:24-48) except beam_vector,
     * whose slots are 2 bytes here */
    const size_t sz[11] = {tens, tens, nt, nt, nt,
                           sizeof(ofk_beam_slot_t) * (size_t)N * OFK_BEAM_WIDTH * (size_t)(T + 1),
                           sizeof(int32_t) * nt, sizeof(float) * 4 * nt, sizeof(float) * nt, sizeof(float) * nt,
                           /* path_sums, not a field of the reference's struct; see enqueue_decode */
                           (state_len <= 4 ? sizeof(float) * S * (size_t)T * (size_t)(N < OFK_SPARSE_SEARCH_MAX_CHUNKS ? N : OFK_SPARSE_SEARCH_MAX_CHUNKS) : 0)};
    size_t total = 0;
    for (int i = 0; i < 11; ++i) total += round_up(sz[i]);
    HIP_OK(hipMalloc(&g->slab, total));
    unsigned char *p = (unsigned char *)g->slab;
    void **field[11] = {(void **)&g->pub.bwd_NTC, (void **)&g->pub.post_NTC, (void **)&g->pub.moves,
                        (void **)&g->pub.sequence, (void **)&g->pub.qstring, &g->pub.beam_vector,
                        &g->pub.states, (void **)&g->pub.qual_data, (void **)&g->pub.base_probs,
                        (void **)&g->pub.total_probs, (void **)&g->path_sums};
    for (int i = 0; i < 11; ++i) {
        *field[i] = sz[i] ? p : NULL;
        p += round_up(sz[i]);
    }
    /* coherent: what kernels write there is in host memory when their end is seen, with no marker behind them */
    HIP_OK(hipHostMalloc((void **)&g->h_out, 3 * nt < 64 ? 64 : 3 * nt, hipHostMallocCoherent));
    HIP_OK(hipHostGetDevicePointer((void **)&g->d_out, g->h_out, 0));
    {
        double tab[OFK_LSE_DOUBLES];
        build_lse_table(tab);
        HIP_OK(hipMalloc((void **)&g->lse_table, sizeof tab));
        HIP_OK(hipMemcpy(g->lse_table, tab, sizeof tab, hipMemcpyHostToDevice));
    }
    open_lanes(g);
    for (int i = 0; i < EV_COUNT; ++i) HIP_OK(hipEventCreate(&g->ev[i]));
    return &g->pub;
}

/* until every kernel and copy of the enqueued decode is done */
static void wait_for_decode(ofa_gpubuf_t *g) {
    if (g->pend_copy) HIP_OK(hipEventSynchronize(g->ev[EV_MOVES]));
    HIP_OK(hipEventSynchronize(g->ev[EV_SEQ_END])); /* the main lane has waited for what ran on the side lane */
    leave_lanes(g);
}

void openfish_gpubuf_free(openfish_gpubuf_t *gpubuf) {
    ofa_gpubuf_t *g = (ofa_gpubuf_t *)gpubuf;
    if (!g) return;
    if (g->magic != OFA_MAGIC) die("gpubuf was not created by openfish_gpubuf_init");
    if (g->pending) { /* an enqueued decode still reads and writes these buffers */
        wait_for_decode(g);
    }
    for (int i = 0; i < EV_COUNT; ++i) HIP_OK(hipEventDestroy(g->ev[i]));
    close_lanes(g);
    HIP_OK(hipHostFree(g->h_out));
    HIP_OK(hipFree(g->lse_table));
    HIP_OK(hipFree(g->slab));
    g->magic = 0;
    free(g);
}

static ofa_gpubuf_t *checked(const openfish_gpubuf_t *gpubuf, int T, int N, int state_len) {
    ofa_gpubuf_t *g = (ofa_gpubuf_t *)gpubuf;
    if (!g || g->magic != OFA_MAGIC) die("gpubuf was not created by openfish_gpubuf_init");
    if (state_len != g->state_len || (size_t)N * (size_t)(T + 1) > (size_t)g->N * (size_t)(g->T + 1) ||
        (size_t)N * (size_t)T > (size_t)g->N * (size_t)g->T)
        die("batch shape exceeds the shape the gpubuf was created for");
    if (g->pending) die("this gpubuf holds an enqueued decode that has not been waited for");
    return g;
}

/* Scores carry, per state, the four step columns, or five with a blank/stay column first (as a
 * CRF head emits them before the blank is dropped).  The kernels read either layout where it
 * lies and never look at the blank column: the stay score is options->blank_score, as for any
 * other input (reference src/beam_search.c:213). */
static void check_scores(int T, int N, int C, const void *scores, int state_len, const openfish_opt_t *opt) {
    check_state_len(state_len);
    if (T < 1 || N < 1) die("T and N must be positive");
    if (T > OFK_MAX_T) die("chunks longer than 8192 time steps are not supported");
    if (C != 4 * states_of(state_len) && C != 5 * states_of(state_len))
        die("C must be 4 * 4^state_len (one score per state and dropped base) or 5 * 4^state_len (a blank "
            "column first)");
    if (!scores) die("scores_TNC is NULL");
    if (!opt) die("options is NULL");
}

static int columns_of(int C, int state_len) { return C / states_of(state_len); }

static float log_beam_cut(const openfish_opt_t *opt) {
    /* reference src/beam_search.c:135 */
    return opt->beam_cut > 0.0f ? logf(opt->beam_cut) : FLT_MAX;
}

/* ---- phred thresholds -------------------------------------------------------
 *
 * The quality character of a base is char(x) = (char)(33.5f + clamp(-10*log10f(x)*scale
 * + shift, 1, 50)) of its miss probability x = 1 - base_prob/total_prob (reference
 * src/beam_search.c:92-97).  log10f is a libm routine whose last bit a device routine
 * cannot be relied on to reproduce, but char(x) only steps 49 times over [0,1]: the
 * thresholds are located here by bisection over the float bit patterns with this
 * host's log10f, the neighbourhood of each is checked for monotonicity, and the
 * kernel compares x against them.
 */

static int phred_char(float x, float scale, float shift) {
    volatile float v = -10.0f * log10f(x);
    volatile float q = v * scale;
    q = q + shift;
    if (q > 50.0f) q = 50.0f;
    if (q < 1.0f) q = 1.0f;
    return (int)(char)(33.5f + q);
}

static float bits_float(uint32_t b) {
    float f;
    memcpy(&f, &b, sizeof f);
    return f;
}

static void build_phred_table(ofk_phred_table_t *tab, float scale, float shift) {
    const uint32_t one = 0x3f800000u; /* 1.0f; bit patterns of [0,1] are ordered like the values */
    for (int j = 0; j < OFK_PHRED_STEPS; ++j) {
        const int limit = 82 - j;
        if (phred_char(1.0f, scale, shift) > limit) {
            tab->thr[j] = 2.0f; /* never reached on [0,1] */
            continue;
        }
        uint32_t lo = 0, hi = one; /* char(lo) > limit >= char(hi) */
        if (phred_char(0.0f, scale, shift) <= limit) hi = 0;
        while (hi - lo > 1 && hi != 0) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (phred_char(bits_float(mid), scale, shift) <= limit) hi = mid;
            else lo = mid;
        }
        tab->thr[j] = bits_float(hi);
        for (uint32_t d = 1; d <= 64; ++d) {
            const int below = hi >= d ? phred_char(bits_float(hi - d), scale, shift) : 127;
            const int above = hi + d <= one ? phred_char(bits_float(hi + d), scale, shift) : 0;
            if (below <= limit || above > limit)
                die("phred character is not monotone in the miss probability near a threshold");
        }
    }
}

void openfish_amd_phred_table(float q_scale, float q_shift, float *thr49) {
    ofk_phred_table_t tab;
    build_phred_table(&tab, q_scale, q_shift);
    memcpy(thr49, tab.thr, sizeof tab.thr);
}

static const ofk_phred_table_t *phred_for(ofa_gpubuf_t *g, const openfish_opt_t *opt) {
    if (!g->phred_valid || g->phred_shift != opt->q_shift || g->phred_scale != opt->q_scale) {
        build_phred_table(&g->phred, opt->q_scale, opt->q_shift);
        g->phred_shift = opt->q_shift;
        g->phred_scale = opt->q_scale;
        g->phred_valid = 1;
    }
    return &g->phred;
}

/* ---- decode ---------------------------------------------------------------- */

/* The three result buffers are the caller's to free (the reference's contract), so they are fresh
 * allocations every call.  They are allocated and touched while the GPU works, which takes the page
 * faults off the path between the last kernel and the return. */
static void alloc_outputs(int T, int N, uint8_t **moves, char **sequence, char **qstring) {
    const size_t nt = (size_t)N * (size_t)T;
    *moves = (uint8_t *)host_alloc(nt);
    *sequence = (char *)host_alloc(nt);
    *qstring = (char *)host_alloc(nt);
    memset(*moves, 0, nt);
    memset(*sequence, 0, nt);
    memset(*qstring, 0, nt);
}

/* all three results over the main stream (the stage-level entry point) */
static void fetch_outputs(ofa_gpubuf_t *g, int T, int N, uint8_t **moves, char **sequence, char **qstring) {
    const size_t nt = (size_t)N * (size_t)T;
    HIP_OK(hipMemcpyAsync(g->h_out, g->pub.moves, nt, hipMemcpyDeviceToHost, g->s_main));
    HIP_OK(hipMemcpyAsync(g->h_out + nt, g->pub.sequence, nt, hipMemcpyDeviceToHost, g->s_main));
    HIP_OK(hipMemcpyAsync(g->h_out + 2 * nt, g->pub.qstring, nt, hipMemcpyDeviceToHost, g->s_main));
    HIP_OK(hipEventRecord(g->ev[EV_MOVES], g->s_main));
    alloc_outputs(T, N, moves, sequence, qstring);
    HIP_OK(hipEventSynchronize(g->ev[EV_MOVES]));
    leave_lanes(g);
    memcpy(*moves, g->h_out, nt);
    memcpy(*sequence, g->h_out + nt, nt);
    memcpy(*qstring, g->h_out + 2 * nt, nt);
}

/* Order the library's streams after everything already queued on the null stream (and on the streams that wait for it).  Where that
 * has ended already, which the query tells in 0.2 us, there is nothing to wait for: the event and the wait for it in another hardware
 * queue put 20 us before a decode's first kernel.  That the query answers for the streams ordered with the null stream too is this
 * runtime's doing, and tested for copies and kernels of both.  It is the current device's null stream: a gpubuf of another device is
 * refused, as recording its event there is by the runtime. */
static void join_null_stream(ofa_gpubuf_t *g) {
    int device;
    HIP_OK(hipGetDevice(&device));
    if (device != g->device) die("the gpubuf belongs to another device than the current one");
    if (hipStreamQuery(0) == hipSuccess) return;
    if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError(); /* the query's answer, but no error that the caller left behind */
    HIP_OK(hipEventRecord(g->ev[EV_JOIN], 0));
    HIP_OK(hipStreamWaitEvent(g->s_main, g->ev[EV_JOIN], 0));
}

/* Which arrangement of the scans a decode finishes soonest with.  What bounds them, after the backward sweep:
 *   split   the longer of the search's chain and of the bytes that search and forward sweep move side by side, per
 *           chunk and step 4C + 12S: fp16 scores and fp32 bwd twice, the posterior once;
 *   merged  the chain of the kernel that holds both, three quarters of those bytes or less; the chain is longer than
 *           the search's alone (256 states by 5 %, 1024 by 16 to 40 %), twice that with two rounds of workgroups;
 *   one     both sweeps of a chunk side by side from its two ends, then the search: the longest, with the fewest launches.
 * Whole blocking calls, ms, one | split | merged, T = 1666 unless stated, inputs and arrangements in turn (more of them in
 * tests/test_arrangement.py):
 *   1024 states: 128 3.33 | 2.61 | 2.74;  168 3.56 | 2.66 | 2.77;  172 3.59 | 3.35 | 2.76;  256 3.99 | 3.81 | 2.87;  257 6.50 | 4.64 | 5.22;
 *                320 6.60 | 5.15 | 5.24;  five columns: 288 6.95 | 5.39 | 5.48;  296 6.96 | 5.48 | 5.46;  304 6.95 | 5.56 | 5.49;
 *                T = 833: five columns 320 3.65 | 2.90 | 2.88;  T = 1200: 338 4.97 | 3.92 | 3.95;  340 4.96 | 4.84 | 3.96;
 *                T = 400: 338 1.75 | 1.39 | 1.52;  340 1.75 | 1.77 | 1.52;  five columns 338 1.83 | 1.48 | 1.54;
 *                T = 2000: 320 7.88 | 6.19 | 6.24;  338 7.96 | 6.46 | 6.29;
 *                T = 8: 64 0.068 | 0.072 | 0.057;  164 0.071 | 0.070 | 0.060;  T = 16: 16 0.091 | 0.077 | 0.076;  97 0.094 | 0.082 | 0.079;
 *                T = 20: 16 0.101 | 0.079 | 0.086;  97 0.105 | 0.089 | 0.092;  T = 64: 338 0.359 | 0.332 | 0.377;  360 0.362 | 0.377 | 0.377;
 *                450 0.380 | 0.399 | 0.381;  512 0.370 | 0.430 | 0.404;  T = 100: 360 0.535 | 0.536 | 0.513;  512 0.543 | 0.622 | 0.561
 *    256 states: 256 1.99 | 1.56 | 1.61;  300 2.24 | 1.73 | 1.73;  340 2.26 | 1.74 | 1.75;  360 2.27 | 1.76 | 1.75;  440 2.34 | 1.90 | 1.78;
 *                512 2.47 | 2.15 | 1.82;  five columns: 305 2.26 | 1.74 | 1.75;  320 2.28 | 1.75 | 1.76;  340 2.29 | 1.77 | 1.76;  512 2.70 | 2.34 | 1.86;
 *                T = 1201: 260 1.64 | 1.29 | 1.29;  340 1.68 | 1.32 | 1.31;  five columns 320 1.68 | 1.32 | 1.32;  T = 400: 340 0.632 | 0.525 | 0.525;
 *                five columns 340 0.636 | 0.526 | 0.532;  T = 96: 300 0.195 | 0.170 | 0.163;
 *                513 3.37 | 2.35 | 3.15;  640 3.44 | 2.86 | 3.31;  680 3.47 | 3.34 | 3.33;  768 3.53 | 3.47 | 3.42;  1024 4.18 | 4.67 | 3.87;
 *                five columns: 640 3.58 | 3.13 | 3.42;  680 3.62 | 3.78 | 3.48;  T = 1201: 768 2.55 | 2.52 | 2.54;  T = 1000: five columns 680
 *                2.18 | 2.24 | 2.21;  768 2.26 | 2.26 | 2.24
 *     64 states: 16 1.48 | 1.19;  512 1.78 | 1.43;  2048 3.83 | 3.21
 * Hence the lines.  Up to 168 chunks of 1024 states the search and the forward sweep find compute units of their own (21 and 11 of an
 * XCD's 32); up to 338, in two rounds, split is ahead while its bytes fit beneath the chain, and short chunks allow more of them:
 * 11.65 MB a step, less 1300 bytes for every step of a chunk.  Chunks of up to 16 steps are decided by launches and
 * set-up, batches above 338 of chunks up to 100 steps by the rounds.  Up to 512 chunks of 256 states the chain of split is
 * shorter, while its bytes fit beneath the chain, 2.5 MB a step (348 chunks, five columns 305; between 2.5 and 2.8 MB the two are within 1 % of each
 * other); above,
 * the search's workgroups hold four chunks, the merged kernel's two, in a second round that takes as long with one chunk as with 512,
 * and split has units left for the forward sweep up to 640 chunks, with shorter chunks up to 768.
 *
 * A decode that is enqueued, or finds another one under way, shares the machine; two at a time, one | split | merged:
 *   1024 states: 128 3.98 | 4.82 | 2.87;  320 9.75 | 9.31 | 7.02;  T = 8: 8 0.082 | 0.120 | 0.070;  T = 64: 8 0.219 | 0.286 | 0.203;
 *                T = 127: 15 0.359 | 0.483 | 0.338
 *    256 states: 128 2.50 | 2.11 | 1.74;  512 5.01 | 4.41 | 3.29;  513 4.91 | 4.51 | 4.83;  530 5.04 | 4.82 | 4.92;  548 5.05 | 4.90 | 4.94;  640 6.01 | 5.37 | 5.00;
 *                five columns: 513 5.21 | 4.96 | 4.99;  530 5.32 | 5.24 | 5.07;  T = 2000: 513 5.86 | 5.44 | 5.66;  530 6.09 | 5.75 | 5.88;  548 6.08 | 5.91 | 5.82;
 *                five columns 513 6.21 | 5.82 | 6.01;  T = 2400: 530 7.18 | 6.89 | 6.99;  T = 4000: 513 12.99 | 12.47 | 12.27;
 *                T = 1201: 560 3.68 | 3.61 | 3.66;  T = 800: 600 2.51 | 2.56 | 2.56;  640 2.96 | 2.62 | 2.59;
 *                T = 400: 608 1.29 | 1.37 | 1.41;  620 1.50 | 1.39 | 1.42;  660 1.49 | 1.42 | 1.43;  five columns 640 1.60 | 1.48 | 1.48;
 *                T = 200: 660 0.782 | 0.755 | 0.796;  704 0.795 | 0.813 | 0.833;  T = 100: 620 0.420 | 0.423 | 0.449;  660 0.424 | 0.442 | 0.453
 *     64 states: five columns 512 2.84 | 2.37;  2048 9.96 | 8.95
 * The merged kernel is ahead with 1024 states at every size.  With 256 states split is ahead where a few chunks above 512 would leave merged
 * workgroups half empty, up to 530 chunks of at most 2400 steps (five columns 518) or 548 of a shorter product of steps and scores,
 * and short chunks go further, because the kernels of one batch end between those of the other.
 *
 * The merged kernel exists for 256 and 1024 states with the default arithmetic and its own states per lane; without it
 * (can_merge = 0) 1024 states keep the one kernel and 256 states the split sweeps where they are ahead of it. */
static int arrangement_by_default(int T, int N, int C, int state_len, int shared, int can_merge) {
    const long step_bytes = (long)N * (4L * C + 12L * states_of(state_len)); /* of split */
    const long chunk_scores = (long)T * C;
    switch (state_len) {
        case 3: return N <= 2048 ? ARR_SPLIT : ARR_ONE;
        case 4:
            if (!can_merge) return N <= 768 ? ARR_SPLIT : ARR_ONE;
            if (N <= 512) return shared || step_bytes > 2500000 ? ARR_MERGED : ARR_SPLIT;
            if (!shared) return N <= 640 || (N <= 768 && chunk_scores <= 1250000) ? ARR_SPLIT : ARR_MERGED;
            if (T <= 400 && N <= 608) return ARR_ONE;
            if (chunk_scores <= 525000 && N <= 660) return T <= 128 ? ARR_ONE : ARR_SPLIT;
            if (chunk_scores <= 950000 && N <= 608) return ARR_SPLIT;
            if (T <= 2400 && N <= 530 && step_bytes <= 4250000) return ARR_SPLIT;
            return chunk_scores <= 1900000 && N <= 548 ? ARR_SPLIT : ARR_MERGED;
        default:
            if (!can_merge) return ARR_ONE;
            if (shared) return ARR_MERGED;
            if (N <= 168) return T <= 16 ? ARR_MERGED : ARR_SPLIT;
            if (N <= 256) return ARR_MERGED;
            if (N <= 338) return step_bytes + 1300L * T <= 11650000 ? ARR_SPLIT : ARR_MERGED;
            return T < 72 || (N >= 512 && T <= 100) ? ARR_ONE : ARR_MERGED;
    }
}

int openfish_amd_scan_arrangement(int T, int N, int C, int state_len, int shared) {
    check_state_len(state_len);
    return arrangement_by_default(T, N, C, state_len, shared, state_len >= 4);
}

/* the arrangement of one decode: what the gpubuf asks for, or by the rule above.  Merged asked for where it does not
 * exist gives way to the choice among the other two. */
static int arrangement_of(const ofa_gpubuf_t *g, int T, int N, int C, int state_len, int shared) {
    const int can_merge = state_len >= 4 && g->scan_mode == OFK_SCAN_TWO_TIER && g->scan_spl == 0;
    if (g->split_scans == ARR_ONE || g->split_scans == ARR_SPLIT) return g->split_scans;
    if (g->split_scans == ARR_MERGED && can_merge) return ARR_MERGED;
    return arrangement_by_default(T, N, C, state_len, shared, can_merge);
}

/* Queue one decode on the gpubuf's streams, results into its pinned staging buffer; returns
 * without waiting for the GPU. */
static void enqueue_decode(ofa_gpubuf_t *g, const int T, const int N, const int C, const void *scores_TNC,
                           const int state_len, const openfish_opt_t *options, const int enqueued) {
    const float stay = options->blank_score; /* as the reference GPU path, src/decode_hip.hip:120 */
    const size_t nt = (size_t)N * (size_t)T;

    const int cols = columns_of(C, state_len);
    const int others = take_main_lane(g), shared = others || enqueued;
    const int search_flags = g->debug_flags | (shared ? 0 : OFK_SEARCH_ALONE);
    g->pend_split = arrangement_of(g, T, N, C, state_len, shared);
    g->pend_apart = 0;
    /* Sums only where the search leaves the machine idle, and not with 1024 states, whose search waits for
     * memory and was measured to take half as long again beside the extra kernel.
     * With split scans the posteriors are complete when the forward kernel ends.  With 64 states that is
     * well before the search does (0.83 against 1.13 ms at 512 chunks), and the sums (0.21 ms) fit in
     * between; with 256 states the two end together and the sequence stage gathers by itself, as it does where
     * another decode waits for the side lane (four decodes of 256 chunks of 64 states: 4.19 ms with sums, 3.69 without;
     * the results have the same bits). */
    const int sums_fit = g->path_sums != NULL && N <= OFK_SPARSE_SEARCH_MAX_CHUNKS;
    const int use_sums = sums_fit && (g->pend_split == ARR_ONE || (g->pend_split == ARR_SPLIT && state_len == 3 && !others));
    g->pend_sums = use_sums;
    g->pend_copy = !shared && nt >= OFA_COPY_MOVES;
    if (g->pend_split == ARR_SPLIT || use_sums || g->pend_copy) take_side_lane(g);
    join_null_stream(g);
    /* A marker, which holds up the first kernel by 3 us.  It has to be ahead of that kernel on the same stream: on the side lane it would be
     * behind whatever another thread's decode, or a stream of the caller's in the same hardware queue, has there meanwhile. */
    HIP_OK(hipEventRecord(g->ev[EV_START], g->s_main));
    if (g->pend_split == ARR_MERGED) {
        /* backward sweep, then the search with the forward sweep and the posterior in its workgroups */
        launch_ok(ofk_bwd_scan(scores_TNC, g->pub.bwd_NTC, T, N, state_len, cols, stay, g->scan_mode, g->scan_spl, g->s_main,
                               g->ev[EV_BWD_END]), "bwd_scan");
        launch_ok(ofk_beam_search_forward(scores_TNC, g->pub.bwd_NTC, g->pub.post_NTC, (ofk_beam_slot_t *)g->pub.beam_vector,
                                          (int32_t *)g->pub.states, g->pub.moves, T, N, state_len, cols,
                                          log_beam_cut(options), stay, g->lse_table, g->debug_flags, g->s_main, g->ev[EV_BEAM_END]),
                  "beam_search_forward");
    } else if (g->pend_split == ARR_ONE) {
        /* both sweeps and the posterior in one kernel, then the beam search, all on one stream */
        launch_ok(ofk_scan_posterior(scores_TNC, g->pub.bwd_NTC, g->pub.post_NTC, T, N, state_len, cols, stay, g->scan_mode,
                                     g->scan_spl, g->s_main, g->ev[EV_BWD_END]), "scan_posterior");
        launch_ok(ofk_beam_search(scores_TNC, g->pub.bwd_NTC, (ofk_beam_slot_t *)g->pub.beam_vector,
                                  (int32_t *)g->pub.states, g->pub.moves, T, N, state_len, cols, log_beam_cut(options),
                                  stay, g->lse_table, search_flags, g->s_main, g->ev[EV_BEAM_END]), "beam_search");
        /* The search keeps one wave per chunk busy and leaves the rest of the machine idle: beside
         * it, on the second stream, the posteriors that a block's quality is made of are summed for
         * every state, so that the sequence stage reads one value per time step instead of nine. */
        if (use_sums) {
            HIP_OK(hipStreamWaitEvent(g->s_side, g->ev[EV_BWD_END], 0));
            launch_ok(ofk_path_sums(g->pub.post_NTC, g->path_sums, T, N, state_len, g->s_side, g->ev[EV_SUMS_END]), "path_sums");
        }
    } else {
        /* A sweep of 1024 states has a compute unit to a chunk.  A batch that leaves half of the units idle, and shares them
         * with no other decode, has the forward sweep on units of its own beside the backward one; only the posterior is then
         * left to do beside the search.  It moves 8 more bytes per state and step, which is why it ends short of 128 chunks.
         * Whole calls, ms, sweep and posterior beside the search | apart: 1 chunk, T = 33 0.171 | 0.160; 8, T = 100 0.317 | 0.264;
         * T = 833: 1 1.48 | 1.23, 37 1.51 | 1.27, 64 1.52 | 1.31, 96 1.53 | 1.33; five columns, T = 1666: 80 2.67 | 2.51,
         * 96 2.68 | 2.57, 112 2.72 | 2.73, 128 2.82 | 2.85. */
        const int apart = g->pend_apart = state_len == 5 && N <= 96 && !shared && g->scan_mode == OFK_SCAN_TWO_TIER && g->scan_spl == 0;
        launch_ok(ofk_bwd_scan(scores_TNC, g->pub.bwd_NTC, T, N, state_len, cols, stay, g->scan_mode, g->scan_spl, g->s_main,
                               g->ev[EV_BWD_END]), "bwd_scan");
        if (apart) {
            HIP_OK(hipStreamWaitEvent(g->s_side, g->ev[EV_START], 0));
            launch_ok(ofk_fwd_scan(scores_TNC, g->pub.post_NTC, T, N, state_len, cols, stay, g->s_side, g->ev[EV_FWD_SCAN_END]),
                      "fwd_scan");
        }

        /* The beam search is the longer of the two stages that follow and wants its workgroups (large
         * LDS blocks) resident before the forward sweep fills the compute units: it stays on the stream
         * the backward sweep ran on and so starts first; the forward sweep follows through an event. */
        launch_ok(ofk_beam_search(scores_TNC, g->pub.bwd_NTC, (ofk_beam_slot_t *)g->pub.beam_vector,
                                  (int32_t *)g->pub.states, g->pub.moves, T, N, state_len, cols, log_beam_cut(options),
                                  stay, g->lse_table, search_flags, g->s_main, g->ev[EV_BEAM_END]), "beam_search");

        HIP_OK(hipStreamWaitEvent(g->s_side, g->ev[EV_BWD_END], 0));
        if (apart)
            launch_ok(ofk_posterior_rows(g->pub.bwd_NTC, g->pub.post_NTC, T, N, state_len, g->s_side, g->ev[EV_FWD_END]),
                      "posterior_rows");
        else
            launch_ok(ofk_fwd_post_scan(scores_TNC, g->pub.bwd_NTC, g->pub.post_NTC, T, N, state_len, cols, stay, g->scan_mode,
                                        g->scan_spl, g->s_side, g->ev[EV_FWD_END]), "fwd_post_scan");
        if (use_sums) {
            launch_ok(ofk_path_sums(g->pub.post_NTC, g->path_sums, T, N, state_len, g->s_side, g->ev[EV_SUMS_END]), "path_sums");
        }
    }

    /* The moves are final once the beam search is.  Of a decode that has the device to itself, and enough of them, they travel, and
     * the host takes them, while the sequence stage runs.  Otherwise that stage writes them to the host itself (0.02 ms),
     * because a copy that waits for the search would hold up another decode's forward sweep behind
     * it on the side lane (two batches of 16 chunks of 64 states in flight: 2.14 ms with the copies, 1.63 without). */
    if (g->pend_copy) {
        HIP_OK(hipStreamWaitEvent(g->s_side, g->ev[EV_BEAM_END], 0));
        HIP_OK(hipMemcpyAsync(g->h_out, g->pub.moves, nt, hipMemcpyDeviceToHost, g->s_side));
        HIP_OK(hipEventRecord(g->ev[EV_MOVES], g->s_side));
    }
    if (use_sums) HIP_OK(hipStreamWaitEvent(g->s_main, g->ev[EV_SUMS_END], 0));
    else if (g->pend_split == ARR_SPLIT) HIP_OK(hipStreamWaitEvent(g->s_main, g->ev[EV_FWD_END], 0));

    /* The last kernel writes bases and qualities straight into the pinned host memory (N * T bytes
     * each, every byte once, 16 bytes a lane): they are in host memory when the
     * kernel ends and no copy follows it, which measured 0.05 ms less per call at 512 x 1666 than two
     * copies after a kernel that is 0.03 ms shorter.  The gpubuf's own sequence and qstring arrays
     * are filled by the stage-level entry points only. */
    launch_ok(ofk_sequence(g->pub.post_NTC, (int32_t *)g->pub.states, g->pub.moves, g->pub.qual_data,
                           g->pub.base_probs, g->pub.total_probs, (char *)g->d_out + nt, (char *)g->d_out + 2 * nt, T, N,
                           state_len, phred_for(g, options), use_sums ? g->path_sums : NULL, g->pend_copy ? NULL : g->d_out, g->s_main, g->ev[EV_SEQ_END]), "sequence");
    /* The host waits for the end of that kernel, which it sees 3 us before the end of a marker behind it.  The markers are for the
     * runtime: a stream that ends with one is known to be done, one that ends with a kernel gets a marker and a wait of its own, 5 us
     * each, in the caller's next hipDeviceSynchronize. */
    HIP_OK(hipEventRecord(g->ev[EV_TAIL], g->s_main));
    if (g->side_lane >= 0 && !g->pend_copy) HIP_OK(hipEventRecord(g->ev[EV_SIDE_TAIL], g->s_side));
    g->pending = 1;
    g->pend_T = T;
    g->pend_N = N;
}

void openfish_decode_gpu(const int T, const int N, const int C, void *scores_TNC, const int state_len,
                         const openfish_opt_t *options, const openfish_gpubuf_t *gpubuf, uint8_t **moves,
                         char **sequence, char **qstring) {
    check_scores(T, N, C, scores_TNC, state_len, options);
    if (!moves || !sequence || !qstring) die("decode: output pointer is NULL");
    ofa_gpubuf_t *g = checked(gpubuf, T, N, state_len);
    const size_t nt = (size_t)N * (size_t)T;
    OPENFISH_LOG_TRACE("scores tensor dim: %d, %d, %d", T, N, C);

    enqueue_decode(g, T, N, C, scores_TNC, state_len, options, 0);
    alloc_outputs(T, N, moves, sequence, qstring);
    if (g->pend_copy) {
        HIP_OK(hipEventSynchronize(g->ev[EV_MOVES]));
        memcpy(*moves, g->h_out, nt);
    }
    wait_for_decode(g);
    if (!g->pend_copy) memcpy(*moves, g->h_out, nt);
    memcpy(*sequence, g->h_out + nt, nt);
    memcpy(*qstring, g->h_out + 2 * nt, nt);
    g->pending = 0;
    g->timed = 1;
}

void openfish_amd_decode_enqueue(int T, int N, int C, const void *scores_TNC, int state_len,
                                 const openfish_opt_t *options, const openfish_gpubuf_t *gpubuf) {
    check_scores(T, N, C, scores_TNC, state_len, options);
    ofa_gpubuf_t *g = checked(gpubuf, T, N, state_len);
    enqueue_decode(g, T, N, C, scores_TNC, state_len, options, 1);
}

void openfish_amd_decode_wait(const openfish_gpubuf_t *gpubuf, const uint8_t **moves, const char **sequence,
                              const char **qstring) {
    ofa_gpubuf_t *g = (ofa_gpubuf_t *)gpubuf;
    if (!g || g->magic != OFA_MAGIC) die("gpubuf was not created by openfish_gpubuf_init");
    if (!g->pending) die("decode_wait: nothing was enqueued on this gpubuf");
    if (!moves || !sequence || !qstring) die("decode_wait: output pointer is NULL");
    const size_t nt = (size_t)g->pend_N * (size_t)g->pend_T;
    wait_for_decode(g);
    *moves = g->h_out;
    *sequence = (const char *)g->h_out + nt;
    *qstring = (const char *)g->h_out + 2 * nt;
    g->pending = 0;
    g->timed = 1;
}

int openfish_amd_last_timings(const openfish_gpubuf_t *gpubuf, float *ms, int n) {
    ofa_gpubuf_t *g = (ofa_gpubuf_t *)gpubuf;
    if (!g || g->magic != OFA_MAGIC) die("gpubuf was not created by openfish_gpubuf_init");
    if (!g->timed || !ms || n < 1) return 0;
    if (g->pend_split != ARR_ONE) {
        HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_BWD], g->ev[EV_START], g->ev[EV_BWD_END]));
        HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_FWD], g->ev[EV_BWD_END],
                                    g->ev[g->pend_split == ARR_MERGED ? EV_BEAM_END : EV_FWD_END])); /* merged: one kernel with the search */
        g->ms[OPENFISH_AMD_STAGE_SCAN] = 0.0f;
    } else {
        g->ms[OPENFISH_AMD_STAGE_BWD] = g->ms[OPENFISH_AMD_STAGE_FWD] = 0.0f;
        HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_SCAN], g->ev[EV_START], g->ev[EV_BWD_END]));
    }
    g->ms[OPENFISH_AMD_STAGE_FWD_SCAN] = 0.0f;
    if (g->pend_split == ARR_SPLIT && g->pend_apart) {
        /* the posteriors' pass begins with the later of the two sweeps' ends */
        float behind = 0.0f;
        HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_FWD_SCAN], g->ev[EV_START], g->ev[EV_FWD_SCAN_END]));
        HIP_OK(hipEventElapsedTime(&behind, g->ev[EV_FWD_SCAN_END], g->ev[EV_FWD_END]));
        if (behind < g->ms[OPENFISH_AMD_STAGE_FWD]) g->ms[OPENFISH_AMD_STAGE_FWD] = behind;
    }
    /* a stage begins where the last one that it waits for ends */
    HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_BEAM], g->ev[EV_BWD_END], g->ev[EV_BEAM_END]));
    HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_TOTAL], g->ev[EV_START], g->ev[EV_SEQ_END]));
    g->ms[OPENFISH_AMD_STAGE_SUMS] = 0.0f;
    if (g->pend_sums)
        HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_SUMS], g->ev[g->pend_split == ARR_ONE ? EV_BWD_END : EV_FWD_END], g->ev[EV_SUMS_END]));
    HIP_OK(hipEventElapsedTime(&g->ms[OPENFISH_AMD_STAGE_SEQ], g->ev[EV_BEAM_END], g->ev[EV_SEQ_END]));
    if (g->pend_sums || g->pend_split == ARR_SPLIT) {
        float behind = 0.0f;
        HIP_OK(hipEventElapsedTime(&behind, g->ev[g->pend_sums ? EV_SUMS_END : EV_FWD_END], g->ev[EV_SEQ_END]));
        if (behind < g->ms[OPENFISH_AMD_STAGE_SEQ]) g->ms[OPENFISH_AMD_STAGE_SEQ] = behind;
    }
    if (n > OPENFISH_AMD_STAGE_COUNT) n = OPENFISH_AMD_STAGE_COUNT;
    memcpy(ms, g->ms, sizeof(float) * (size_t)n);
    return n;
}

/* ---- stages ---------------------------------------------------------------- */

static void check_scan_mode(int scan_mode) {
    if (scan_mode != OFK_SCAN_TWO_TIER && scan_mode != OFK_SCAN_PRECISE && scan_mode != OFK_SCAN_FAST)
        die("scan mode must be OPENFISH_AMD_SCAN_TWO_TIER, _PRECISE or _FAST");
}

void openfish_amd_bwd_scan(int T, int N, int C, const void *scores, int state_len, float stay_score, int scan_mode,
                           float *bwd) {
    openfish_opt_t o = DECODER_INIT;
    check_scores(T, N, C, scores, state_len, &o);
    check_scan_mode(scan_mode);
    launch_ok(ofk_bwd_scan(scores, bwd, T, N, state_len, columns_of(C, state_len), stay_score, scan_mode, 0, NULL, NULL), "bwd_scan");
    HIP_OK(hipStreamSynchronize(0));
}

void openfish_amd_fwd_post_scan(int T, int N, int C, const void *scores, int state_len, float stay_score,
                                int scan_mode, const float *bwd, float *post) {
    openfish_opt_t o = DECODER_INIT;
    check_scores(T, N, C, scores, state_len, &o);
    check_scan_mode(scan_mode);
    launch_ok(ofk_fwd_post_scan(scores, bwd, post, T, N, state_len, columns_of(C, state_len), stay_score, scan_mode, 0, NULL, NULL), "fwd_post_scan");
    HIP_OK(hipStreamSynchronize(0));
}

void openfish_amd_scan_posterior(int T, int N, int C, const void *scores, int state_len, float stay_score,
                                 int scan_mode, float *bwd, float *post) {
    openfish_opt_t o = DECODER_INIT;
    check_scores(T, N, C, scores, state_len, &o);
    check_scan_mode(scan_mode);
    launch_ok(ofk_scan_posterior(scores, bwd, post, T, N, state_len, columns_of(C, state_len), stay_score, scan_mode, 0, NULL, NULL), "scan_posterior");
    HIP_OK(hipStreamSynchronize(0));
}

void openfish_amd_beam_search(int T, int N, int C, const void *scores, int state_len,
                              const openfish_opt_t *options, const float *bwd, const openfish_gpubuf_t *gpubuf) {
    check_scores(T, N, C, scores, state_len, options);
    ofa_gpubuf_t *g = checked(gpubuf, T, N, state_len);
    launch_ok(ofk_beam_search(scores, bwd, (ofk_beam_slot_t *)g->pub.beam_vector, (int32_t *)g->pub.states,
                              g->pub.moves, T, N, state_len, columns_of(C, state_len), log_beam_cut(options),
                              options->blank_score,
                              g->lse_table, g->debug_flags, NULL, NULL),
              "beam_search");
    HIP_OK(hipStreamSynchronize(0));
}

void openfish_amd_beam_search_static_prepare(void) {
    if (ofk_beam_search_static_ready()) return;
    double tab[OFK_LSE_DOUBLES];
    build_lse_table(tab);
    launch_ok(ofk_beam_search_static_prepare(tab), "beam_search_static_prepare");
}

void openfish_amd_beam_search_static(int T, int N, int C, const void *scores, int state_len,
                                     const openfish_opt_t *options, const float *bwd, int32_t *states,
                                     uint8_t *moves, void *stream) {
    check_scores(T, N, C, scores, state_len, options);
    if (!bwd || !states || !moves) die("beam_search_static: bwd, states and moves must be device pointers");
    const int rc = ofk_beam_search_static(scores, bwd, states, moves, T, N, state_len, columns_of(C, state_len),
                                          log_beam_cut(options), options->blank_score, 0, stream);
    if (rc == OFK_NOT_PREPARED)
        die("beam_search_static: call openfish_amd_beam_search_static_prepare() on this device first");
    if (rc == OFK_TOO_LARGE) {
        fprintf(stderr, "openfish: beam_search_static: N * (T + 1) * 64 = %zu bytes of beam slots exceed the static "
                        "scratch array of %u bytes; use openfish_amd_beam_search with a gpubuf\n",
                (size_t)N * (size_t)(T + 1) * 64, (unsigned)OFK_STATIC_SLOT_BYTES);
        exit(EXIT_FAILURE);
    }
    launch_ok(rc, "beam_search_static");
}

size_t openfish_amd_device_free_bytes(void) {
    size_t free_b = 0, total_b = 0;
    HIP_OK(hipMemGetInfo(&free_b, &total_b));
    return free_b;
}

void openfish_amd_sequence(int T, int N, int state_len, const openfish_opt_t *options, const float *post,
                           const openfish_gpubuf_t *gpubuf) {
    if (!options) die("options is NULL");
    ofa_gpubuf_t *g = checked(gpubuf, T, N, state_len);
    launch_ok(ofk_sequence(post, (int32_t *)g->pub.states, g->pub.moves, g->pub.qual_data, g->pub.base_probs,
                           g->pub.total_probs, g->pub.sequence, g->pub.qstring, T, N, state_len,
                           phred_for(g, options), NULL, NULL, NULL, NULL), "sequence");
    HIP_OK(hipStreamSynchronize(0));
}

void openfish_amd_decode_from_tensors(int T, int N, int C, const void *scores, int state_len,
                                      const openfish_opt_t *options, const float *bwd, const float *post,
                                      const openfish_gpubuf_t *gpubuf, uint8_t **moves, char **sequence,
                                      char **qstring) {
    check_scores(T, N, C, scores, state_len, options);
    if (!moves || !sequence || !qstring) die("decode: output pointer is NULL");
    ofa_gpubuf_t *g = checked(gpubuf, T, N, state_len);
    take_main_lane(g);
    join_null_stream(g);
    launch_ok(ofk_beam_search(scores, bwd, (ofk_beam_slot_t *)g->pub.beam_vector, (int32_t *)g->pub.states,
                              g->pub.moves, T, N, state_len, columns_of(C, state_len), log_beam_cut(options),
                              options->blank_score,
                              g->lse_table, g->debug_flags, g->s_main, NULL), "beam_search");
    /* the quality stage as a whole decode runs it: from per-state sums where the gpubuf holds room for them */
    const float *sums = NULL;
    if (g->path_sums != NULL && N <= OFK_SPARSE_SEARCH_MAX_CHUNKS) {
        launch_ok(ofk_path_sums(post, g->path_sums, T, N, state_len, g->s_main, NULL), "path_sums");
        sums = g->path_sums;
    }
    launch_ok(ofk_sequence(post, (int32_t *)g->pub.states, g->pub.moves, g->pub.qual_data, g->pub.base_probs,
                           g->pub.total_probs, g->pub.sequence, g->pub.qstring, T, N, state_len,
                           phred_for(g, options), sums, NULL, g->s_main, NULL), "sequence");
    fetch_outputs(g, T, N, moves, sequence, qstring);
}

/* ---- rotary embedding ------------------------------------------------------ */

void openfish_rotary_emb_gpu(void *x_gpu, void *sin_gpu, void *cos_gpu, int batch_size, int seqlen, int nheads,
                             int head_dim, int rotary_half, int stride_batch, int stride_seq, int stride_head) {
    (void)head_dim; /* unused by the reference as well (src/rotary_emb_hip.h:36-45) */
    launch_ok(ofk_rotary_emb(x_gpu, (const float *)sin_gpu, (const float *)cos_gpu, batch_size, seqlen, nheads,
                             rotary_half, stride_batch, stride_seq, stride_head, NULL), "rotary_emb");
    HIP_OK(hipStreamSynchronize(0));
}

/* ---- CPU entry points of the reference API: not carried by this library ---- */

void openfish_decode_cpu(const int T, const int N, const int C, int nthreads, void *scores_TNC,
                         const int state_len, const openfish_opt_t *options, uint8_t **moves, char **sequence,
                         char **qstring) {
    (void)T; (void)N; (void)C; (void)nthreads; (void)scores_TNC; (void)state_len; (void)options;
    (void)moves; (void)sequence; (void)qstring;
    die("openfish_decode_cpu: this library carries the GPU path only");
}

void openfish_rotary_emb_cpu(void *x, void *sin_buf, void *cos_buf, int batch_size, int seqlen, int nheads,
                             int head_dim, int rotary_half, int stride_batch, int stride_seq, int stride_head,
                             int nthreads) {
    (void)x; (void)sin_buf; (void)cos_buf; (void)batch_size; (void)seqlen; (void)nheads; (void)head_dim;
    (void)rotary_half; (void)stride_batch; (void)stride_seq; (void)stride_head; (void)nthreads;
    die("openfish_rotary_emb_cpu: this library carries the GPU path only");
}

/* ---- device helpers -------------------------------------------------------- */

void set_device_hip(int device) { HIP_OK(hipSetDevice(device)); }

void *upload_scores_to_hip(const int T, const int N, const int C, const void *scores_TNC) {
    void *dev = NULL;
    const size_t bytes = 2 * (size_t)T * (size_t)N * (size_t)C;
    HIP_OK(hipMalloc(&dev, bytes));
    HIP_OK(hipMemcpy(dev, scores_TNC, bytes, hipMemcpyHostToDevice));
    return dev;
}

void free_scores_hip(void *scores_TNC_gpu) { HIP_OK(hipFree(scores_TNC_gpu)); }

static void dump_blob(const char *name, const void *dev, size_t bytes) {
    void *host = host_alloc(bytes);
    HIP_OK(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost));
    FILE *fp = fopen(name, "w");
    if (!fp || fwrite(host, 1, bytes, fp) != bytes) {
        fprintf(stderr, "openfish: error writing %s: %s\n", name, strerror(errno));
        exit(EXIT_FAILURE);
    }
    fclose(fp);
    free(host);
}

void write_gpubuf_hip(const uint64_t T, const uint64_t N, const int state_len, const openfish_gpubuf_t *gpubuf) {
    check_state_len(state_len);
    const size_t S = (size_t)states_of(state_len), tens = sizeof(float) * N * (T + 1) * S, nt = N * T;
    dump_blob("bwd_NTC.blob", gpubuf->bwd_NTC, tens);
    dump_blob("post_NTC.blob", gpubuf->post_NTC, tens);
    dump_blob("qual_data.blob", gpubuf->qual_data, sizeof(float) * 4 * nt);
    dump_blob("base_probs.blob", gpubuf->base_probs, sizeof(float) * nt);
    dump_blob("total_probs.blob", gpubuf->total_probs, sizeof(float) * nt);
}

void *openfish_amd_malloc(size_t bytes) {
    void *dev = NULL;
    HIP_OK(hipMalloc(&dev, bytes ? bytes : 1));
    return dev;
}
void openfish_amd_free(void *dev) { HIP_OK(hipFree(dev)); }
void openfish_amd_memcpy_h2d(void *dev, const void *host, size_t bytes) { HIP_OK(hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice)); }
void openfish_amd_memcpy_d2h(void *host, const void *dev, size_t bytes) { HIP_OK(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost)); }
void openfish_amd_memset(void *dev, int value, size_t bytes) { HIP_OK(hipMemset(dev, value, bytes)); }
void openfish_amd_sync(void) { HIP_OK(hipDeviceSynchronize()); }
void openfish_amd_copy(void *dst, const void *src, size_t bytes) {
    launch_ok(ofk_copy(dst, src, bytes, NULL), "copy");
    HIP_OK(hipStreamSynchronize(0));
}

void openfish_amd_probe_hw_math(double *errors4, unsigned int *identities) {
    if (!errors4 || !identities) die("probe_hw_math: output pointer is NULL");
    void *dev = NULL;
    unsigned char host[40];
    HIP_OK(hipMalloc(&dev, sizeof host));
    launch_ok(ofk_probe_hw_math(dev, NULL), "probe_hw_math");
    HIP_OK(hipStreamSynchronize(0));
    HIP_OK(hipMemcpy(host, dev, sizeof host, hipMemcpyDeviceToHost));
    HIP_OK(hipFree(dev));
    memcpy(errors4, host, 4 * sizeof(double));
    memcpy(identities, host + 32, sizeof *identities);
    for (int k = 0; k < 4; ++k) errors4[k] *= 16777216.0; /* in units of 2^-24 */
}

int openfish_amd_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return n;
}

/* Settings live in the gpubuf and are read when a decode is enqueued on it, so callers with one
 * gpubuf each (one per host thread) do not see each other's settings. */
static ofa_gpubuf_t *owned(const openfish_gpubuf_t *gpubuf) {
    ofa_gpubuf_t *g = (ofa_gpubuf_t *)gpubuf;
    if (!g || g->magic != OFA_MAGIC) die("gpubuf was not created by openfish_gpubuf_init");
    return g;
}

void openfish_amd_gpubuf_set_debug_flags(const openfish_gpubuf_t *gpubuf, int flags) {
    owned(gpubuf)->debug_flags = flags & 3;
}

void openfish_amd_gpubuf_set_scan_mode(const openfish_gpubuf_t *gpubuf, int scan_mode) {
    check_scan_mode(scan_mode);
    owned(gpubuf)->scan_mode = scan_mode;
}

void openfish_amd_gpubuf_set_split_scans(const openfish_gpubuf_t *gpubuf, int split) {
    owned(gpubuf)->split_scans = split < 0 ? -1 : split == 2 ? ARR_MERGED : split ? ARR_SPLIT : ARR_ONE;
}

void openfish_amd_gpubuf_set_scan_states_per_lane(const openfish_gpubuf_t *gpubuf, int spl) {
    if (spl != 0 && spl != 1 && spl != 2 && spl != 4) die("states per lane must be 0 (automatic), 1, 2 or 4");
    owned(gpubuf)->scan_spl = spl;
}

const char *openfish_amd_version(void) { return "openfish-amd gfx950"; }
