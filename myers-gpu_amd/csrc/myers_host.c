/*
 * Host side of the candidate-verification library: the buffer API of
 * src-api/myers-interface.h, re-designed for one MI355X.
 *
 * Plain C over the HIP runtime C API.  Kernels are launched through the
 * extern "C" shims of the .hip files (myers_kernels.h).
 *
 * Life of a batch (src-api/myersGPU.c:466-524 is the reference flow):
 *   send:    async H2D of Peq entries, qinfo and candidates on the buffer's
 *            stream -> kernel launches -> async D2H of the results (a launch
 *            over one bin of short reads uses the host arrays as they are).  The
 *            kernels write results in the caller's candidate order, so the
 *            reference's host reorder (myersGPU.c:351-422) and result
 *            scatter (myersGPU.c:500-513) do not exist here.
 *   launch:  the host scans qinfo (O(queries)) for the length bins present.
 *            One bin -> one launch over the candidates as they are.  More
 *            bins, or a large batch -> device-side binning (count, scan,
 *            scatter), then one launch per present bin in turn (plain engine),
 *            one queue launch per kernel class (persistent engine) or one
 *            resident launch per bin on forked streams (binned engine).  Small
 *            batches split their candidates over waves (split_plan), mid-sized
 *            ones of long reads share one launch (long_plan), large ones of
 *            long reads run the sliced kernel (wide_bins).
 *   receive: hipStreamSynchronize; results are in the pinned results buffer.
 *
 * All buffers of a library instance live on one device and share one copy
 * of the packed reference in HBM (the reference freed it once per buffer,
 * myersGPU.c:661).
 */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

#include "myers-interface.h"
#include "myers-amd.h"
#include "myers_internal.h"
#include "myers_kernels.h"

#define GUARD_WORDS      64u            /* all-N words after the reference */
#define ALL_N_WORD       0x44444444u
#define MAX_QUERY_WORDS  (MYERS_MAX_QUERY_SIZE / 32u)
#define BIN_ROWS         (MAX_QUERY_WORDS + 1u)
#define STAGE_BYTES      (64u << 20)    /* pinned staging for the reference upload */
#define DEFAULT_BUFFER_CAP (2ull << 30)
#define EV_RING          32u            /* kernel-timing event pairs per buffer */
#define GROUP_N_WORDS    12u             /* reads of more words: candidates grouped by N in the read */
#define SIDE_STREAMS     4u             /* fork width of a persistent launch */

typedef struct myers_ctx {
    int       device;
    int       num_cus;
    uint32_t *d_ref;
    uint64_t  ref_words;         /* stored words */
    uint64_t  ref_words_alloc;   /* stored + guard */
    uint64_t  ref_size;          /* bases */
    uint32_t *d_planes;          /* bit planes of d_ref for the one-lane variants */
    uint32_t  plane_blocks;
    uint32_t  num_variants;
    myers_variant_desc_t variants[MYERS_MAX_VARIANTS];
    int       occupancy[MYERS_MAX_VARIANTS];       /* plain kernel, workgroups per CU */
    int       occupancy_p[MYERS_MAX_VARIANTS];     /* persistent kernel */
    uint64_t  multi_lane, deep;   /* masks: variants of several lanes; one-lane ones of 8 words or more */
    uint32_t  chunk_factor[MYERS_MAX_VARIANTS];    /* persistent: chunks per queue pull */
    uint32_t  long_seq;                            /* long-read launches so far (placement rotation) */
    /* workgroups per CU of the multi-lane queue kernel, its threshold form and the two
     * one-lane kernels, each for the dynamic LDS size beside it (0: not queried) */
    int       queue_occ[4];
    uint32_t  queue_occ_lds[4];
    uint8_t   bin_of_words[BIN_ROWS];              /* the caller's table or the tuning file's */
    uint8_t   fine_of_words[BIN_ROWS];             /* the same with a bin per word count of one-lane reads (bins_of) */
    uint8_t  *d_bin_of_words;                      /* both, one after the other */
    uint32_t  in_flight;         /* buffers with a batch sent and not yet received */
    uint64_t  tune_gen;          /* bumped when the bin table or chunk factors change */
    uint32_t *d_scratch;         /* this device's static workspace (myersVerifyDeviceNoAlloc) */
} myers_ctx_t;

typedef struct myers_buffer {
    myers_ctx_t *ctx;
    uint32_t     num_buffers;
    uint32_t     id_buffer;
    uint32_t     max_peq_entries;
    uint32_t     max_candidates;
    uint32_t     max_queries;
    hipStream_t  stream;
    qryEntry_t  *h_peq;
    qryEntry_t  *d_peq;
    qryInfo_t   *h_qinfo;
    qryInfo_t   *d_qinfo;
    candInfo_t  *h_cands;
    candInfo_t  *d_cands;
    resEntry_t  *h_results;
    resEntry_t  *d_results;
    void        *hd_peq, *hd_qinfo, *hd_cands, *hd_results;     /* the host arrays' addresses on the device */
    uint32_t    *d_order;
    uint32_t    *d_work;          /* MYERS_WORK_WORDS: ranges | queue part heads | block counts */
    uint32_t    *d_split;         /* the split launch's pool, from its first use on (split_pool) */
    uint32_t    *h_err;           /* error flag of the binning, which writes it here (pinned) */
    uint32_t    *d_err;           /* its address on the device */
    hipEvent_t   ev_batch_start, ev_batch_end;
    /* HIP events around the verification launches of each batch, in a ring
     * so that batches enqueued back to back are all timed; folded into the
     * stats in order when the stream is synchronised. */
    hipEvent_t   ev_kernel[EV_RING][3];   /* start, end, start of the verification launches */
    uint32_t     ev_launches[EV_RING];
    uint8_t      ev_marked[EV_RING];      /* event 2 was recorded (eager batches after binning) */
    int          mark_slot;               /* slot whose event 2 enqueue_pipeline records, or -1 */
    uint32_t     ev_head, ev_pending;
    /* launches of one batch that run side by side: forked streams joined by events */
    hipStream_t  side[SIDE_STREAMS];
    hipEvent_t   ev_fork, ev_join[SIDE_STREAMS];
    /* steady-state graph of the last device-resident batch shape */
    hipGraphExec_t graph_exec;
    uint64_t     graph_key[14];
    int          graph_valid;
    int          graph_binned;
    uint32_t     graph_launches;
    int          exit_on_error;
    float        threshold;       /* < 0: off (myersSetThreshold) */
    int          last_error;
    int          pending;         /* a batch was enqueued and not yet received */
    int          binned;
    uint32_t     num_candidates;
    myersStats_t stats;
    myers_launch_info_t ran, graph_ran;
} myers_buffer_t;

static void load_default_tuning(myers_ctx_t *ctx);

/* ------------------------------------------------------------------ errors */

const char *myersGetErrorString(int error)
{
    switch (error) {
    case MYERS_SUCCESS:                return "Myers - Success";
    case MYERS_E_OPENING_FILE:         return "Myers - Error: opening file";
    case MYERS_E_READING_FILE:         return "Myers - Error: reading file";
    case MYERS_E_INSUFFICIENT_MEM_GPU: return "Myers - Error: there aren't enough GPU memory space";
    case MYERS_E_ALLOCATE_MEM:         return "Myers - Error: allocating data";
    case MYERS_E_INCOMPATIBLE_GPU:     return "Myers - Error: incompatible GPU";
    case MYERS_E_INVALID_ARGUMENT:     return "Myers - Error: invalid argument";
    case MYERS_E_CAPACITY:             return "Myers - Error: batch exceeds the buffer capacity";
    case MYERS_E_HIP:                  return "Myers - Error: HIP runtime call failed";
    case MYERS_E_QUERY_TOO_LONG:       return "Myers - Error: query longer than the supported maximum";
    case MYERS_E_NO_DEVICE:            return "Myers - Error: no HIP device";
    case MYERS_E_REFERENCE_TOO_LARGE:  return "Myers - Error: reference too large";
    default:                           return "Myers - Unknown error";
    }
}

static int hip_fail(hipError_t e, const char *what, const char *file, int line)
{
    if (e == hipSuccess) return MYERS_SUCCESS;
    fprintf(stderr, "Myers - HIP error '%s' in %s (%s:%d)\n", hipGetErrorString(e), what, file, line);
    return MYERS_E_HIP;
}
#define HIP_TRY(call) do { int _rc = hip_fail((call), #call, __FILE__, __LINE__); if (_rc) return _rc; } while (0)

/* The reference prints and exits on any error (src-api/myersGPU.c:24-47);
 * buffers created by initMyers keep that behaviour for the void calls. */
static void report(myers_buffer_t *b, int rc, const char *where)
{
    if (b) b->last_error = rc;
    if (rc != MYERS_SUCCESS && (b == NULL || b->exit_on_error)) {
        fprintf(stderr, "%s in %s\n", myersGetErrorString(rc), where);
        exit(EXIT_FAILURE);
    }
}

/* ---------------------------------------------------------------- getters */

qryEntry_t *getPEQBuffer(void *myersBuffer)        { return ((myers_buffer_t *)myersBuffer)->h_peq; }
candInfo_t *getCandidatesBuffer(void *myersBuffer) { return ((myers_buffer_t *)myersBuffer)->h_cands; }
qryInfo_t  *getPEQInfoBuffer(void *myersBuffer)    { return ((myers_buffer_t *)myersBuffer)->h_qinfo; }
resEntry_t *getResultsBuffer(void *myersBuffer)    { return ((myers_buffer_t *)myersBuffer)->h_results; }
uint32_t getMaxPEQEntries(void *myersBuffer)       { return ((myers_buffer_t *)myersBuffer)->max_peq_entries; }
uint32_t getMaxCandidates(void *myersBuffer)       { return ((myers_buffer_t *)myersBuffer)->max_candidates; }
uint32_t getMaxQueries(void *myersBuffer)          { return ((myers_buffer_t *)myersBuffer)->max_queries; }
uint32_t myersGetNumBuffers(void *myersBuffer)     { return ((myers_buffer_t *)myersBuffer)->num_buffers; }
uint64_t myersGetReferenceSize(void *myersBuffer)  { return ((myers_buffer_t *)myersBuffer)->ctx->ref_size; }
int myersGetLastError(void *myersBuffer)           { return myersBuffer ? ((myers_buffer_t *)myersBuffer)->last_error : MYERS_E_INVALID_ARGUMENT; }
void *myersGetStream(void *myersBuffer)            { return (void *)((myers_buffer_t *)myersBuffer)->stream; }

void myersDefaultConfig(myersConfig_t *cfg)
{
    memset(cfg, 0, sizeof(*cfg));
    cfg->structSize = sizeof(*cfg);
    cfg->device = 0;
    cfg->exitOnError = 1;
    cfg->bufferBytes = 0;
}

/* ------------------------------------------------------------ bin table */

static uint32_t variant_cost(const myers_variant_desc_t *v)
{
    /* Estimated issue slots per candidate column: ~10 VALU ops per u32 word
     * plus ~12 per lane (text, score, minimum) and ~6 per lane for the
     * diagonal hand-over when L > 1.  Variants whose LDS leaves room for
     * fewer than two waves per SIMD (over 20 KB per one-wave workgroup)
     * cannot use the dual-issue rate of and/or/bitop3 and pay ~40%. */
    uint32_t cost = v->total_words * 10u + 12u * v->lanes + (v->lanes > 1u ? 6u * v->lanes : 0u);
    if (v->lds_bytes > 20u * 1024u) cost += (cost * 2u) / 5u;
    return cost;
}

/* Default length-bin table: for w query words pick the variant that covers
 * them with the least estimated VALU work per column. */
static void default_bin_table(myers_ctx_t *ctx)
{
    for (uint32_t w = 0; w <= MAX_QUERY_WORDS; w++) {
        uint32_t best = 0, best_cost = 0xFFFFFFFFu;
        for (uint32_t v = 0; v < ctx->num_variants; v++) {
            const myers_variant_desc_t *d = &ctx->variants[v];
            if (d->total_words < (w ? w : 1u)) continue;
            uint32_t cost = variant_cost(d);
            if (cost < best_cost) { best_cost = cost; best = v; }
        }
        ctx->bin_of_words[w] = (uint8_t)best;
    }
}

/* The bins of a batch.  A chunk of the sliced kernel holds reads of one word
 * count, so the persistent engine, whose launches take any number of bins, has one
 * per word count of the reads that the table gives a one-lane variant.  The engines
 * with a launch per bin keep the table's rows: with a bin per word count, 60K reads
 * of 200-1000 bases took 14.9 ms on the plain engine instead of 8.6. */
static int fine_bins(uint32_t flags)
{
    const uint32_t engine = flags & MYERS_ENGINE_MASK;
    return engine == MYERS_ENGINE_AUTO || engine == MYERS_ENGINE_PERSISTENT;
}

static const uint8_t *bins_of(const myers_ctx_t *ctx, uint32_t flags)
{
    return fine_bins(flags) ? ctx->fine_of_words : ctx->bin_of_words;
}

static int find_variant(const myers_ctx_t *ctx, uint32_t lanes, uint32_t words)
{
    for (uint32_t v = 0; v < ctx->num_variants; v++)
        if (ctx->variants[v].lanes == lanes && ctx->variants[v].words == words) return (int)v;
    return -1;
}

/* Derive fine_of_words from the table and copy both to the device. */
static int upload_bins(myers_ctx_t *ctx)
{
    for (uint32_t w = 0; w < BIN_ROWS; w++) {
        const uint32_t v = ctx->bin_of_words[w];
        const int one = ctx->variants[v].lanes == 1u ? find_variant(ctx, 1u, w ? w : 1u) : -1;
        ctx->fine_of_words[w] = one < 0 ? (uint8_t)v : (uint8_t)one;
    }
    HIP_TRY(hipMemcpy(ctx->d_bin_of_words, ctx->bin_of_words, BIN_ROWS, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(ctx->d_bin_of_words + BIN_ROWS, ctx->fine_of_words, BIN_ROWS, hipMemcpyHostToDevice));
    return MYERS_SUCCESS;
}

static uint32_t max_supported_words(const myers_ctx_t *ctx)
{
    uint32_t m = 0;
    for (uint32_t v = 0; v < ctx->num_variants; v++)
        if (ctx->variants[v].total_words > m) m = ctx->variants[v].total_words;
    return m < MAX_QUERY_WORDS ? m : MAX_QUERY_WORDS;
}

/* ------------------------------------------------------------- reference */

static int read_reference_file(const char *fn, uint32_t **words, uint64_t *num_words, uint64_t *size)
{
    FILE *fp = fopen(fn, "rb");
    if (fp == NULL) return MYERS_E_OPENING_FILE;
    uint32_t hdr[2];
    if (fread(hdr, sizeof(uint32_t), 2, fp) != 2) { fclose(fp); return MYERS_E_READING_FILE; }
    uint32_t *w = (uint32_t *)malloc(sizeof(uint32_t) * ((size_t)hdr[0] + 1u));
    if (w == NULL) { fclose(fp); return MYERS_E_ALLOCATE_MEM; }
    if (fread(w, sizeof(uint32_t), hdr[0], fp) != hdr[0]) { free(w); fclose(fp); return MYERS_E_READING_FILE; }
    fclose(fp);
    *words = w;
    *num_words = hdr[0];
    *size = hdr[1];
    return MYERS_SUCCESS;
}

/* The kernels index reference words with signed 32-bit offsets (a lane's
 * first text word can lie before the window, and reads are clamped to
 * [0, last word]), so the stored words plus the guard must stay below 2^31:
 * 17 Gbases, four times the largest .4bits.ref header (u32 base count). */
static int check_reference_size(uint64_t num_words, uint64_t size)
{
    if (num_words + GUARD_WORDS > (uint64_t)INT32_MAX) return MYERS_E_REFERENCE_TOO_LARGE;
    if (size > num_words * 8u) return MYERS_E_INVALID_ARGUMENT;
    return MYERS_SUCCESS;
}

static int upload_reference(myers_ctx_t *ctx, const uint32_t *words, uint64_t num_words, uint64_t size)
{
    int rc0 = check_reference_size(num_words, size);
    if (rc0) return rc0;
    size_t free_b = 0, total_b = 0;
    HIP_TRY(hipMemGetInfo(&free_b, &total_b));
    const uint64_t bytes = (num_words + GUARD_WORDS) * sizeof(uint32_t);
    const uint64_t blocks = (num_words + GUARD_WORDS + 3u) / 4u;        /* 32 bases each */
    if (bytes + 3u * sizeof(uint32_t) * blocks > free_b) return MYERS_E_INSUFFICIENT_MEM_GPU;
    HIP_TRY(hipMalloc((void **)&ctx->d_ref, bytes));
    HIP_TRY(hipMalloc((void **)&ctx->d_planes, 3u * sizeof(uint32_t) * blocks));
    /* Stream the words through a pinned staging buffer. */
    void *stage = NULL;
    size_t stage_bytes = STAGE_BYTES;
    if (stage_bytes > num_words * sizeof(uint32_t)) stage_bytes = num_words * sizeof(uint32_t) + 4u;
    HIP_TRY(hipHostMalloc(&stage, stage_bytes, hipHostMallocDefault));
    uint64_t done = 0;
    int rc = MYERS_SUCCESS;
    while (done < num_words && rc == MYERS_SUCCESS) {
        uint64_t n = stage_bytes / sizeof(uint32_t);
        if (n > num_words - done) n = num_words - done;
        memcpy(stage, words + done, n * sizeof(uint32_t));
        rc = hip_fail(hipMemcpy(ctx->d_ref + done, stage, n * sizeof(uint32_t), hipMemcpyHostToDevice),
                      "hipMemcpy(reference)", __FILE__, __LINE__);
        done += n;
    }
    hipHostFree(stage);
    if (rc) return rc;
    HIP_TRY(hipMemsetD32((hipDeviceptr_t)(ctx->d_ref + num_words), (int)ALL_N_WORD, GUARD_WORDS));
    rc = myers_launch_planes(ctx->d_ref, num_words + GUARD_WORDS, ctx->d_planes, (uint32_t)blocks, NULL);
    if (rc) return hip_fail((hipError_t)rc, "reference planes launch", __FILE__, __LINE__);
    HIP_TRY(hipDeviceSynchronize());
    ctx->plane_blocks = (uint32_t)blocks;
    ctx->ref_words = num_words;
    ctx->ref_words_alloc = num_words + GUARD_WORDS;
    ctx->ref_size = size;
    return MYERS_SUCCESS;
}

/* ---------------------------------------------------------------- buffers */

static void free_buffer(myers_buffer_t *b)
{
    if (b == NULL) return;
    if (b->h_peq) hipHostFree(b->h_peq);
    if (b->h_qinfo) hipHostFree(b->h_qinfo);
    if (b->h_cands) hipHostFree(b->h_cands);
    if (b->h_results) hipHostFree(b->h_results);
    if (b->h_err) hipHostFree(b->h_err);
    if (b->d_peq) hipFree(b->d_peq);
    if (b->d_qinfo) hipFree(b->d_qinfo);
    if (b->d_cands) hipFree(b->d_cands);
    if (b->d_results) hipFree(b->d_results);
    if (b->d_order) hipFree(b->d_order);
    if (b->d_work) hipFree(b->d_work);
    if (b->d_split) hipFree(b->d_split);
    if (b->ev_batch_start) hipEventDestroy(b->ev_batch_start);
    if (b->ev_batch_end) hipEventDestroy(b->ev_batch_end);
    for (uint32_t i = 0; i < EV_RING; i++) {
        for (uint32_t k = 0; k < 3; k++)
            if (b->ev_kernel[i][k]) hipEventDestroy(b->ev_kernel[i][k]);
    }
    if (b->graph_exec) hipGraphExecDestroy(b->graph_exec);
    for (uint32_t i = 0; i < SIDE_STREAMS; i++) {
        if (b->side[i]) hipStreamDestroy(b->side[i]);
        if (b->ev_join[i]) hipEventDestroy(b->ev_join[i]);
    }
    if (b->ev_fork) hipEventDestroy(b->ev_fork);
    if (b->stream) hipStreamDestroy(b->stream);
    free(b);
}

static int init_buffer(myers_buffer_t *b)
{
    const size_t peq_b = (size_t)b->max_peq_entries * sizeof(qryEntry_t);
    const size_t qi_b = (size_t)b->max_queries * sizeof(qryInfo_t);
    const size_t ca_b = (size_t)b->max_candidates * sizeof(candInfo_t);
    const size_t re_b = (size_t)b->max_candidates * sizeof(resEntry_t);
    HIP_TRY(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
    HIP_TRY(hipHostMalloc((void **)&b->h_peq, peq_b, hipHostMallocDefault));
    HIP_TRY(hipHostMalloc((void **)&b->h_qinfo, qi_b, hipHostMallocDefault));
    HIP_TRY(hipHostMalloc((void **)&b->h_cands, ca_b, hipHostMallocDefault));
    HIP_TRY(hipHostMalloc((void **)&b->h_results, re_b, hipHostMallocDefault));
    HIP_TRY(hipHostMalloc((void **)&b->h_err, sizeof(uint32_t), hipHostMallocDefault));
    HIP_TRY(hipHostGetDevicePointer((void **)&b->d_err, b->h_err, 0));
    HIP_TRY(hipHostGetDevicePointer(&b->hd_peq, b->h_peq, 0));
    HIP_TRY(hipHostGetDevicePointer(&b->hd_qinfo, b->h_qinfo, 0));
    HIP_TRY(hipHostGetDevicePointer(&b->hd_cands, b->h_cands, 0));
    HIP_TRY(hipHostGetDevicePointer(&b->hd_results, b->h_results, 0));
    HIP_TRY(hipMalloc((void **)&b->d_peq, peq_b));
    HIP_TRY(hipMalloc((void **)&b->d_qinfo, qi_b));
    HIP_TRY(hipMalloc((void **)&b->d_cands, ca_b));
    HIP_TRY(hipMalloc((void **)&b->d_results, re_b));
    HIP_TRY(hipMalloc((void **)&b->d_order, (size_t)b->max_candidates * sizeof(uint32_t)));
    HIP_TRY(hipMalloc((void **)&b->d_work, MYERS_WORK_WORDS * sizeof(uint32_t)));
    for (uint32_t i = 0; i < SIDE_STREAMS; i++) {
        HIP_TRY(hipStreamCreateWithFlags(&b->side[i], hipStreamNonBlocking));
        HIP_TRY(hipEventCreateWithFlags(&b->ev_join[i], hipEventDisableTiming));
    }
    HIP_TRY(hipEventCreateWithFlags(&b->ev_fork, hipEventDisableTiming));
    HIP_TRY(hipEventCreate(&b->ev_batch_start));
    HIP_TRY(hipEventCreate(&b->ev_batch_end));
    for (uint32_t i = 0; i < EV_RING; i++) {
        for (uint32_t k = 0; k < 3; k++) HIP_TRY(hipEventCreate(&b->ev_kernel[i][k]));
    }
    memset(b->h_results, 0, re_b);
    *b->h_err = 0;
    b->stats.structSize = sizeof(myersStats_t);
    b->mark_slot = -1;
    return MYERS_SUCCESS;
}

static int create_context(myers_ctx_t **out, int device)
{
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return MYERS_E_NO_DEVICE;
    if (device < 0 || device >= ndev) return MYERS_E_INVALID_ARGUMENT;
    HIP_TRY(hipSetDevice(device));
    myers_ctx_t *ctx = (myers_ctx_t *)calloc(1, sizeof(myers_ctx_t));
    if (ctx == NULL) return MYERS_E_ALLOCATE_MEM;
    ctx->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) { free(ctx); return MYERS_E_HIP; }
    ctx->num_cus = prop.multiProcessorCount;
    /* the allocation-free entry point's static workspace on this device */
    if (myers_scratch_init(device, &ctx->d_scratch) != 0) {
        free(ctx);
        return MYERS_E_HIP;
    }
    ctx->num_variants = myers_num_variants();
    for (uint32_t v = 0; v < ctx->num_variants; v++) {
        myers_variant_desc(v, &ctx->variants[v]);
        int occ = 0;
        if (myers_variant_occupancy(v, &occ) != 0 || occ <= 0) occ = 1;
        ctx->occupancy[v] = occ;
        occ = 0;
        if (myers_variant_occupancy_persistent(v, &occ) != 0 || occ <= 0) occ = 1;
        ctx->occupancy_p[v] = occ;
        ctx->chunk_factor[v] = 1u;
        if (ctx->variants[v].lanes > 1u) ctx->multi_lane |= 1ull << v;
        else if (ctx->variants[v].words >= 8u) ctx->deep |= 1ull << v;
    }
    default_bin_table(ctx);
    if (hipMalloc((void **)&ctx->d_bin_of_words, 2u * BIN_ROWS) != hipSuccess) {
        free(ctx);
        return MYERS_E_HIP;
    }
    if (upload_bins(ctx) != MYERS_SUCCESS) {
        hipFree(ctx->d_bin_of_words);
        free(ctx);
        return MYERS_E_HIP;
    }
    load_default_tuning(ctx);
    *out = ctx;
    return MYERS_SUCCESS;
}

static void free_context(myers_ctx_t *ctx)
{
    if (ctx == NULL) return;
    if (ctx->d_ref) hipFree(ctx->d_ref);
    if (ctx->d_planes) hipFree(ctx->d_planes);
    if (ctx->d_bin_of_words) hipFree(ctx->d_bin_of_words);
    free(ctx);
}

/* Capacities from the per-buffer byte budget, with the reference's formulas
 * (src-api/myersGPU.c:312-330). */
static int size_buffers(myers_ctx_t *ctx, uint32_t num_buffers, int32_t avg_query, int32_t cands_per_query,
                        uint64_t buffer_bytes, uint32_t *max_cands, uint32_t *max_queries, uint32_t *max_peq)
{
    if (avg_query <= 0) avg_query = 1024;
    if (cands_per_query <= 0) cands_per_query = 1;
    size_t free_b = 0, total_b = 0;
    HIP_TRY(hipMemGetInfo(&free_b, &total_b));
    uint64_t budget = buffer_bytes;
    if (budget == 0) {
        budget = (uint64_t)((double)free_b * 0.95) / num_buffers;
        if (budget > DEFAULT_BUFFER_CAP) budget = DEFAULT_BUFFER_CAP;
    }
    if (budget * num_buffers > (uint64_t)free_b) return MYERS_E_INSUFFICIENT_MEM_GPU;
    const uint32_t entries = ((uint32_t)avg_query + 127u) / 128u;
    const double per_cand = ((double)entries * sizeof(qryEntry_t) + sizeof(qryInfo_t)) / cands_per_query
                            + sizeof(candInfo_t) + sizeof(resEntry_t) + sizeof(uint32_t);
    double mc = (double)budget / per_cand;
    if (mc > 4.0e9) mc = 4.0e9;
    *max_cands = (uint32_t)mc;
    *max_queries = *max_cands / (uint32_t)cands_per_query;
    double mp = (double)(*max_queries) * entries;
    if (mp > 4.0e9) mp = 4.0e9;
    *max_peq = (uint32_t)mp;
    (void)ctx;
    if (*max_cands < 1u || *max_queries < 1u) return MYERS_E_INSUFFICIENT_MEM_GPU;
    return MYERS_SUCCESS;
}

static int init_common(void ***out, uint32_t num_buffers, const uint32_t *words, uint64_t num_words,
                       uint64_t size, int32_t avg_query, int32_t cands_per_query, const myersConfig_t *cfg_in)
{
    if (out == NULL || num_buffers == 0 || words == NULL) return MYERS_E_INVALID_ARGUMENT;
    int rc = check_reference_size(num_words, size);      /* before any device work */
    if (rc) return rc;
    myersConfig_t cfg;
    myersDefaultConfig(&cfg);
    if (cfg_in) cfg = *cfg_in;
    *out = NULL;
    myers_ctx_t *ctx = NULL;
    rc = create_context(&ctx, cfg.device);
    if (rc) return rc;
    rc = upload_reference(ctx, words, num_words, size);
    if (rc) { free_context(ctx); return rc; }
    uint32_t mc = 0, mq = 0, mp = 0;
    rc = size_buffers(ctx, num_buffers, avg_query, cands_per_query, cfg.bufferBytes, &mc, &mq, &mp);
    if (rc) { free_context(ctx); return rc; }
    myers_buffer_t **bufs = (myers_buffer_t **)calloc(num_buffers, sizeof(myers_buffer_t *));
    if (bufs == NULL) { free_context(ctx); return MYERS_E_ALLOCATE_MEM; }
    for (uint32_t i = 0; i < num_buffers && rc == MYERS_SUCCESS; i++) {
        myers_buffer_t *b = (myers_buffer_t *)calloc(1, sizeof(myers_buffer_t));
        if (b == NULL) { rc = MYERS_E_ALLOCATE_MEM; break; }
        bufs[i] = b;
        b->ctx = ctx;
        b->num_buffers = num_buffers;
        b->id_buffer = i;
        b->max_candidates = mc;
        b->max_queries = mq;
        b->max_peq_entries = mp;
        b->exit_on_error = cfg.exitOnError;
        b->threshold = -1.0f;
        rc = init_buffer(b);
    }
    if (rc) {
        for (uint32_t i = 0; i < num_buffers; i++) free_buffer(bufs[i]);
        free(bufs);
        free_context(ctx);
        return rc;
    }
    *out = (void **)bufs;
    return MYERS_SUCCESS;
}

int myersInitFromMemory(void ***myersBuffer, uint32_t numBuffers, const uint32_t *refWords,
                        uint64_t numWords, uint64_t refSize, int32_t averageQuerySize,
                        int32_t candidatesPerQuery, const myersConfig_t *cfg)
{
    return init_common(myersBuffer, numBuffers, refWords, numWords, refSize, averageQuerySize,
                       candidatesPerQuery, cfg);
}

int myersInitEx(void ***myersBuffer, uint32_t numBuffers, const char *referenceFileName,
                int32_t averageQuerySize, int32_t candidatesPerQuery, const myersConfig_t *cfg)
{
    if (referenceFileName == NULL) return MYERS_E_INVALID_ARGUMENT;
    uint32_t *words = NULL;
    uint64_t nw = 0, size = 0;
    int rc = read_reference_file(referenceFileName, &words, &nw, &size);
    if (rc) return rc;
    rc = init_common(myersBuffer, numBuffers, words, nw, size, averageQuerySize, candidatesPerQuery, cfg);
    free(words);
    return rc;
}

int initMyers(void ***myersBuffer, uint32_t numBuffers, const char *referenceFileName,
              int32_t averageQuerySize, int32_t candidatesPerQuery)
{
    return myersInitEx(myersBuffer, numBuffers, referenceFileName, averageQuerySize,
                       candidatesPerQuery, NULL);
}

int myersEnd(void ***myersBuffer)
{
    if (myersBuffer == NULL || *myersBuffer == NULL) return MYERS_E_INVALID_ARGUMENT;
    myers_buffer_t **bufs = (myers_buffer_t **)(*myersBuffer);
    myers_ctx_t *ctx = bufs[0]->ctx;
    const uint32_t n = bufs[0]->num_buffers;
    hipSetDevice(ctx->device);
    int rc = hip_fail(hipDeviceSynchronize(), "hipDeviceSynchronize", __FILE__, __LINE__);
    for (uint32_t i = 0; i < n; i++) free_buffer(bufs[i]);
    free(bufs);
    free_context(ctx);   /* the shared reference is freed once */
    *myersBuffer = NULL;
    return rc;
}

void endMyers(void ***myersBuffer)
{
    int rc = myersEnd(myersBuffer);
    if (rc) {
        fprintf(stderr, "%s in endMyers\n", myersGetErrorString(rc));
        exit(EXIT_FAILURE);
    }
}

/* ----------------------------------------------------------------- launch */

typedef struct {
    uint64_t present;      /* bitmask of variants present */
    uint32_t num_present;
    uint32_t single;       /* the variant when num_present == 1 */
    int      too_long;
    int      sized;        /* reads[] / max_m[] below are filled in */
    uint32_t reads[MYERS_MAX_VARIANTS];   /* reads per variant */
    uint32_t max_m[MYERS_MAX_VARIANTS];   /* longest read per variant (up to 32 words perhaps the longest it could be) */
    int      counted;      /* cands[] below is filled in */
    uint32_t cands[MYERS_MAX_VARIANTS];   /* candidates per variant */
} bin_scan_t;

#define SCAN_HIST_READS 2048u
static void scan_qinfo(const myers_ctx_t *ctx, const uint8_t *bins, const qryInfo_t *qinfo, uint32_t nq, bin_scan_t *s)
{
    const uint32_t maxw = max_supported_words(ctx);
    memset(s, 0, sizeof(*s));
    s->sized = 1;
    uint32_t q = 0;
    if (nq >= SCAN_HIST_READS) {
        /* reads per word count first, in four counts so that neighbours of one
         * length do not wait for each other's increment (0.45 ns per read against
         * 1.0 read by read); the longest read only where it is asked for */
        uint32_t hist[4][MAX_QUERY_WORDS + 2];
        uint32_t top[MAX_QUERY_WORDS + 2];
        memset(hist, 0, sizeof(hist));
        memset(top, 0, sizeof(top));
        for (; q + 4u <= nq; q += 4u) {
            for (uint32_t k = 0; k < 4u; k++) {
                const uint32_t m = qinfo[q + k].size;
                uint32_t w = (m + 31u) >> 5;
                if (w > 32u) {
                    if (w > maxw) w = MAX_QUERY_WORDS + 1u;
                    if (m > top[w]) top[w] = m;
                }
                hist[k][w]++;
            }
        }
        if (hist[0][MAX_QUERY_WORDS + 1u] | hist[1][MAX_QUERY_WORDS + 1u] | hist[2][MAX_QUERY_WORDS + 1u] |
            hist[3][MAX_QUERY_WORDS + 1u])
            s->too_long = 1;
        for (uint32_t w = 0; w <= maxw; w++) {
            const uint32_t reads = hist[0][w] + hist[1][w] + hist[2][w] + hist[3][w];
            if (reads == 0) continue;
            const uint32_t v = bins[w], m = w > 32u ? top[w] : 32u * w;
            s->present |= 1ull << v;
            s->reads[v] += reads;
            if (m > s->max_m[v]) s->max_m[v] = m;
        }
    }
    for (; q < nq; q++) {
        const uint32_t m = qinfo[q].size;
        uint32_t w = (m + 31u) >> 5;
        if (w > maxw) { s->too_long = 1; continue; }
        const uint32_t v = bins[w];
        s->present |= 1ull << v;
        s->reads[v]++;
        if (m > s->max_m[v]) s->max_m[v] = m;
    }
    for (uint32_t v = 0; v < ctx->num_variants; v++)
        if (s->present & (1ull << v)) { s->num_present++; s->single = v; }
}

static uint32_t grid_for(const myers_ctx_t *ctx, uint32_t v, uint32_t count, int persistent)
{
    const uint32_t slots = ctx->variants[v].slots;
    uint64_t chunks = ((uint64_t)count + slots - 1u) / slots;
    if (chunks == 0) chunks = 1;
    if (persistent) {
        uint64_t resident = (uint64_t)ctx->num_cus * (uint64_t)ctx->occupancy[v];
        /* keep the grid a multiple of 8 (one share per XCD) */
        resident = (resident + 7u) & ~7ull;
        if (chunks > resident) chunks = resident;
    }
    if (chunks > 0x7FFFFFFFull) chunks = 0x7FFFFFFFull;
    return (uint32_t)chunks;
}

/* Fold the oldest timed batch into the stats (waits for its end event). */
static int fold_oldest_timing(myers_buffer_t *b)
{
    const uint32_t slot = (b->ev_head + EV_RING - b->ev_pending) % EV_RING;
    int rc = hip_fail(hipEventSynchronize(b->ev_kernel[slot][1]), "hipEventSynchronize", __FILE__, __LINE__);
    if (rc) return rc;
    float ms = 0.0f, vms = 0.0f;
    if (hipEventElapsedTime(&ms, b->ev_kernel[slot][0], b->ev_kernel[slot][1]) == hipSuccess) {
        if (!b->ev_marked[slot] ||
            hipEventElapsedTime(&vms, b->ev_kernel[slot][2], b->ev_kernel[slot][1]) != hipSuccess)
            vms = ms;
        b->stats.kernelMs = ms;
        b->stats.kernelMsTotal += ms;
        b->stats.verifyMs = vms;
        b->stats.verifyMsTotal += vms;
        b->stats.kernelLaunchesTotal += b->ev_launches[slot];
        b->stats.batchesTotal++;
    }
    b->ev_pending--;
    return MYERS_SUCCESS;
}

static int timing_begin(myers_buffer_t *b, uint32_t *slot)
{
    if (b->ev_pending == EV_RING) {
        int rc = fold_oldest_timing(b);
        if (rc) return rc;
    }
    *slot = b->ev_head;
    b->ev_marked[*slot] = 0;
    return hip_fail(hipEventRecord(b->ev_kernel[*slot][0], b->stream), "hipEventRecord", __FILE__, __LINE__);
}

static int timing_end(myers_buffer_t *b, uint32_t slot, uint32_t launches)
{
    int rc = hip_fail(hipEventRecord(b->ev_kernel[slot][1], b->stream), "hipEventRecord", __FILE__, __LINE__);
    if (rc) return rc;
    b->ev_launches[slot] = launches;
    b->ev_head = (slot + 1u) % EV_RING;
    b->ev_pending++;
    return MYERS_SUCCESS;
}

typedef struct {
    const void *d_peq, *d_qinfo, *d_cands;
    void       *d_results;
    uint32_t    num_entries, num_queries, num_cands, flags;
    float       distance;
    float       threshold;
    uint32_t   *d_work;      /* MYERS_WORK_WORDS of pipeline workspace */
    uint32_t   *d_order;     /* slot -> candidate, num_cands words */
    uint32_t   *d_list;      /* num_cands words, or NULL */
    myers_buffer_t *pool_of; /* the buffer whose pool the split launch may use, or NULL */
    double      share;       /* of the chip that the batch can expect (chip_share) */
} batch_t;

static int large_batch(const myers_ctx_t *ctx, uint32_t num_cands)
{
    return (uint64_t)num_cands >= (uint64_t)ctx->num_cus * 2048u;
}

/* Threshold mode: whether the one-lane launch runs the first rows of its candidates
 * first (slice_first_rows) and the rest of those kept in a second launch.
 *
 * The rows left out save their share of the bins' time, which batches of a round
 * or two of waves spend at about 125e12 cells per second; the second launch takes
 * one chunk of its kernel and 0.25 ms of launches, binning and tail.  8 candidates
 * per read, threshold 0.05 m, all rows and first rows: 100K candidates of 1000 bases
 * 1.04 and 1.15 ms, 150K 1.33 and 1.17; 100K of 800 0.69 and 0.84, 200K 1.15 and
 * 0.92; 150K of 600 0.55 and 0.60, 400K 1.13 and 0.89; 250K of six lengths from 100
 * to 1000 1.08 and 1.12. */
#define FIRST_ROWS_MIN_CANDS 384u        /* per CU: below, all rows whatever the reads */
static int first_rows_pay(const myers_ctx_t *ctx, const bin_scan_t *scan, const batch_t *bt)
{
    if (bt->threshold < 0.0f || bt->d_list == NULL || bt->num_queries == 0 ||
        (uint64_t)bt->num_cands < (uint64_t)FIRST_ROWS_MIN_CANDS * (uint64_t)ctx->num_cus)
        return 0;
    if (!scan->sized) return (uint64_t)bt->num_cands >= 1024u * (uint64_t)ctx->num_cus;
    const double cpr = (double)bt->num_cands / (double)bt->num_queries;
    double saved = 0.0, second = 0.0;                /* ns */
    for (uint64_t left = scan->present & ~ctx->multi_lane; left; left &= left - 1u) {
        const uint32_t v = (uint32_t)__builtin_ctzll(left);
        const double m = 32.0 * (double)ctx->variants[v].words;
        const double share = myers_slice_first_rows(ctx->variants[v].words, bt->threshold) * 32.0 / m;
        if (share <= 0.0) continue;
        const double cands = scan->counted ? (double)scan->cands[v] : (double)scan->reads[v] * cpr;
        const double chunk = (1.25 * m + 96.0) * (60.0 + 28.0 * (double)((ctx->variants[v].words + 1u) / 2u));
        saved += (1.0 - share) * cands * 1.2 * m * m / 125e3;
        if (chunk > second) second = chunk;
    }
    return saved > second + 250e3;
}

/* Auto: mixed lengths go to the persistent engine.  A batch of one length bin
 * runs on the plain engine (no binning pass) unless it holds more than ~2.7
 * rounds of what the chip keeps resident (2048 candidates per CU): there the
 * queue launch's pulls leave a shorter tail than one workgroup per chunk
 * (1.1M candidates of 1,000 bases: 8.70 against 8.78 ms), or threshold mode's first
 * rows pay, which need the binning's ranges. */
static uint32_t resolve_engine(const myers_ctx_t *ctx, const bin_scan_t *scan, const batch_t *bt, int first_rows)
{
    uint32_t engine = bt->flags & MYERS_ENGINE_MASK;
    if (engine == MYERS_ENGINE_AUTO) {
        const int single = scan->num_present == 1 && !scan->too_long;
        engine = (single && !large_batch(ctx, bt->num_cands) && !first_rows) ? MYERS_ENGINE_PLAIN : MYERS_ENGINE_PERSISTENT;
    }
    return engine;
}

/* Variants present, most words first (longest candidates start first). */
static uint32_t present_by_cost(const myers_ctx_t *ctx, uint64_t present, uint32_t *out)
{
    uint32_t n = 0;
    for (; present; present &= present - 1u) out[n++] = (uint32_t)__builtin_ctzll(present);
    for (uint32_t i = 1; i < n; i++) {
        uint32_t x = out[i], j = i;
        while (j > 0 && ctx->variants[out[j - 1]].total_words < ctx->variants[x].total_words) {
            out[j] = out[j - 1];
            j--;
        }
        out[j] = x;
    }
    return n;
}

/* Long-read bins of a persistent batch that go into one launch
 * (myers_launch_long): bins of 4..64 lanes per candidate, longest reads
 * first, when their chunks (counted from the host's candidates, or estimated
 * from the reads per bin and the batch's candidates per read) fit a few
 * rounds of one wave per SIMD.  Such bins are
 * bound by each candidate's chain of column steps; larger long-read batches
 * are throughput work and keep one launch per bin.
 *
 * A bin of reads over 256 words can instead run each candidate on a whole
 * 4-wave workgroup, which shortens its chain (measured: 20,000 bases in 2.9 ms
 * against 5.9 ms on one wave) for 4 SIMDs instead of one.  The plan widens
 * the bin with the longest estimated chain while that lowers the estimated
 * time of the launch, max(longest chain, SIMD-time of all items / SIMDs).
 * Per column step, from single-candidate runs: one wave of W words per lane
 * ~40 + 20 W ns, a workgroup of W words per lane ~63 + 18.5 W ns.  Returns the
 * bins taken (0: none) and the estimated time. */
#define LONG_ROUNDS 4u
static double chain_ns(uint32_t max_m, uint32_t lanes, uint32_t words, int wide)
{
    const double steps = 1.2 * (double)max_m + (double)lanes;
    return steps * (wide ? 63.0 + 18.5 * (double)words : 40.0 + 20.0 * (double)words);
}

static uint32_t long_plan(const myers_ctx_t *ctx, const bin_scan_t *scan, const batch_t *bt,
                          const uint32_t *order, uint32_t n, myers_long_plan_t *lp, double *ns)
{
    memset(lp, 0, sizeof(*lp));
    if (ns) *ns = 0.0;
    if (!scan->sized || bt->num_queries == 0) return 0;
    const double cpr = (double)bt->num_cands / (double)bt->num_queries;
    const double simds = (double)MYERS_LONG_WAVES * (double)ctx->num_cus;
    const uint32_t wide_lanes = 64u * MYERS_LONG_WAVES;
    uint32_t take[MYERS_LONG_MAX], nt = 0;
    double waves[MYERS_LONG_MAX], chain[MYERS_LONG_MAX], total_waves = 0.0, work = 0.0;
    int wide[MYERS_LONG_MAX] = {0};
    for (uint32_t i = 0; i < n && nt < MYERS_LONG_MAX; i++) {
        const uint32_t v = order[i];
        if (!myers_variant_long_ok(v, NULL)) continue;
        const myers_variant_desc_t *d = &ctx->variants[v];
        const double cands = scan->counted ? (double)scan->cands[v] : (double)scan->reads[v] * cpr;
        waves[nt] = cands / (double)d->slots;
        chain[nt] = cands > 0.0 ? chain_ns(scan->max_m[v], d->lanes, d->words, 0) : 0.0;
        total_waves += waves[nt];
        work += waves[nt] * chain[nt];
        take[nt++] = v;
    }
    if (nt == 0 || total_waves > (double)LONG_ROUNDS * simds) return 0;
    for (;;) {
        uint32_t top = 0;
        double longest = 0.0;
        for (uint32_t k = 0; k < nt; k++)
            if (chain[k] > longest) { longest = chain[k]; top = k; }
        const myers_variant_desc_t *d = &ctx->variants[take[top]];
        if (longest <= 0.0 || wide[top] || d->total_words <= wide_lanes ||
            d->total_words > wide_lanes * MYERS_WIDE_MAX_WORDS)
            break;
        const uint32_t ww = (d->total_words + wide_lanes - 1u) / wide_lanes;
        const double cands = waves[top] * (double)d->slots;
        const double c_wide = chain_ns(scan->max_m[take[top]], wide_lanes, ww, 1);
        const double work_wide = work - waves[top] * chain[top] + (double)MYERS_LONG_WAVES * cands * c_wide;
        double next = c_wide;
        for (uint32_t k = 0; k < nt; k++)
            if (k != top && chain[k] > next) next = chain[k];
        const double before = longest > work / simds ? longest : work / simds;
        const double after = next > work_wide / simds ? next : work_wide / simds;
        if (after >= before) break;
        wide[top] = 1;
        chain[top] = c_wide;
        work = work_wide;
    }
    if (ns) {
        *ns = work / (simds * bt->share);
        for (uint32_t k = 0; k < nt; k++)
            if (chain[k] > *ns) *ns = chain[k];
    }
    for (uint32_t k = 0; k < nt; k++) {            /* wide bins keep the longest-first order */
        const uint32_t v = take[k];
        const uint32_t words = ctx->variants[v].total_words;
        if (wide[k]) {
            lp->wide_variant[lp->n_wide] = v;
            lp->wide_words[lp->n_wide] = (words + wide_lanes - 1u) / wide_lanes;
            lp->n_wide++;
            continue;
        }
        uint32_t u4 = 0;
        myers_variant_long_ok(v, &u4);
        lp->variant[lp->n] = v;
        lp->key[lp->n] = (ctx->variants[v].lanes << 8) | ctx->variants[v].words;
        lp->n++;
        if (u4 > lp->ws_u4) lp->ws_u4 = u4;
    }
    if (lp->n_wide) {
        const uint32_t u4 = (myers_long_wide_lds_bytes() + 16u * MYERS_LONG_WAVES - 1u) / (16u * MYERS_LONG_WAVES);
        if (u4 > lp->ws_u4) lp->ws_u4 = u4;
    }
    return nt;
}

/* Workgroups of a resident grid of the multi-lane queue kernel (which = 0, 1:
 * its threshold form) or a one-lane kernel (2: 16 lanes per group, 3: 32) with
 * `lds` bytes of dynamic LDS (queried once per size). */
static uint32_t queue_grid(myers_ctx_t *ctx, uint32_t which, uint32_t lds)
{
    if (ctx->queue_occ_lds[which] != lds) {
        int occ = 0;
        const int rc = which >= 2u ? myers_slice_occupancy(16u * (which - 1u), lds, &occ) : myers_queue_occupancy((int)which, lds, &occ);
        if (rc != 0 || occ <= 0) occ = 1;
        ctx->queue_occ[which] = occ;
        ctx->queue_occ_lds[which] = lds;
    }
    return (uint32_t)ctx->num_cus * (uint32_t)ctx->queue_occ[which];
}

/* How a batch's one-lane bins run: see slice_lanes(). */
typedef struct {
    uint32_t num_cands;
    double   per_wave;      /* work of the batch's one-lane bins, in the unit of slice_lanes(), per wave that the chip
                               holds (0: not known) */
    int      binned;
} slice_load_t;

static slice_load_t slice_load(const myers_ctx_t *ctx, const bin_scan_t *scan, uint32_t num_queries,
                               uint32_t num_cands, int binned)
{
    slice_load_t l = {num_cands, 0.0, binned};
    if (!scan->sized || num_queries == 0) return l;
    double work = 0.0;
    for (uint64_t left = scan->present & ~ctx->multi_lane; left; left &= left - 1u) {
        const uint32_t v = (uint32_t)__builtin_ctzll(left);
        const double w = (double)ctx->variants[v].words;
        work += (double)scan->reads[v] * w * w;
    }
    l.per_wave = work * (double)num_cands / (double)num_queries / 64.0 / (12.0 * (double)ctx->num_cus);
    return l;
}

/* Form of the one-lane kernels for a bin of reads of up to `words` words.
 *
 * Chunks of 128 candidates (16 lanes per group) spend less beside the
 * recurrence than chunks of 64 (32 lanes) but take twice as long each (about
 * 2 words^2 in units of words^2), so a bin takes them where the batch's work
 * is 1.5 of its chunks or more per wave (880K candidates of 100 bases: 300 us
 * of kernels with 16 lanes, 374 with 32; 1.65M of 36-400 bases 736 us, 818
 * with 32 lanes for all and 739 with 16 for all up to 384 bases) and the batch
 * is large enough for the second launch (440K of 50, 100 and 150 bases: 280 us
 * with both forms, 250 with 32 lanes).
 *
 * Batches that fill the chip for a few chunks only, of short reads, are bound
 * by the latency of a chunk, which is less for the bit-vector kernel (one
 * candidate per lane): 110K candidates of 100 bases 32 us against 41, 440K 85
 * against 102; from 8 words on the sliced form is faster at every size (250
 * bases, 5.5K candidates: 73 against 80 us). */
static uint32_t slice_lanes(const myers_ctx_t *ctx, uint32_t words, const slice_load_t *l)
{
    const uint64_t few = (uint64_t)ctx->num_cus * (l->binned ? 1024u : 2048u);
    if (words <= myers_slice_max_words(1u) && l->num_cands < few) return 1u;
    const double w = (double)words;
    return words <= myers_slice_max_words(16u) && (uint64_t)l->num_cands >= (uint64_t)ctx->num_cus * 2048u &&
                   3.0 * w * w <= l->per_wave ? 16u : 32u;
}

/* Add variant v (one lane) to a plan of the one-lane kernel with this form. */
static void slice_plan_add(const myers_ctx_t *ctx, myers_queue_plan_t *p, uint32_t v, uint32_t lanes)
{
    const uint32_t words = ctx->variants[v].words;
    const uint32_t u4 = myers_slice_ws_u4(lanes, words);
    p->cls = lanes == 16u ? MYERS_QUEUE_ONE_LANE_16 : MYERS_QUEUE_ONE_LANE;
    p->variant[p->n] = v;
    p->key[p->n] = (lanes << 8) | words;
    p->n++;
    if (u4 > p->ws_u4) p->ws_u4 = u4;
}

/* The bins of a batch whose reads of over 1024 bases run the sliced kernel
 * (myers_launch_wide_slice): all of them, or none.
 *
 * That kernel has about 1.6 times the rate of the multi-lane bit-vector
 * kernels, but a chunk of 32 candidates takes as long as many rounds of
 * theirs, so it pays where the batch fills the chip with chunks.  Both times
 * are estimated, a bin's mean read counting 0.8 of its longest: a step of 12
 * waves costs 28 ns per row of a lane and 60 ns beside (T waves per chunk, steps
 * for 1.25 m columns and the lag over the waves) and the last chunks leave 0.4
 * of one chunk's time idle; the bit-vector kernels run 120e12 cells per second
 * behind one candidate's chain (in threshold mode they stop unrelated
 * candidates before the window's end).  1000-4000 bases, 4 candidates each:
 * 16,000 reads 3.9 ms against 5.4 bit-vector, 8,000 reads 3.8 against 3.1; 2-20
 * kb: 20,000 reads 46 against 68 (threshold mode, k of 0.2 m: 62), 6,400 reads
 * 22.6 and 22.6, 3,200 reads 22.1 against 12.5. */
static uint64_t wide_bins(const myers_ctx_t *ctx, const bin_scan_t *scan, const batch_t *bt)
{
    const uint32_t engine = bt->flags & MYERS_ENGINE_MASK;
    if (!(scan->present & ctx->multi_lane) || !scan->sized || scan->too_long || bt->num_queries == 0 ||
        (engine != MYERS_ENGINE_AUTO && engine != MYERS_ENGINE_PERSISTENT))
        return 0;
    const double cpr = (double)bt->num_cands / (double)bt->num_queries;
    uint64_t mask = 0;
    double cells = 0.0, old_chain = 0.0, work = 0.0, longest = 0.0;      /* times in ns */
    for (uint32_t v = 0; v < ctx->num_variants; v++) {
        const myers_variant_desc_t *d = &ctx->variants[v];
        if (!(scan->present & (1ull << v)) || d->lanes == 1u) continue;
        const uint32_t team = myers_wide_slice_team(d->total_words);
        const double cands = scan->counted ? (double)scan->cands[v] : (double)scan->reads[v] * cpr;
        if (team == 0u) return 0;
        if (cands <= 0.0) continue;
        const double m = (double)scan->max_m[v];
        const double rows = (double)((scan->max_m[v] + 64u * team - 1u) / (64u * team));
        const double chunk = (1.25 * m + 96.0 * team) * (60.0 + 28.0 * rows);
        const uint32_t four = 64u * MYERS_LONG_WAVES;
        const double chain = d->total_words > four
                                 ? chain_ns(scan->max_m[v], four, (d->total_words + four - 1u) / four, 1)
                                 : chain_ns(scan->max_m[v], d->lanes, d->words, 0);
        work += (1.0 + 0.8 * cands / (32.0 * (MYERS_WIDE_SLICE_WAVES / team))) * chunk;
        cells += 0.8 * cands * 1.25 * m * m;
        if (chunk > longest) longest = chunk;
        if (chain > old_chain) old_chain = chain;
        mask |= 1ull << v;
    }
    const double wide = work / (double)ctx->num_cus + 0.4 * longest;
    double stop = bt->threshold >= 0.0f ? 0.78 + 0.65 * (double)bt->threshold : 1.0;
    if (stop > 1.0) stop = 1.0;
    return (wide > longest ? wide : longest) < stop * cells / 120e3 + old_chain ? mask : 0;
}

/* Estimate of a split launch (myers_launch_split), in ns.
 *
 * A step of a part costs about as much as its instructions of a wave alone on
 * its SIMD, so parts of few words shorten a candidate's chain but spend more
 * of the chip on it, and a second wave per SIMD gains some throughput for longer
 * chains.  Measured ns per step of a part, and of a SIMD's time per step: `kinds`.
 * A batch takes the longer of its longest chain (every part runs about 130
 * columns behind the one below) and the work over all SIMDs, and 0.3 of a chain
 * more where it is more than one part per wave. */
enum { SPLIT_KINDS = 6 };
static const struct { uint32_t words, per_simd; double chain, work; } split_kinds[SPLIT_KINDS] = {
    {1u, 1u, 52.0, 52.0}, {1u, 2u, 75.0, 47.0}, {2u, 1u, 70.0, 70.0}, {2u, 2u, 95.0, 59.0},
    {4u, 1u, 105.0, 105.0}, {4u, 2u, 180.0, 85.0}};
typedef struct {
    double chain[SPLIT_KINDS], work[SPLIT_KINDS], items[SPLIT_KINDS];
} split_est_t;

static void split_est_add(split_est_t *e, uint32_t total_words, double m, double cands)
{
    for (uint32_t k = 0; k < (uint32_t)SPLIT_KINDS; k++) {
        const uint32_t w = 64u * split_kinds[k].words;
        const double parts = (double)((total_words + w - 1u) / w);
        const double ns = (1.25 * m + 64.0 + 130.0 * (parts - 1.0)) * split_kinds[k].chain;
        if (ns > e->chain[k]) e->chain[k] = ns;
        e->items[k] += cands * parts;
        e->work[k] += 0.9 * cands * parts * (1.25 * m + 64.0) * split_kinds[k].work;
    }
}

static double split_est_ns(const split_est_t *e, double simds, uint32_t *best)
{
    double least = 0.0;
    for (uint32_t k = 0; k < (uint32_t)SPLIT_KINDS; k++) {
        double ns = e->work[k] / simds;
        if (e->items[k] > simds * split_kinds[k].per_simd) ns += 0.3 * e->chain[k];
        if (ns < e->chain[k]) ns = e->chain[k];
        if (k == 0 || ns < least) {
            least = ns;
            *best = k;
        }
    }
    return least;
}

/* The split launch's pool of a buffer, allocated (12.6 MB, 0.3 ms) and zeroed when a
 * batch of the buffer first needs it, so that a buffer takes no more memory than
 * its batches use.  NULL (and another launch) if there is no room, or a caller
 * captures the stream. */
static uint32_t *split_pool(myers_buffer_t *b)
{
    if (b == NULL || b->d_split) return b ? b->d_split : NULL;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(b->stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return NULL;
    /* (relaxed: the allocation does not end another thread's capture) */
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return NULL;
    void *pool = NULL;
    const hipError_t e = hipMalloc(&pool, MYERS_SPLIT_WORDS * sizeof(uint32_t));
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return NULL;
    }
    if (hip_fail(hipMemsetAsync(pool, 0, MYERS_SPLIT_WORDS * sizeof(uint32_t), b->stream), "hipMemsetAsync", __FILE__,
                 __LINE__)) {
        hipFree(pool);
        return NULL;
    }
    return b->d_split = (uint32_t *)pool;
}

/* The bins of a batch that run split over waves.  Returns the words per lane
 * (0: none).
 *
 * Multi-lane bins, all of them or none: where the estimate is below that of the
 * bit-vector launches (2-20 kb, 4 candidates each: 25-100 reads 1.6 ms against
 * 3.0, 200 reads 2.0 against 3.5, 400 reads 2.9 against 5.6, 800 reads 5.0
 * against 6.3, 1,600 reads would be 9.1 against 8.4; one read of 20,000 bases 1.6
 * against 6.4; 1,100-4,000 bases:
 * 250 reads 0.37 against 1.04, 1,000 reads 0.73 against 1.07, 2,000 reads would
 * be 1.2 against 1.1).  One-lane bins, whose chunks of the sliced kernel take
 * about 16.6 ns per word and step: beside multi-lane bins those of 8 words or
 * more, most words first, while a chunk would take longer than the launch with
 * them; without multi-lane bins all or none, which keeps the batch one launch
 * (100-1000 bases, 11 candidates per read: 100 reads 129 us against 700), and
 * where that is one bin of one part per candidate without binning (8 candidates
 * per read: 100 reads of 100 bases 31 us against 34 with the bit-vector kernel,
 * 200 reads would be 35.5 against 34.5; 100 reads of 250 bases 41 against 88, of
 * 1000 bases 87 against 680, 1,000 reads of 1000 bases 415 against 680).
 * The split launch spends more of the chip per cell than the launches it stands
 * in for (60-98e12 cells per second against 110-130e12), so a batch beside others
 * weighs the work with its share of the chip. */
static uint32_t split_plan(const myers_ctx_t *ctx, const bin_scan_t *scan, const batch_t *bt, const uint32_t *order,
                           uint32_t n, myers_split_plan_t *sp, uint32_t *grid)
{
    const uint32_t engine = bt->flags & MYERS_ENGINE_MASK;
    sp->n = 0;
    *grid = 0;
    if ((scan->num_present > 1 && !(scan->present & (ctx->multi_lane | ctx->deep))) || !scan->sized || scan->too_long || bt->num_queries == 0 ||
        (bt->flags & MYERS_NO_LONG_LAUNCH) ||
        (engine != MYERS_ENGINE_AUTO && engine != MYERS_ENGINE_PERSISTENT))
        return 0;
    const double cpr = (double)bt->num_cands / (double)bt->num_queries;
    const double simds = 4.0 * (double)ctx->num_cus * bt->share, rate = 120e3 * bt->share;
    /* the binning, which a batch of one bin does without, also here if it is one
     * part per candidate */
    const int one = engine == MYERS_ENGINE_AUTO && scan->num_present == 1;
    double extra = 0.0;
    split_est_t est = {{0.0}, {0.0}, {0.0}};
    double cells = 0.0, old_chain = 0.0, old = 0.0, now = 0.0;
    uint32_t longest = 0, best = 0, i = 0;
    for (; i < n && ctx->variants[order[i]].lanes > 1u && sp->n < (uint32_t)MYERS_QUEUE_MAX; i++) {
        const uint32_t v = order[i];
        const myers_variant_desc_t *d = &ctx->variants[v];
        if (d->lanes > 64u) return 0;
        const double cands = scan->counted ? (double)scan->cands[v] : (double)scan->reads[v] * cpr;
        const double m = (double)scan->max_m[v], c = chain_ns(scan->max_m[v], d->lanes, d->words, 0);
        sp->variant[sp->n++] = v;
        if (d->total_words > longest) longest = d->total_words;
        if (cands <= 0.0) continue;
        split_est_add(&est, d->total_words, m, cands);
        cells += 0.8 * cands * 1.25 * m * m;
        if (c > old_chain) old_chain = c;
    }
    if (sp->n) {
        myers_long_plan_t lp;
        /* (a quarter of a chain: what the tail of the long-read launch took over its estimate) */
        if (scan->num_present > 1 && long_plan(ctx, scan, bt, order, n, &lp, &old)) old += 0.25 * old_chain;
        else old = cells / rate > old_chain ? cells / rate : old_chain;
        now = split_est_ns(&est, simds, &best);
        if (one && ctx->variants[sp->variant[0]].total_words > 64u * split_kinds[best].words) extra = 50e3;
        if (now + extra >= old) return 0;
    }
    const uint32_t nlong = sp->n;
    double slowest = 0.0;                   /* of the one-lane launch, without multi-lane bins */
    for (; i < n && sp->n < (uint32_t)MYERS_QUEUE_MAX; i++) {
        const uint32_t v = order[i];
        const myers_variant_desc_t *d = &ctx->variants[v];
        if (d->lanes > 1u || (nlong && d->words < 8u)) break;
        const double cands = scan->counted ? (double)scan->cands[v] : (double)scan->reads[v] * cpr;
        const double m = (double)scan->max_m[v];
        double chunk = d->words < 8u ? 1.25 * m * (40.0 + 20.0 * (double)d->words)
                                     : (1.25 * m + 31.0) * (20.0 + 16.6 * (double)d->words);
        if (cands * 1.25 * m * m / (220e3 * bt->share) > chunk) chunk = cands * 1.25 * m * m / (220e3 * bt->share);
        if (chunk > slowest) slowest = chunk;
        split_est_t with = est;
        uint32_t kind = 0;
        split_est_add(&with, d->total_words, m, cands);
        const double then = split_est_ns(&with, simds, &kind);
        if (nlong && then >= (now > chunk ? now : chunk)) break;
        est = with;
        now = then;
        best = kind;
        sp->variant[sp->n++] = v;
        if (d->total_words > longest) longest = d->total_words;
    }
    if (!nlong && (i < n || now + extra + 2e3 >= slowest)) return 0;
    /* slots for the longest window that a bin's reads can have */
    const double cols = 32.0 * (double)longest * (1.0 + 2.0 * (double)bt->distance) + 64.0;
    if (sp->n == 0 || !(cols >= 64.0) || cols > 1e6) return 0;
    const uint32_t words = split_kinds[best].words;
    uint32_t *pool = NULL;
    for (uint32_t j = 0; j < sp->n; j++) {
        sp->parts[j] = (ctx->variants[sp->variant[j]].total_words + 64u * words - 1u) / (64u * words);
        if (sp->parts[j] > 1u && pool == NULL && (pool = split_pool(bt->pool_of)) == NULL) return 0;
    }
    sp->stride = ((uint32_t)cols + 128u) / 64u * 2u + 4u;
    sp->nslots = (uint32_t)MYERS_SPLIT_POOL_WORDS / 2u / sp->stride;
    if (sp->nslots > (uint32_t)MYERS_SPLIT_MAX_SLOTS) sp->nslots = MYERS_SPLIT_MAX_SLOTS;
    if (sp->nslots < (uint32_t)MYERS_SPLIT_MIN_SLOTS) return 0;
    sp->pool = (uint64_t *)pool;
    sp->done = pool ? pool + MYERS_SPLIT_POOL_WORDS : NULL;
    *grid = (uint32_t)ctx->num_cus * split_kinds[best].per_simd;
    return words;
}

/* The cut-off kernel for a bin of reads of up to `words` words with about `cands`
 * candidates in threshold mode (its variant), or -1: the sliced kernel.
 *
 * Low thresholds leave the cut-off a few rows per column: 8 candidates per read of
 * 1000 bases, threshold 0.05 m, 20K candidates 0.73 ms against 0.81 with the sliced
 * kernel, 100K 0.95 against 1.04; 0.1 m 0.77 and 0.81, 0.98 and 1.02; 0.2 m 0.83 and
 * 0.81.  Shorter reads' sliced chunks take less time than the cut-off's unless
 * waves share the SIMDs (800 bases, 0.05 m: 50K 0.49 and 0.47, 100K 0.63 and 0.69;
 * 600 bases 0.31 and 0.30, 0.40 and 0.42); at 400 bases it gains nothing. */
static int cut_variant(const myers_ctx_t *ctx, uint32_t words, float threshold, double cands)
{
    if (threshold < 0.0f || threshold > 0.1f || words < 17u ||
        (words <= 28u && cands < 288.0 * (double)ctx->num_cus))
        return -1;
    for (uint32_t v = 0; v < ctx->num_variants; v++)
        if (ctx->variants[v].lanes == 1u && ctx->variants[v].words >= words && myers_variant_cut_ok(v)) return (int)v;
    return -1;
}

/* Launch one bin: variant v over a->start / count or its bin range, with a
 * fixed grid (resident = 0) or a resident grid that pulls from the variant's
 * part heads. */
static int launch_bin(myers_buffer_t *b, uint32_t v, myers_verify_args_t *a, const slice_load_t *load, double cands_in_bin,
                      int resident, hipStream_t stream)
{
    myers_ctx_t *ctx = b->ctx;
    b->ran.ran |= MYERS_RAN_BIN;
    const myers_variant_desc_t *d = &ctx->variants[v];
    const uint32_t num_cands = load->num_cands;
    a->variant = v;
    a->chunk_factor = ctx->chunk_factor[v];
    if (d->lanes == 1u) {
        const int cut = resident ? -1 : cut_variant(ctx, d->words, a->threshold, cands_in_bin);
        if (cut >= 0) b->ran.ran |= MYERS_RAN_CUT;
        if (cut >= 0)
            return myers_launch_verify((uint32_t)cut, a, grid_for(ctx, v, num_cands, a->bin_ranges != NULL), 0, stream);
        myers_queue_plan_t p;
        memset(&p, 0, sizeof(p));
        const uint32_t lanes = slice_lanes(ctx, d->words, load), cands = lanes == 16u ? 128u : 64u;
        if (lanes == 1u && !resident)
            return myers_launch_verify(v, a, grid_for(ctx, v, num_cands, a->bin_ranges != NULL), 0, stream);
        slice_plan_add(ctx, &p, v, lanes);
        const uint32_t chunks = (num_cands + cands - 1u) / cands;
        const uint32_t full = queue_grid(ctx, lanes == 16u ? 2u : 3u, p.ws_u4 * 16u);
        uint32_t grid = chunks;
        if (a->bin_ranges && grid > full) grid = full;      /* the bin may hold any part of them */
        return myers_launch_slice(a, &p, resident ? MYERS_SLICE_RANGES : MYERS_SLICE_PLAIN, grid, stream);
    }
    if (resident)
        return myers_launch_verify(v, a, (uint32_t)ctx->num_cus * (uint32_t)ctx->occupancy_p[v], 1, stream);
    return myers_launch_verify(v, a, grid_for(ctx, v, num_cands, a->bin_ranges != NULL), 0, stream);
}

/* Queue launches of a persistent batch: the bins (already in longest-first
 * order) of each kernel class go into one plan, in that order; bins of no
 * class (multi-lane W = 16, multi-wave variants) are left in `other`. */
static void queue_plans(const myers_ctx_t *ctx, const uint32_t *bins, uint32_t n, const slice_load_t *load,
                        uint64_t wide, myers_queue_plan_t *qp, uint32_t *other, uint32_t *nother)
{
    memset(qp, 0, sizeof(myers_queue_plan_t) * MYERS_QUEUE_CLASSES);
    *nother = 0;
    for (uint32_t c = 0; c < (uint32_t)MYERS_QUEUE_CLASSES; c++) qp[c].cls = c;
    for (uint32_t i = 0; i < n; i++) {
        uint32_t u4 = 0;
        int cls = myers_variant_queue_class(bins[i], &u4);
        uint32_t lanes = 0;
        if (cls == MYERS_QUEUE_ONE_LANE) {
            lanes = slice_lanes(ctx, ctx->variants[bins[i]].words, load);
            if (lanes == 16u) cls = MYERS_QUEUE_ONE_LANE_16;
        }
        if ((wide >> bins[i]) & 1ull) cls = MYERS_QUEUE_WIDE;
        if (cls < 0 || qp[cls].n >= (uint32_t)MYERS_QUEUE_MAX) {
            other[(*nother)++] = bins[i];
            continue;
        }
        myers_queue_plan_t *q = &qp[cls];
        if (lanes) {
            slice_plan_add(ctx, q, bins[i], lanes);
            continue;
        }
        q->variant[q->n] = bins[i];
        q->key[q->n] = cls == MYERS_QUEUE_WIDE ? myers_wide_slice_team(ctx->variants[bins[i]].total_words)
                                               : (ctx->variants[bins[i]].lanes << 8) | ctx->variants[bins[i]].words;
        q->n++;
        if (u4 > q->ws_u4) q->ws_u4 = u4;
    }
}

/* The variants of a plan, as a mask. */
static uint64_t plan_bins(const myers_queue_plan_t *p)
{
    uint64_t bins = 0;
    for (uint32_t i = 0; i < p->n; i++) bins |= 1ull << p->variant[i];
    return bins;
}

/* Device-side binning of a batch. */
static int enqueue_binning(myers_buffer_t *b, const batch_t *bt)
{
    myers_ctx_t *ctx = b->ctx;
    const int rc = myers_launch_binning((const uint32_t *)bt->d_qinfo, bt->num_queries, bt->d_cands, bt->num_cands,
                                        ctx->d_bin_of_words + (fine_bins(bt->flags) ? BIN_ROWS : 0u),
                                        max_supported_words(ctx), ctx->num_variants,
                                        bt->d_work + MYERS_WORK_BLOCKS, bt->d_work + MYERS_WORK_RANGES, bt->d_order,
                                        b->d_err, bt->d_results, bt->d_work + MYERS_WORK_HEADS, b->stream);
    return rc ? hip_fail((hipError_t)rc, "binning launch", __FILE__, __LINE__) : MYERS_SUCCESS;
}

/* Enqueue the on-device pipeline of one batch on b->stream (no timing events, so
 * that it can be captured into a graph); binned: its binning is enqueued. */
static int enqueue_pipeline(myers_buffer_t *b, const batch_t *bt, const bin_scan_t *scan, int binned)
{
    myers_ctx_t *ctx = b->ctx;
    myers_verify_args_t a;
    memset(&a, 0, sizeof(a));
    a.ref = ctx->d_ref;
    a.ref_words = ctx->ref_words_alloc;
    a.ref_size = ctx->ref_size;
    a.planes = ctx->d_planes;
    a.plane_blocks = ctx->plane_blocks;
    a.peq = (const uint32_t *)bt->d_peq;
    a.qinfo = (const uint32_t *)bt->d_qinfo;
    a.num_peq_entries = bt->num_entries;
    a.num_queries = bt->num_queries;
    a.cands = bt->d_cands;
    a.mode = bt->flags & 1u;
    a.distance = bt->distance;
    a.threshold = bt->threshold;
    a.results = bt->d_results;

    const uint64_t wide = wide_bins(ctx, scan, bt);
    uint32_t order[MYERS_MAX_VARIANTS];
    const uint32_t n = present_by_cost(ctx, scan->present, order);
    myers_split_plan_t sp;
    uint32_t split_grid = 0;
    const uint32_t split = wide ? 0u : split_plan(ctx, scan, bt, order, n, &sp, &split_grid);
    const int first_rows = first_rows_pay(ctx, scan, bt);
    const uint32_t engine =
        wide || split ? (uint32_t)MYERS_ENGINE_PERSISTENT : resolve_engine(ctx, scan, bt, first_rows);
    b->stats.launches = 0;
    b->stats.variantsUsed = 0;
    b->binned = 0;
    memset(&b->ran, 0, sizeof(b->ran));
    int rc;
    if (bt->num_cands == 0) return MYERS_SUCCESS;
    const int one_bin = engine == MYERS_ENGINE_PLAIN && scan->num_present == 1 && !scan->too_long;
    const slice_load_t load = slice_load(ctx, scan, bt->num_queries, bt->num_cands, !one_bin);
    const int one_part = split && scan->num_present == 1 && sp.parts[0] == 1u && !binned &&
                         (bt->flags & MYERS_ENGINE_MASK) == MYERS_ENGINE_AUTO;
    if (one_bin || one_part) {
        const uint32_t v = scan->single;
        a.start = 0;
        a.count = bt->num_cands;
        const uint32_t waves = (bt->num_cands + 3u) / 4u;
        rc = one_part ? myers_launch_split(&a, &sp, split, split_grid < waves ? split_grid : waves, b->stream)
                      : launch_bin(b, v, &a, &load, (double)bt->num_cands, 0, b->stream);
        if (rc) return hip_fail((hipError_t)rc, "verify launch", __FILE__, __LINE__);
        if (one_part) b->ran.ran |= MYERS_RAN_SPLIT;
        b->ran.split_words = one_part ? split : 0u;
        b->stats.launches = 1;
        b->stats.variantsUsed = 1;
        return MYERS_SUCCESS;
    }
    /* Chunks of the sliced kernels with an N in some read run slower; in a
     * large batch the candidates of such reads are put together.  The two
     * passes take about 12 us per million candidates, which pays where the
     * chunks are long: bins of over GROUP_N_WORDS words, in batches whose
     * one-lane reads average that (1000 bases: 7.08 -> 6.7 ms; 100 bases, if it
     * were done: 1.02 -> 1.10 ms). */
    uint64_t group_n = 0;
    if ((uint64_t)bt->num_cands >= 1024u * (uint64_t)ctx->num_cus &&
        load.per_wave * 64.0 * 12.0 * (double)ctx->num_cus >= (double)(GROUP_N_WORDS * GROUP_N_WORDS) * (double)bt->num_cands) {
        for (uint32_t v = 0; v < ctx->num_variants; v++)
            if (ctx->variants[v].lanes == 1u && ctx->variants[v].words > GROUP_N_WORDS) group_n |= scan->present & (1ull << v);
    }
    if (!binned && (rc = enqueue_binning(b, bt))) return rc;
    uint32_t *ranges = bt->d_work + MYERS_WORK_RANGES;
    uint32_t *heads = bt->d_work + MYERS_WORK_HEADS;
    if (group_n || wide) {
        /* (up to the longest read that a bin holds: a size near 2^32 counts as one of
         * no words in the binning, and its Peq is not there) */
        rc = myers_launch_read_n(&a, bt->num_cands, group_n ? 32u * GROUP_N_WORDS : 32u * myers_slice_max_words(32u),
                                 32u * (wide ? max_supported_words(ctx) : myers_slice_max_words(32u)), b->stream);
        if (rc) return hip_fail((hipError_t)rc, "read N launch", __FILE__, __LINE__);
    }
    if (group_n) {
        rc = myers_launch_group_n(ranges, ctx->num_variants, group_n, bt->num_cands, bt->d_order, bt->d_results,
                                  b->stream);
        if (rc) return hip_fail((hipError_t)rc, "group N launch", __FILE__, __LINE__);
    }
    if (wide) {
        rc = myers_launch_sort_len(&a, ranges, ctx->num_variants, wide, bt->num_cands, bt->d_order, b->stream);
        if (rc) return hip_fail((hipError_t)rc, "sort launch", __FILE__, __LINE__);
    }
    if (b->mark_slot >= 0) {
        /* eager batches: the verification launches are timed apart from the binning */
        HIP_TRY(hipEventRecord(b->ev_kernel[b->mark_slot][2], b->stream));
        b->ev_marked[b->mark_slot] = 1;
    }
    b->binned = 1;
    a.order = bt->d_order;
    a.bin_ranges = ranges;
    a.queue_heads = heads;
    uint32_t launches = n;
    if (engine == MYERS_ENGINE_PLAIN) {
        /* one launch per length bin, in turn */
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t v = order[i];
            const double cands = !scan->sized || bt->num_queries == 0 ? 0.0 :
                                 scan->counted ? (double)scan->cands[v] :
                                 (double)scan->reads[v] * (double)bt->num_cands / (double)bt->num_queries;
            rc = launch_bin(b, v, &a, &load, cands, 0, b->stream);
            if (rc) return hip_fail((hipError_t)rc, "verify launch", __FILE__, __LINE__);
        }
    } else {
        /* Persistent engines.  The long-read bins of a latency-bound batch
         * share one launch (long_plan).  MYERS_ENGINE_PERSISTENT puts the
         * other bins into one queue launch per kernel class (one launch for
         * a batch of one class); MYERS_ENGINE_BINNED gives every bin its own
         * resident grid.  Bins without a queue class keep their own grid.
         * When more than one launch results, they run on forked streams
         * (long-read launch first), so that each one's tail overlaps the
         * others. */
        myers_long_plan_t lp;
        uint32_t nlong = 0;
        if (wide || split || (bt->flags & MYERS_NO_LONG_LAUNCH)) memset(&lp, 0, sizeof(lp));
        else nlong = long_plan(ctx, scan, bt, order, n, &lp, NULL);
        uint32_t rest[MYERS_MAX_VARIANTS], nrest = 0;
        for (uint32_t i = 0; i < n; i++) {
            int in_long = 0;
            for (uint32_t j = 0; j < lp.n; j++) in_long |= lp.variant[j] == order[i];
            for (uint32_t j = 0; j < lp.n_wide; j++) in_long |= lp.wide_variant[j] == order[i];
            for (uint32_t j = 0; split && j < sp.n; j++) in_long |= sp.variant[j] == order[i];
            if (!in_long) rest[nrest++] = order[i];
        }
        myers_queue_plan_t qp[MYERS_QUEUE_CLASSES];
        uint32_t other[MYERS_MAX_VARIANTS], nother = 0, nqueue = 0;
        if (engine == MYERS_ENGINE_PERSISTENT) {
            queue_plans(ctx, rest, nrest, &load, wide, qp, other, &nother);
            for (uint32_t c = 0; c < (uint32_t)MYERS_QUEUE_CLASSES; c++) nqueue += qp[c].n ? 1u : 0u;
        } else {
            memset(qp, 0, sizeof(qp));
            memcpy(other, rest, nrest * sizeof(uint32_t));
            nother = nrest;
        }
        launches = (nlong ? 1u : 0u) + (split ? 1u : 0u) + nqueue + nother;
        const int fork = launches > 1u;
        const uint32_t width = !fork ? 0u : (launches < SIDE_STREAMS ? launches : SIDE_STREAMS);
        uint32_t next = 0;    /* launches placed so far: launch k goes on side stream k % width */
#define NEXT_STREAM() (fork ? b->side[(next++) % width] : b->stream)
        if (fork) {
            HIP_TRY(hipEventRecord(b->ev_fork, b->stream));
            for (uint32_t j = 0; j < width; j++) HIP_TRY(hipStreamWaitEvent(b->side[j], b->ev_fork, 0));
        }
        if (split) {
            rc = myers_launch_split(&a, &sp, split, split_grid, NEXT_STREAM());
            if (rc) return hip_fail((hipError_t)rc, "split launch", __FILE__, __LINE__);
            b->ran.ran |= MYERS_RAN_SPLIT;
            for (uint32_t j = 0; j < sp.n; j++)
                if (sp.parts[j] > 1u) b->ran.ran |= MYERS_RAN_HANDOVERS;
            b->ran.split_words = split;
            b->ran.split_slots = sp.nslots;
        }
        if (nlong) {
            /* successive launches start their first items a golden-ratio step
             * of workgroups apart (overlapping batches use other CUs) */
            const uint32_t seq = __atomic_fetch_add(&ctx->long_seq, 1u, __ATOMIC_RELAXED);
            const uint32_t wg = (uint32_t)(((uint64_t)seq * 2654435769ull & 0xFFFFFFFFull) * ctx->num_cus >> 32);
            lp.rotate = wg * MYERS_LONG_WAVES;
            rc = myers_launch_long(&a, &lp, ctx->num_cus, NEXT_STREAM());
            if (rc) return hip_fail((hipError_t)rc, "long-read launch", __FILE__, __LINE__);
            b->ran.ran |= MYERS_RAN_LONG;
        }
        /* (longest reads first) */
        for (uint32_t k = 0; k < (uint32_t)MYERS_QUEUE_CLASSES; k++) {
            const uint32_t c = (k + (uint32_t)MYERS_QUEUE_WIDE) % (uint32_t)MYERS_QUEUE_CLASSES;
            if (qp[c].n == 0) continue;
            if (c == MYERS_QUEUE_WIDE) {
                rc = myers_launch_wide_slice(&a, &qp[c], ctx->num_cus, NEXT_STREAM());
                if (rc) return hip_fail((hipError_t)rc, "queue launch", __FILE__, __LINE__);
                b->ran.ran |= MYERS_RAN_WIDE_SLICE;
                continue;
            }
            const int multi = c == MYERS_QUEUE_MULTI_LANE;
            b->ran.ran |= multi ? MYERS_RAN_QUEUE : MYERS_RAN_SLICE;
            const uint32_t which = !multi ? (c == MYERS_QUEUE_ONE_LANE_16 ? 2u : 3u) : (bt->threshold >= 0.0f ? 1u : 0u);
            const uint32_t grid = queue_grid(ctx, which, qp[c].ws_u4 * 16u);
            hipStream_t stream = NEXT_STREAM();
            if (multi) {
                rc = myers_launch_queue(&a, &qp[c], grid, stream);
            } else {
                myers_verify_args_t two = a;
                const int filter = first_rows && c == (uint32_t)MYERS_QUEUE_ONE_LANE;
                if (filter) {
                    two.list = bt->d_list;
                    two.list_ranges = bt->d_work + MYERS_WORK_LIST;
                    two.tally = bt->d_work + MYERS_WORK_TALLY;
                }
                rc = myers_launch_slice(&two, &qp[c], MYERS_SLICE_QUEUE, grid, stream);
                if (!rc && filter && group_n)
                    rc = myers_launch_group_n(two.list_ranges, ctx->num_variants, group_n & plan_bins(&qp[c]),
                                              bt->num_cands, two.list, bt->d_results, stream);
                if (!rc && filter) {
                    two.order = two.list;
                    two.bin_ranges = two.list_ranges;
                    two.queue_heads = heads + 1;
                    two.list = NULL;
                    myers_queue_plan_t rest = qp[c];
                    rest.cls = MYERS_QUEUE_WIDE;
                    for (uint32_t j = 0; j < rest.n; j++)
                        rest.key[j] = myers_wide_slice_team(ctx->variants[rest.variant[j]].total_words);
                    rc = myers_launch_wide_slice(&two, &rest, ctx->num_cus, stream);
                    b->ran.ran |= MYERS_RAN_FIRST_ROWS;
                    launches++;
                }
            }
            if (rc) return hip_fail((hipError_t)rc, "queue launch", __FILE__, __LINE__);
        }
        for (uint32_t i = 0; i < nother; i++) {
            rc = launch_bin(b, other[i], &a, &load, 0.0, 1, NEXT_STREAM());
            if (rc) return hip_fail((hipError_t)rc, "persistent launch", __FILE__, __LINE__);
        }
#undef NEXT_STREAM
        for (uint32_t j = 0; j < width; j++) {
            HIP_TRY(hipEventRecord(b->ev_join[j], b->side[j]));
            HIP_TRY(hipStreamWaitEvent(b->stream, b->ev_join[j], 0));
        }
    }
    b->stats.launches = launches;
    b->stats.variantsUsed = n;
    return MYERS_SUCCESS;
}

/* Candidates per variant, for batches with long-read bins (the long-read
 * plan sizes its rounds with them; reads carry very different candidate
 * counts across lengths).  Short-read batches skip this pass. */
static void scan_cands(const myers_ctx_t *ctx, const uint8_t *bins, const qryInfo_t *qinfo, uint32_t nq, const candInfo_t *cands,
                       uint32_t nc, bin_scan_t *s)
{
    uint64_t long_mask = 0;
    for (uint32_t v = 0; v < ctx->num_variants; v++)
        if (myers_variant_long_ok(v, NULL)) long_mask |= 1ull << v;
    if (!(s->present & long_mask)) return;
    const uint32_t maxw = max_supported_words(ctx);
    for (uint32_t i = 0; i < nc; i++) {
        const uint32_t q = cands[i].query;
        if (q >= nq) continue;
        const uint32_t w = (qinfo[q].size + 31u) >> 5;
        if (w <= maxw) s->cands[bins[w]]++;
    }
    s->counted = 1;
}

static void make_scan(myers_ctx_t *ctx, const batch_t *bt, const qryInfo_t *h_qinfo, const candInfo_t *h_cands,
                      bin_scan_t *scan)
{
    const uint8_t *bins = bins_of(ctx, bt->flags);
    if (h_qinfo) {
        scan_qinfo(ctx, bins, h_qinfo, bt->num_queries, scan);
        if (h_cands) scan_cands(ctx, bins, h_qinfo, bt->num_queries, h_cands, bt->num_cands, scan);
    } else {
        memset(scan, 0, sizeof(*scan));
        scan->present = ctx->num_variants >= 64 ? ~0ull : ((1ull << ctx->num_variants) - 1u);
        scan->num_present = ctx->num_variants;
        scan->too_long = 1;   /* unknown: let the device check */
    }
}

/* Enqueue the verification of a batch on b->stream, timed with HIP events;
 * with MYERS_USE_GRAPH the pipeline is captured once per batch shape and
 * replayed as a graph. */
static int enqueue_verify(myers_buffer_t *b, const batch_t *bt, const qryInfo_t *h_qinfo, const candInfo_t *h_cands)
{
    bin_scan_t scan;
    uint32_t slot = 0;
    int rc;
    if (!(bt->flags & MYERS_USE_GRAPH) || bt->num_cands == 0) {
        if ((rc = timing_begin(b, &slot))) return rc;
        /* A large batch is binned whatever its reads are (resolve_engine), so
         * that starts before the host looks at them (with scan_qinfo's counts,
         * 150K reads of 36-400 bases: 716 -> 678 us). */
        const int early = (bt->flags & MYERS_ENGINE_MASK) == MYERS_ENGINE_AUTO && large_batch(b->ctx, bt->num_cands);
        if (early && (rc = enqueue_binning(b, bt))) return rc;
        make_scan(b->ctx, bt, h_qinfo, h_cands, &scan);
        b->mark_slot = (int)slot;
        rc = enqueue_pipeline(b, bt, &scan, early);
        b->mark_slot = -1;
        if (rc) return rc;
        return timing_end(b, slot, b->stats.launches);
    }
    make_scan(b->ctx, bt, h_qinfo, h_cands, &scan);
    uint32_t dist_bits, thr_bits;
    memcpy(&dist_bits, &bt->distance, sizeof(dist_bits));
    memcpy(&thr_bits, &bt->threshold, sizeof(thr_bits));
    uint32_t order[MYERS_MAX_VARIANTS];
    myers_long_plan_t lp;
    myers_split_plan_t sp;
    uint32_t split_grid = 0;
    const uint32_t split =
        split_plan(b->ctx, &scan, bt, order, present_by_cost(b->ctx, scan.present, order), &sp, &split_grid);
    const uint64_t plan_key = (bt->flags & MYERS_NO_LONG_LAUNCH) ? 0u :
                              ((uint64_t)long_plan(b->ctx, &scan, bt, order,
                                                   present_by_cost(b->ctx, scan.present, order), &lp, NULL) |
                               ((uint64_t)lp.n_wide << 32));
    const uint64_t key[14] = {(uint64_t)(uintptr_t)bt->d_peq, (uint64_t)(uintptr_t)bt->d_qinfo,
                              (uint64_t)(uintptr_t)bt->d_cands, (uint64_t)(uintptr_t)bt->d_results,
                              ((uint64_t)bt->num_entries << 32) | bt->num_queries,
                              ((uint64_t)bt->num_cands << 32) | bt->flags,
                              (uint64_t)dist_bits, scan.present,
                              (uint64_t)scan.too_long, b->ctx->tune_gen, (uint64_t)thr_bits, plan_key,
                              wide_bins(b->ctx, &scan, bt), (uint64_t)split | ((uint64_t)sp.n << 8) |
                                  ((uint64_t)first_rows_pay(b->ctx, &scan, bt) << 31) | ((uint64_t)split_grid << 32)};
    if (!b->graph_valid || memcmp(key, b->graph_key, sizeof(key)) != 0) {
        if (b->graph_exec) {
            hipGraphExecDestroy(b->graph_exec);
            b->graph_exec = NULL;
        }
        b->graph_valid = 0;
        hipGraph_t graph = NULL;
        HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        rc = enqueue_pipeline(b, bt, &scan, 0);
        hipError_t e = hipStreamEndCapture(b->stream, &graph);
        if (rc) {
            if (graph) hipGraphDestroy(graph);
            return rc;
        }
        HIP_TRY(e);
        e = hipGraphInstantiate(&b->graph_exec, graph, NULL, NULL, 0);
        hipGraphDestroy(graph);
        HIP_TRY(e);
        memcpy(b->graph_key, key, sizeof(key));
        b->graph_valid = 1;
        b->graph_binned = b->binned;
        b->graph_launches = b->stats.launches;
        b->graph_ran = b->ran;
        b->stats.graphCaptures++;
    }
    if ((rc = timing_begin(b, &slot))) return rc;
    HIP_TRY(hipGraphLaunch(b->graph_exec, b->stream));
    b->binned = b->graph_binned;
    b->ran = b->graph_ran;
    b->stats.launches = b->graph_launches;
    b->stats.variantsUsed = b->graph_launches;
    return timing_end(b, slot, b->graph_launches);
}

static uint64_t nominal_cells(const qryInfo_t *qinfo, const candInfo_t *cands, uint32_t nc, float d)
{
    uint64_t cells = 0;
    for (uint32_t i = 0; i < nc; i++) {
        uint32_t m = qinfo[cands[i].query].size;
        volatile float f = (float)m * (1.0f + 2.0f * d);
        cells += (uint64_t)m * (uint64_t)(uint32_t)f;
    }
    return cells;
}

/* The share of the chip that a batch of this buffer can expect beside the library's
 * other buffers with a batch in flight.  One other is mostly near its end when the
 * batch starts; two count for half of it (three buffers served at 16.5e6 candidates
 * per second of the serving mix: p50 11.5 ms and p99 27 ms as if alone, 10.1 and 21.5;
 * at 8e6 4.2 ms either way, 5.3 if every other counted for one).  A captured pipeline
 * runs beside whatever its replays meet, and keeps one plan. */
static double chip_share(const myers_buffer_t *b, uint32_t flags)
{
    if (flags & MYERS_USE_GRAPH) return 1.0;
    const uint32_t others = __atomic_load_n(&b->ctx->in_flight, __ATOMIC_RELAXED) - (b->pending ? 1u : 0u);
    return others > 1u ? 2.0 / (1.0 + (double)others) : 1.0;
}

static void set_pending(myers_buffer_t *b, int pending)
{
    if (pending && !b->pending) __atomic_fetch_add(&b->ctx->in_flight, 1u, __ATOMIC_RELAXED);
    if (!pending && b->pending) __atomic_fetch_sub(&b->ctx->in_flight, 1u, __ATOMIC_RELAXED);
    b->pending = pending;
}

/* The threshold as the kernels take it (< 0: off). */
static float kernel_threshold(const myers_buffer_t *b)
{
    return b->threshold < MYERS_MAX_THRESHOLD ? b->threshold : MYERS_MAX_THRESHOLD;
}

/* Whether a batch's one launch reads and writes the pinned host arrays itself:
 * one-lane reads of one bin in a batch that is not binned (every array is then
 * read about once, and the launch does not wait for three copies, nor the caller
 * for a fourth).  11 candidates per read of 150 bases: 1 read 70 -> 55 us, 256
 * reads 132 -> 86, 20,000 reads 1573 -> 1494; 1000 bases: 64 reads 142 -> 114 us,
 * 20,000 reads the same.  Binned batches read the candidates three times (64
 * reads of 100-1000 bases: 156 -> 162 us), long reads' parts the Peq (64 reads of
 * 2-20 kb: 1.64 -> 1.72 ms). */
static int reads_host_arrays(const myers_buffer_t *b, uint32_t flags, uint32_t num_queries, uint32_t num_cands)
{
    if ((flags & MYERS_ENGINE_MASK) != MYERS_ENGINE_AUTO || (flags & MYERS_USE_GRAPH) || num_queries == 0 ||
        num_cands == 0 || large_batch(b->ctx, num_cands))
        return 0;
    const uint32_t first = (b->h_qinfo[0].size + 31u) >> 5;
    if (first > 32u) return 0;
    /* (such a batch may be binned: first_rows_pay) */
    if (b->threshold >= 0.0f && (uint64_t)num_cands >= (uint64_t)FIRST_ROWS_MIN_CANDS * (uint64_t)b->ctx->num_cus &&
        myers_slice_first_rows(first, b->threshold) != 0u)
        return 0;
    const uint8_t *bin = bins_of(b->ctx, flags);
    for (uint32_t q = 1; q < num_queries; q++) {
        const uint32_t w = (b->h_qinfo[q].size + 31u) >> 5;
        if (w != first && (w > 32u || bin[w] != bin[first])) return 0;
    }
    return b->ctx->variants[bin[first]].lanes == 1u;
}

/* Room for the second launch's list (threshold mode) of a batch in the buffer's
 * arrays: what its candidates or Peq entries leave free, else NULL (every row of
 * every candidate then runs at once). */
static uint32_t *spare_list(const myers_buffer_t *b, uint32_t entries, uint32_t cands)
{
    const uint64_t need = (uint64_t)cands * sizeof(uint32_t);
    if ((uint64_t)(b->max_candidates - cands) * sizeof(candInfo_t) >= need) return (uint32_t *)(b->d_cands + cands);
    if ((uint64_t)(b->max_peq_entries - entries) * sizeof(qryEntry_t) >= need) return (uint32_t *)(b->d_peq + entries);
    return NULL;
}

int myersSendEx(void *myersBuffer, float distance, uint32_t numPEQEntries, uint32_t numQueries,
                uint32_t numCandidates, uint32_t flags)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL) return MYERS_E_INVALID_ARGUMENT;
    if (flags & ~(1u | MYERS_ENGINE_MASK | MYERS_USE_GRAPH | MYERS_NO_LONG_LAUNCH))
        return (b->last_error = MYERS_E_INVALID_ARGUMENT);
    if (numPEQEntries > b->max_peq_entries || numQueries > b->max_queries || numCandidates > b->max_candidates)
        return (b->last_error = MYERS_E_CAPACITY);
    int rc = hip_fail(hipSetDevice(b->ctx->device), "hipSetDevice", __FILE__, __LINE__);
    if (rc) return (b->last_error = rc);
    /* candidates must name a query of this batch */
    for (uint32_t i = 0; i < numCandidates; i++)
        if (b->h_cands[i].query >= numQueries) return (b->last_error = MYERS_E_INVALID_ARGUMENT);
    *b->h_err = 0;
    b->num_candidates = numCandidates;
    hipStream_t s = b->stream;
#define SEND_TRY(call) do { rc = hip_fail((call), #call, __FILE__, __LINE__); if (rc) return (b->last_error = rc); } while (0)
    SEND_TRY(hipEventRecord(b->ev_batch_start, s));
    const int direct = reads_host_arrays(b, flags, numQueries, numCandidates);
    if (numPEQEntries && !direct)
        SEND_TRY(hipMemcpyAsync(b->d_peq, b->h_peq, (size_t)numPEQEntries * sizeof(qryEntry_t), hipMemcpyHostToDevice, s));
    if (numQueries && !direct)
        SEND_TRY(hipMemcpyAsync(b->d_qinfo, b->h_qinfo, (size_t)numQueries * sizeof(qryInfo_t), hipMemcpyHostToDevice, s));
    if (numCandidates && !direct)
        SEND_TRY(hipMemcpyAsync(b->d_cands, b->h_cands, (size_t)numCandidates * sizeof(candInfo_t), hipMemcpyHostToDevice, s));
    const batch_t bt = {direct ? b->hd_peq : (void *)b->d_peq, direct ? b->hd_qinfo : (void *)b->d_qinfo,
                        direct ? b->hd_cands : (void *)b->d_cands, direct ? b->hd_results : (void *)b->d_results,
                        numPEQEntries, numQueries, numCandidates, flags, distance, kernel_threshold(b), b->d_work, b->d_order,
                        spare_list(b, numPEQEntries, numCandidates), b, chip_share(b, flags)};
    rc = enqueue_verify(b, &bt, b->h_qinfo, b->h_cands);
    if (rc) return (b->last_error = rc);
    if (numCandidates && !direct)
        SEND_TRY(hipMemcpyAsync(b->h_results, b->d_results, (size_t)numCandidates * sizeof(resEntry_t), hipMemcpyDeviceToHost, s));
    SEND_TRY(hipEventRecord(b->ev_batch_end, s));
#undef SEND_TRY
    b->stats.cells = nominal_cells(b->h_qinfo, b->h_cands, numCandidates, distance);
    b->stats.candidates = numCandidates;
    set_pending(b, 1);
    b->last_error = MYERS_SUCCESS;
    return MYERS_SUCCESS;
}

static int finish_batch(myers_buffer_t *b, int with_batch_events)
{
    int rc = hip_fail(hipStreamSynchronize(b->stream), "hipStreamSynchronize", __FILE__, __LINE__);
    if (rc) return rc;
    while (b->ev_pending) {
        rc = fold_oldest_timing(b);
        if (rc) return rc;
    }
    if (!b->pending) return MYERS_SUCCESS;
    set_pending(b, 0);
    float ms = 0.0f;
    if (with_batch_events && hipEventElapsedTime(&ms, b->ev_batch_start, b->ev_batch_end) == hipSuccess)
        b->stats.batchMs = ms;
    b->stats.binned = (uint32_t)b->binned;
    if (b->binned && (*b->h_err & 1u)) return MYERS_E_QUERY_TOO_LONG;
    if (b->binned && (*b->h_err & 2u)) return MYERS_E_INVALID_ARGUMENT;
    return MYERS_SUCCESS;
}

int myers_launch_info(void *myersBuffer, myers_launch_info_t *out)
{
    const myers_buffer_t *b = (const myers_buffer_t *)myersBuffer;
    if (b == NULL || out == NULL) return MYERS_E_INVALID_ARGUMENT;
    *out = b->ran;
    return MYERS_SUCCESS;
}

int myers_serve_plan(void *myersBuffer, myers_serve_plan_t *out)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || out == NULL) return MYERS_E_INVALID_ARGUMENT;
    const myers_ctx_t *ctx = b->ctx;
    memset(out, 0, sizeof(*out));
    out->device = ctx->device;
    out->num_cus = ctx->num_cus;
    out->d_ref = ctx->d_ref;
    out->ref_words = ctx->ref_words_alloc;
    out->ref_size = ctx->ref_size;
    out->threshold = kernel_threshold(b);
    uint32_t var_of[MYERS_SERVE_MAX_WORDS + 1];
    uint64_t used = 0;
    const uint32_t maxw = max_supported_words(ctx);
    for (uint32_t w = 0; w <= maxw && w <= MYERS_SERVE_MAX_WORDS; w++) {
        uint32_t v = ctx->bin_of_words[w];
        if (!myers_variant_serve_ok(v, NULL)) {
            uint32_t best = 0xFFFFFFFFu, best_cost = 0xFFFFFFFFu;
            for (uint32_t u = 0; u < ctx->num_variants; u++) {
                if (!myers_variant_serve_ok(u, NULL) || ctx->variants[u].total_words < (w ? w : 1u)) continue;
                const uint32_t c = variant_cost(&ctx->variants[u]);
                if (c < best_cost) { best_cost = c; best = u; }
            }
            if (best == 0xFFFFFFFFu) break;      /* longer reads: none can run there */
            v = best;
        }
        var_of[w] = v;
        used |= 1ull << v;
        out->max_words = w;
    }
    /* ranks: the used variants, most words per candidate first */
    uint32_t order[MYERS_MAX_VARIANTS];
    const uint32_t n = present_by_cost(ctx, used, order);
    uint32_t rank_of_var[MYERS_MAX_VARIANTS];
    for (uint32_t r = 0; r < n; r++) {
        const myers_variant_desc_t *d = &ctx->variants[order[r]];
        uint32_t u4 = 0;
        myers_variant_serve_ok(order[r], &u4);
        rank_of_var[order[r]] = r;
        out->rank_key[r] = (d->lanes << 8) | d->words;
        out->rank_slots[r] = d->slots;
        if (u4 * 16u > out->lds_bytes) out->lds_bytes = u4 * 16u;
    }
    out->num_ranks = n;
    for (uint32_t w = 0; w <= out->max_words; w++) out->rank_of_words[w] = (uint8_t)rank_of_var[var_of[w]];
    return MYERS_SUCCESS;
}

int myers_buffer_ready(void *myersBuffer)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    hipError_t e = hipStreamQuery(b->stream);
    if (e == hipSuccess) return 1;
    if (e == hipErrorNotReady) return 0;
    return -(int)e;
}

int myersReceiveEx(void *myersBuffer)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL) return MYERS_E_INVALID_ARGUMENT;
    int rc = hip_fail(hipSetDevice(b->ctx->device), "hipSetDevice", __FILE__, __LINE__);
    if (rc == MYERS_SUCCESS) rc = finish_batch(b, 1);
    b->last_error = rc;
    return rc;
}

void sendMyersBuffer(void *myersBuffer, float distance, uint32_t numPEQEntries, uint32_t numQueries,
                     uint32_t numCandidates)
{
    int rc = myersSendEx(myersBuffer, distance, numPEQEntries, numQueries, numCandidates, 0u);
    report((myers_buffer_t *)myersBuffer, rc, "sendMyersBuffer");
}

void receiveMyersBuffer(void *myersBuffer)
{
    int rc = myersReceiveEx(myersBuffer);
    report((myers_buffer_t *)myersBuffer, rc, "receiveMyersBuffer");
}

/* ------------------------------------------------------- device batches */

static int verify_device(myers_buffer_t *b, const void *d_peq, uint32_t numPEQEntries, const void *d_qinfo,
                         uint32_t numQueries, const void *d_candidates, uint32_t numCandidates,
                         float distance, uint32_t flags, void *d_results, const qryInfo_t *h_qinfo,
                         uint32_t *d_work, uint32_t *d_order, uint32_t *d_list, myers_buffer_t *pool_of)
{
    int rc = hip_fail(hipSetDevice(b->ctx->device), "hipSetDevice", __FILE__, __LINE__);
    if (rc) return (b->last_error = rc);
    *b->h_err = 0;
    const batch_t bt = {d_peq, d_qinfo, d_candidates, d_results, numPEQEntries, numQueries, numCandidates,
                        flags, distance, kernel_threshold(b), d_work, d_order, d_list, pool_of, chip_share(b, flags)};
    rc = enqueue_verify(b, &bt, h_qinfo, NULL);
    b->stats.cells = 0;
    b->stats.candidates = numCandidates;
    set_pending(b, rc == MYERS_SUCCESS);
    b->last_error = rc;
    return rc;
}

int myersVerifyDevice(void *myersBuffer, const void *d_peq, uint32_t numPEQEntries, const void *d_qinfo,
                      uint32_t numQueries, const void *d_candidates, uint32_t numCandidates,
                      float distance, uint32_t flags, void *d_results, const qryInfo_t *h_qinfo)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL) return MYERS_E_INVALID_ARGUMENT;
    if ((flags & ~(1u | MYERS_ENGINE_MASK | MYERS_USE_GRAPH | MYERS_NO_LONG_LAUNCH)) ||
        (numCandidates && (!d_peq || !d_qinfo || !d_candidates || !d_results)))
        return (b->last_error = MYERS_E_INVALID_ARGUMENT);
    if (numCandidates > b->max_candidates) return (b->last_error = MYERS_E_CAPACITY);
    /* (the buffer's own candidate array is free meanwhile: the second launch's list) */
    return verify_device(b, d_peq, numPEQEntries, d_qinfo, numQueries, d_candidates, numCandidates, distance,
                         flags, d_results, h_qinfo, b->d_work, b->d_order, (uint32_t *)b->d_cands, b);
}

/* myersVerifyDevice with the pipeline workspace in the device's static
 * array instead of the buffer's: nothing is allocated.  Every call on one
 * GPU shares that array, so calls that overlap on one GPU race; the binning
 * kernels re-initialise every part that must start at zero, so such calls
 * spoil no later one.  The split launch's pool does not start anew (and its
 * waves wait for each other), so no candidate runs in several parts here. */
int myersVerifyDeviceNoAlloc(void *myersBuffer, const void *d_peq, uint32_t numPEQEntries, const void *d_qinfo,
                             uint32_t numQueries, const void *d_candidates, uint32_t numCandidates,
                             float distance, uint32_t flags, void *d_results, const qryInfo_t *h_qinfo)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL) return MYERS_E_INVALID_ARGUMENT;
    /* graph instantiation may allocate: not on this path */
    if ((flags & ~(1u | MYERS_ENGINE_MASK | MYERS_NO_LONG_LAUNCH)) ||
        (numCandidates && (!d_peq || !d_qinfo || !d_candidates || !d_results)))
        return (b->last_error = MYERS_E_INVALID_ARGUMENT);
    if (numCandidates > MYERS_NOALLOC_MAX_CANDIDATES) {
        fprintf(stderr, "Myers - myersVerifyDeviceNoAlloc: %u candidates exceed the static workspace "
                "maximum of %u\n", numCandidates, (unsigned)MYERS_NOALLOC_MAX_CANDIDATES);
        return (b->last_error = MYERS_E_CAPACITY);
    }
    uint32_t *scratch = b->ctx->d_scratch;
    return verify_device(b, d_peq, numPEQEntries, d_qinfo, numQueries, d_candidates, numCandidates, distance,
                         flags, d_results, h_qinfo, scratch, scratch + MYERS_WORK_WORDS,
                         scratch + MYERS_WORK_WORDS + MYERS_NOALLOC_MAX_CANDIDATES, NULL);
}

int myersSetThreshold(void *myersBuffer, float errorRate)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || errorRate != errorRate) return MYERS_E_INVALID_ARGUMENT;
    b->threshold = errorRate < 0.0f ? -1.0f : errorRate;
    return MYERS_SUCCESS;
}

float myersGetThreshold(void *myersBuffer)
{
    const myers_buffer_t *b = (const myers_buffer_t *)myersBuffer;
    return b == NULL ? -1.0f : b->threshold;
}

int myersSynchronize(void *myersBuffer)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL) return MYERS_E_INVALID_ARGUMENT;
    int rc = hip_fail(hipSetDevice(b->ctx->device), "hipSetDevice", __FILE__, __LINE__);
    if (rc == MYERS_SUCCESS) rc = finish_batch(b, 0);
    b->last_error = rc;
    return rc;
}

int myersGetStats(void *myersBuffer, myersStats_t *out)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || out == NULL) return MYERS_E_INVALID_ARGUMENT;
    /* callers built against an older, shorter struct get its fields only */
    const size_t n = out->structSize && out->structSize < sizeof(*out) ? out->structSize : sizeof(*out);
    memcpy(out, &b->stats, n);
    out->structSize = (uint32_t)n;
    return MYERS_SUCCESS;
}

void myersResetStats(void *myersBuffer)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL) return;
    b->stats.kernelMsTotal = 0.0;
    b->stats.verifyMsTotal = 0.0;
    b->stats.kernelLaunchesTotal = 0;
    b->stats.batchesTotal = 0;
}

/* -------------------------------------------------------------- helpers */

int myersDeviceMalloc(void **ptr, size_t bytes)
{
    if (ptr == NULL) return MYERS_E_INVALID_ARGUMENT;
    return hip_fail(hipMalloc(ptr, bytes ? bytes : 1u), "hipMalloc", __FILE__, __LINE__);
}

int myersDeviceFree(void *ptr)
{
    return hip_fail(hipFree(ptr), "hipFree", __FILE__, __LINE__);
}

int myersMemcpyHtoD(void *dst, const void *src, size_t bytes)
{
    return hip_fail(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "hipMemcpy(HtoD)", __FILE__, __LINE__);
}

int myersMemcpyDtoH(void *dst, const void *src, size_t bytes)
{
    return hip_fail(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "hipMemcpy(DtoH)", __FILE__, __LINE__);
}

uint32_t myersNumVariants(void) { return myers_num_variants(); }

int myersGetVariantInfo(void *myersBuffer, uint32_t variant, myersVariantInfo_t *out)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || out == NULL || variant >= b->ctx->num_variants) return MYERS_E_INVALID_ARGUMENT;
    const myers_variant_desc_t *d = &b->ctx->variants[variant];
    out->lanes = d->lanes;
    out->words = d->words;
    out->maxQuerySize = 32u * d->total_words;
    out->candidatesPerWave = d->slots;
    out->ldsBytes = d->lds_bytes;
    out->workgroupsPerCU = b->ctx->occupancy[variant];
    return MYERS_SUCCESS;
}

int myersGetBinTable(void *myersBuffer, uint8_t *bin, uint32_t maxWords)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || bin == NULL) return MYERS_E_INVALID_ARGUMENT;
    for (uint32_t w = 0; w <= maxWords && w <= MAX_QUERY_WORDS; w++) bin[w] = b->ctx->bin_of_words[w];
    return MYERS_SUCCESS;
}

int myersSetBinTable(void *myersBuffer, const uint8_t *bin, uint32_t maxWords)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || bin == NULL || maxWords > MAX_QUERY_WORDS) return MYERS_E_INVALID_ARGUMENT;
    myers_ctx_t *ctx = b->ctx;
    for (uint32_t w = 0; w <= maxWords; w++) {
        if (bin[w] >= ctx->num_variants) return MYERS_E_INVALID_ARGUMENT;
        if (ctx->variants[bin[w]].total_words < (w ? w : 1u)) return MYERS_E_INVALID_ARGUMENT;
    }
    int rc = hip_fail(hipSetDevice(ctx->device), "hipSetDevice", __FILE__, __LINE__);
    if (rc) return rc;
    /* the table is shared by every buffer: wait for in-flight work first */
    rc = hip_fail(hipDeviceSynchronize(), "hipDeviceSynchronize", __FILE__, __LINE__);
    if (rc) return rc;
    for (uint32_t w = 0; w <= maxWords; w++) ctx->bin_of_words[w] = bin[w];
    ctx->tune_gen++;
    return upload_bins(ctx);
}

int myersSetChunkFactor(void *myersBuffer, uint32_t variant, uint32_t chunks)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || variant >= b->ctx->num_variants || chunks < 1u || chunks > 64u) return MYERS_E_INVALID_ARGUMENT;
    b->ctx->chunk_factor[variant] = chunks;
    b->ctx->tune_gen++;   /* cached graphs baked in the old factor */
    return MYERS_SUCCESS;
}

int myersGetChunkFactor(void *myersBuffer, uint32_t variant, uint32_t *chunks)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || chunks == NULL || variant >= b->ctx->num_variants) return MYERS_E_INVALID_ARGUMENT;
    *chunks = b->ctx->chunk_factor[variant];
    return MYERS_SUCCESS;
}

/* Apply a tuning table to a context (not yet shared with running work). */
static int load_tuning_ctx(myers_ctx_t *ctx, const char *path)
{
    FILE *fp = fopen(path, "r");
    if (fp == NULL) return MYERS_E_OPENING_FILE;
    uint8_t bin[MAX_QUERY_WORDS + 1];
    memcpy(bin, ctx->bin_of_words, sizeof(bin));
    uint32_t cf[MYERS_MAX_VARIANTS];
    memcpy(cf, ctx->chunk_factor, sizeof(cf));
    char line[256];
    uint32_t lo = 0;
    int rc = MYERS_SUCCESS;
    while (fgets(line, sizeof(line), fp)) {
        char *hash = strchr(line, '#');
        if (hash) *hash = 0;
        unsigned mw, lanes, words, chunks;
        int got = sscanf(line, "%u %u %u %u", &mw, &lanes, &words, &chunks);
        if (got <= 0) continue;
        if (got != 4 || mw < lo || mw > MAX_QUERY_WORDS || chunks < 1u || chunks > 64u) { rc = MYERS_E_READING_FILE; break; }
        int v = find_variant(ctx, lanes, words);
        if (v < 0 || ctx->variants[v].total_words < mw) { rc = MYERS_E_READING_FILE; break; }
        for (uint32_t w = lo; w <= mw; w++) bin[w] = (uint8_t)v;
        cf[v] = chunks;
        lo = mw + 1u;
    }
    fclose(fp);
    if (rc) return rc;
    memcpy(ctx->bin_of_words, bin, sizeof(bin));
    memcpy(ctx->chunk_factor, cf, sizeof(cf));
    ctx->tune_gen++;
    return upload_bins(ctx);
}

int myersLoadTuning(void *myersBuffer, const char *path)
{
    myers_buffer_t *b = (myers_buffer_t *)myersBuffer;
    if (b == NULL || path == NULL) return MYERS_E_INVALID_ARGUMENT;
    int rc = hip_fail(hipSetDevice(b->ctx->device), "hipSetDevice", __FILE__, __LINE__);
    if (rc) return rc;
    rc = hip_fail(hipDeviceSynchronize(), "hipDeviceSynchronize", __FILE__, __LINE__);
    if (rc) return rc;
    return load_tuning_ctx(b->ctx, path);
}

/* $MYERS_TUNING_FILE, else <library dir>/../tuning/gfx950.tsv; silently
 * keeps the built-in table when neither exists. */
static void load_default_tuning(myers_ctx_t *ctx)
{
    const char *env = getenv("MYERS_TUNING_FILE");
    if (env && *env) {
        if (load_tuning_ctx(ctx, env) != MYERS_SUCCESS)
            fprintf(stderr, "Myers - warning: could not apply tuning file %s\n", env);
        return;
    }
    Dl_info info;
    if (dladdr((void *)&load_default_tuning, &info) == 0 || info.dli_fname == NULL) return;
    char path[4096];
    size_t n = strlen(info.dli_fname);
    if (n + 32 >= sizeof(path)) return;
    memcpy(path, info.dli_fname, n + 1);
    char *slash = strrchr(path, '/');
    if (slash == NULL) return;
    strcpy(slash, "/../tuning/gfx950.tsv");
    FILE *fp = fopen(path, "r");
    if (fp == NULL) return;
    fclose(fp);
    if (load_tuning_ctx(ctx, path) != MYERS_SUCCESS)
        fprintf(stderr, "Myers - warning: could not apply tuning file %s\n", path);
}
